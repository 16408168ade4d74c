"""The one-kernel compaction of small tensors, and of larger ones in chunks that are no whole half rows, where its tiles
and its groups of 64 tiles begin and end, against the three kernels: values, mask, offsets and count, three runs on one
workspace with other data in each."""
import pytest

pytestmark = pytest.mark.gpu

KB = 1024
# tiles of 8192 elements up to 2 M elements, of 16384 above, 4096 of them at most; whole half rows per chunk, and any length
SHAPES = [(1, 1), (8191, 16), (8192, 256), (8193, 7), (64 * 8192, 1024), (64 * 8192 + 1, 1024), (65 * 8192 - 5, 333),
          (128 * 8192, 4096), (129 * 8192 + 31, 16384), (192 * 8192 + 1, 50), (2048 * KB, 2048), (2048 * KB + 1, 2048),
          (2048 * KB + 64, 2049), (64 * 16384 * 3 - 1, 16384), (8192 * KB, 16384), (8192 * KB + 1, 8192), (8192 * KB + 16384, 16383),
          (16384 * KB - 1, 16384), (16384 * KB + 1, 16384), (30_105_600, 16384), (65536 * KB - 49157, 16384), (3_000_000, 1), (3_000_001, 65536), (700_000, 700_000)]


@pytest.mark.parametrize("n,process", SHAPES)
def test_tiles_against_three_kernels(n, process):
    import torch

    from cswap_amd import api
    from cswap_amd._lib import check, lib

    L = lib()
    W, active = L.cswap_zvc_chunk_words(n, process), L.cswap_zvc_active_chunks(n, process)
    ws = api.zvc_workspace(process)
    gen = torch.Generator(device="cuda").manual_seed(n)
    before = L.cswap_zvc_set_single_pass_bytes(64 << 20)
    try:
        for zeros in (0.5, 0.0, 0.97):
            x = torch.randn(n, generator=gen, device="cuda") * (torch.rand(n, generator=gen, device="cuda") >= zeros)
            want = api.zvc_compress(x, process)
            got = [torch.full((n,), -3.0, device="cuda"), torch.full((W * process,), -1, dtype=torch.int32, device="cuda"),
                   torch.full((process,), -1, dtype=torch.int32, device="cuda"), torch.full((1,), -9, dtype=torch.int32, device="cuda")]
            check(L.cswap_zvc_compress_fused(x.data_ptr(), n, process, ws.data_ptr(), got[2].data_ptr(), got[3].data_ptr(),
                                             got[0].data_ptr(), got[1].data_ptr(), None), "fused")
            torch.cuda.synchronize()
            k = int(want[3].item())
            assert int(got[3].item()) == k
            assert torch.equal(got[0][:k], want[0][:k]) and bool((got[0][k:] == -3.0).all())
            assert torch.equal(got[1], want[1]) and torch.equal(got[2][:active], want[2][:active])
        words = ws.view(torch.int32)
        assert int(words[1].item()) == 0 and int(words[4].item()) == 3
        assert int(words[16:].count_nonzero().item()) == 256  # the totals of the last run, nothing else
    finally:
        L.cswap_zvc_set_single_pass_bytes(before)


def test_more_than_the_groups_hold_runs_the_three_kernels():
    import torch

    from cswap_amd import api
    from cswap_amd._lib import check, lib

    n, process = 65536 * KB + 1, 16384
    L = lib()
    x = torch.randn(n, device="cuda").clamp_(min=0.0)
    want = api.zvc_compress(x, process)
    got = [torch.zeros_like(o) for o in want]
    ws = api.zvc_workspace(process)
    check(L.cswap_zvc_compress_fused(x.data_ptr(), n, process, ws.data_ptr(), got[2].data_ptr(), got[3].data_ptr(),
                                     got[0].data_ptr(), got[1].data_ptr(), None), "fused")
    torch.cuda.synchronize()
    k = int(want[3].item())
    assert int(got[3].item()) == k and torch.equal(got[0][:k], want[0][:k]) and torch.equal(got[1], want[1])
    assert int(ws.view(torch.int32)[4].item()) == 0


# either side of the sizes from which the pipeline kernel reads its input, and stores its values, with the nontemporal hint
@pytest.mark.parametrize("mib,off", [(80, -16384), (80, 0), (80, 16384), (320, -16384), (320, 0), (328, 0)])
def test_pipeline_hints_against_three_kernels(mib, off):
    import torch

    from cswap_amd import api
    from cswap_amd._lib import check, lib

    process = 16384
    n = (mib << 18) + 32 * off
    L = lib()
    assert L.cswap_zvc_takes_single_pass(n, process) == 1
    x = torch.empty(n, device="cuda").normal_(generator=torch.Generator(device="cuda").manual_seed(mib)).clamp_(min=0.0)
    want = api.zvc_compress(x, process)
    got = [torch.zeros_like(o) for o in want]
    ws = api.zvc_workspace(process)
    for _ in range(2):
        check(L.cswap_zvc_compress_fused(x.data_ptr(), n, process, ws.data_ptr(), got[2].data_ptr(), got[3].data_ptr(),
                                         got[0].data_ptr(), got[1].data_ptr(), None), "fused")
    torch.cuda.synchronize()
    k = int(want[3].item())
    assert int(got[3].item()) == k and torch.equal(got[0][:k], want[0][:k])
    assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])


# the staged expansion lays its rows out from the line that a chunk begins in: chunks below and above one word, one row and
# the eight rows of a turn, destinations at every kind of place in a line, nothing stored outside
@pytest.mark.parametrize("length", [1, 31, 32, 33, 255, 257, 2016, 2017, 2048, 2049, 4133])
@pytest.mark.parametrize("off", [0, 1, 4, 15, 31])
@pytest.mark.parametrize("short", [0, 1])
def test_staged_expansion_at_any_place_of_a_line(length, off, short):
    import torch

    from cswap_amd import api
    from cswap_amd._lib import check, lib

    process = 37
    n = length * process - min(short, length - 1)
    x = torch.randn(n, device="cuda").clamp_(min=0.0)
    values, mask, begin, _ = api.zvc_compress(x, process)
    L = lib()
    before = L.cswap_zvc_set_staged_compact_bytes(0)
    try:
        room = torch.full((n + 96,), -7.0, device="cuda")
        at = 32 + off
        check(L.cswap_zvc_expand(values.data_ptr(), mask.data_ptr(), begin.data_ptr(), n, process,
                                 room.data_ptr() + 4 * at, torch.cuda.current_stream().cuda_stream), "expand")
        torch.cuda.synchronize()
    finally:
        L.cswap_zvc_set_staged_compact_bytes(before)
    assert torch.equal(room[at:at + n], x)
    assert bool((room[:at] == -7.0).all()) and bool((room[at + n:] == -7.0).all())
