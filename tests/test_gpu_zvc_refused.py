"""The one-kernel compaction of shapes that never report failure, on workspaces that it finds unusable: the last tile of
every group of 64 compacts the group."""
import pytest

pytestmark = pytest.mark.gpu

KB = 1024


def outputs(n, process):
    import torch

    from cswap_amd._lib import lib

    return (torch.full((n + 1,), -3.0, device="cuda"),
            torch.full((lib().cswap_zvc_chunk_words(n, process) * process,), -1, dtype=torch.int32, device="cuda"),
            torch.full((process,), -1, dtype=torch.int32, device="cuda"), torch.full((1,), -9, dtype=torch.int32, device="cuda"))


def fused(x, process, ws, out):
    from cswap_amd._lib import check, lib

    check(lib().cswap_zvc_compress_fused(x.data_ptr(), x.numel(), process, ws.data_ptr(), out[2].data_ptr(), out[3].data_ptr(),
                                         out[0].data_ptr(), out[1].data_ptr(), None), "fused")


def flagged(x, process, out):
    """A workspace on which a wait has run out."""
    import torch

    from cswap_amd import api
    from cswap_amd._lib import lib

    ws = api.zvc_workspace(process)
    lib().cswap_zvc_debug_set_lookback(4, 1)
    try:
        print("a wait runs out", flush=True)
        fused(x, process, ws, out)
        torch.cuda.synchronize()
    finally:
        lib().cswap_zvc_debug_set_lookback(0, 0)
    assert int(ws.view(torch.int32)[1].item()) == 1
    return ws


# tiles of 8192, 16384 and 16384 (half as many wavefronts) elements: one, a whole group, one more, groups and a part, chunks of one
# element, of a whole tensor, chunks that end with tiles, whole half rows (the last three), and more than 64 MiB
@pytest.mark.parametrize("n,process", [(5000, 16), (64 * 8192, 1000), (64 * 8192 + 1, 1024), (65 * 8192, 65 * 8192), (200 * 8192 - 3, 1),
                                       (130 * 16384 + 5, 16384), (192 * 16384 - 1, 999), (600 * 16384 + 77, 16384), (30_105_600, 16384),
                                       (16384 * KB - 64, 16384), (8192 * KB + 16384, 8192 + 16), (16384 * KB - 16384, 16383)])
@pytest.mark.parametrize("state", ["flagged", "never prepared"])
def test_unusable_workspace(n, process, state):
    import torch

    from cswap_amd import api
    from cswap_amd._lib import lib

    assert lib().cswap_zvc_takes_single_pass(n, process) == 0
    x = torch.randn(n, generator=torch.Generator(device="cuda").manual_seed(n), device="cuda").clamp_(min=0.0)
    if state == "flagged" and n > 8192:      # (one tile waits for nobody)
        ws = flagged(x, process, outputs(n, process))
    else:
        ws = torch.full_like(api.zvc_workspace(process), 0xa5)
    want, active = api.zvc_compress(x, process), api.zvc_geometry(n, process)[2]
    held = ws.clone()
    out = outputs(n, process)
    fused(x, process, ws, out)
    torch.cuda.synchronize()
    k = int(want[3].item())
    assert int(out[3].item()) == k
    assert torch.equal(out[0][:k], want[0][:k]) and bool((out[0][k:] == -3.0).all())
    assert torch.equal(out[1], want[1]) and torch.equal(out[2][:active], want[2][:active]) and bool((out[2][active:] == -1).all())
    assert torch.equal(ws, held)


def test_time_grows_with_the_size_and_not_its_square():
    import torch

    times = []
    for n in (15_052_800, 60_211_200):
        process = 16384
        x = torch.randn(n, device="cuda").clamp_(min=0.0)
        out = outputs(n, process)
        ws = flagged(x, process, out)
        took = []
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            fused(x, process, ws, out)
            b.record()
            b.synchronize()
            took.append(a.elapsed_time(b))
        times.append(min(took))
    print(times, flush=True)
    assert times[1] < 8.0 * times[0]  # four times the size; the square is sixteen times
