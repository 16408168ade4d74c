"""Few elements in many chunks: the mask words of the chunks that hold none are cleared by workgroups of their own."""
import pytest

pytestmark = pytest.mark.gpu


def buffers(n, process):
    import torch

    from cswap_amd import api
    from cswap_amd._lib import lib

    words = lib().cswap_zvc_chunk_words(n, process) * process
    return (torch.full((n,), -3.0, device="cuda"), torch.full((words + 64,), -1, dtype=torch.int32, device="cuda"),
            torch.full((process,), -1, dtype=torch.int32, device="cuda"), torch.full((1,), -9, dtype=torch.int32, device="cuda"),
            api.zvc_workspace(process), words)


def compress(x, process, out):
    from cswap_amd._lib import check, lib

    values, mask, begin, nnz, ws, _ = out
    check(lib().cswap_zvc_compress_fused(x.data_ptr(), x.numel(), process, ws.data_ptr(), begin.data_ptr(), nnz.data_ptr(),
                                         values.data_ptr(), mask.data_ptr(), None), "fused")


# a tile of 16 x 8 rows takes up to 8192 words with it and leaves more to others: either side of that, of one workgroup's share,
# of 1024 of them, and of two tiles
@pytest.mark.parametrize("n,process", [(100, 8291), (100, 8293), (100, 8293 + 4096), (1, 1 << 20), (8192, 1 << 20), (8193, 1 << 20), (9000, 9000 + 16384),
                                       (9000, 9000 + 16385), (33, 1 << 20), (300_000, 1 << 20)])
def test_words_without_elements_are_zero(n, process):
    import torch

    from cswap_amd import api

    x = torch.randn(n, generator=torch.Generator(device="cuda").manual_seed(n), device="cuda").clamp_(min=0.0)
    want = api.zvc_compress(x, process)
    out = buffers(n, process)
    for _ in range(2):
        out[1].fill_(-1)
        compress(x, process, out)
    torch.cuda.synchronize()
    k, active, words = int(want[3].item()), api.zvc_geometry(n, process)[2], out[5]
    assert int(out[3].item()) == k
    assert torch.equal(out[0][:k], want[0][:k]) and bool((out[0][k:] == -3.0).all())
    assert torch.equal(out[1][:words], want[1]) and bool((out[1][words:] == -1).all())
    assert torch.equal(out[2][:active], want[2][:active])


def test_half_a_million_words_take_no_longer_than_a_few():
    """2 MB of zeros are a microsecond of memory; one workgroup alone stores them in 20.  The medians of ten calls each."""
    import torch

    n = 8192
    x = torch.randn(n, device="cuda").clamp_(min=0.0)

    def took(process):
        out = buffers(n, process)
        times = []
        for k in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                compress(x, process, out)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 100.0)
        return sorted(times[1:])[3]

    few, many = took(16384), took(1 << 19)
    print(few, many, flush=True)
    assert many < 2.0 * few
