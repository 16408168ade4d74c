"""Waits of the one-kernel compaction that run out where its counts are all there: before a clearing, and in front of a
workgroup that starts afterwards.  Forced from the host; every kernel still exits normally."""
import pytest

pytestmark = pytest.mark.gpu

FIRST_MARK, LAST_REFUSED = 2, 4


def fused(L, ws, x, process):
    import torch

    from cswap_amd import api
    from cswap_amd._lib import check

    n = x.numel()
    _, words, active = api.zvc_geometry(n, process)
    values = torch.full((n,), -3.0, device="cuda")
    mask = torch.full((words * process,), -1, dtype=torch.int32, device="cuda")
    begin = torch.full((process,), -1, dtype=torch.int32, device="cuda")
    nnz = torch.full((1,), 77, dtype=torch.int32, device="cuda")
    check(L.cswap_zvc_compress_fused(x.data_ptr(), n, process, ws.data_ptr(), begin.data_ptr(), nnz.data_ptr(),
                                     values.data_ptr(), mask.data_ptr(), None), "fused")
    torch.cuda.synchronize()
    return int(nnz.item()), values, mask, begin[:active]


def same(got, x, process):
    import torch

    from cswap_amd import api

    values, mask, begin, nnz = api.zvc_compress(x, process)
    k = int(nnz.item())
    assert got[0] == k
    assert torch.equal(got[1][:k], values[:k]) and torch.equal(got[2], mask) and torch.equal(got[3], begin[:got[3].numel()])


# the first tile's count is cleared by the last tile of the third group (512 and 501 tiles in 8 groups), by the last tile of all
# (2 groups); one that reports failure and, in chunks of any length, one that must not
@pytest.mark.parametrize("n,process", [(512 * 16384, 16384), (128 * 8192, 4096), (500 * 16384 + 7, 16384), (250 * 4096, 4096)])
@pytest.mark.parametrize("skip", [FIRST_MARK, LAST_REFUSED])
def test_failed_run_reports_itself(n, process, skip):
    import torch

    from cswap_amd import api
    from cswap_amd._lib import check, lib

    L = lib()
    may_fail = L.cswap_zvc_takes_single_pass(n, process) == 2
    assert may_fail == (L.cswap_zvc_chunk_elems(n, process) % 32 == 0)
    x = torch.randn(n, generator=torch.Generator(device="cuda").manual_seed(n), device="cuda").clamp_(min=0.0)
    ws = api.zvc_workspace(process)
    same(fused(L, ws, x, process), x, process)
    L.cswap_zvc_debug_set_lookback(20000, skip)
    try:
        print("a wait runs out", flush=True)
        got = fused(L, ws, x, process)
    finally:
        L.cswap_zvc_debug_set_lookback(0, 0)
    if may_fail:
        assert got[0] == -1
    else:
        same(got, x, process)
    if skip == FIRST_MARK:
        assert int(ws.view(torch.int32)[1].item()) == 1
        again = fused(L, ws, x, process)       # until it is cleared
        if may_fail:
            assert again[0] == -1
        else:
            same(again, x, process)
    check(L.cswap_zvc_workspace_clear(ws.data_ptr(), process, None), "clear")
    same(fused(L, ws, x, process), x, process)
