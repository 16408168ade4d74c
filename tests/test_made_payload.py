"""A tensor between the sizes at which the selector probes and at which it compresses: the probe makes the
ZVC payload, and the engine sends it if what is left to pay for it is less than the raw swap."""
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("zeros,sends", [(0.55, True), (0.9, True), (0.05, False), (0.0, False)])
def test_payload_that_the_probe_has_made_is_sent_where_it_pays(zeros, sends):
    import torch

    from cswap_amd import swap
    from cswap_amd.workloads import field_dims

    shape = (64, 256, 8, 8)                                  # 4.2 MB
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(shape, generator=gen, device="cuda")
    x[torch.rand(shape, generator=gen, device="cuda") < zeros] = 0.0
    nnz = int((x != 0).sum().item())
    eng = swap.SwapEngine(pinned_bytes=32 << 20, device_bytes=32 << 20)
    try:
        tk = eng.pre(x, swap.AUTO)
        info = eng.info(tk)
        assert eng.probe_count() == 1
        if zeros < 0.9:                                      # by its full price the selector would send it raw
            assert swap.select_field(*field_dims(shape), nnz).policy == swap.NONE
        assert info.policy == (swap.SPARSE if sends else swap.NONE) and info.nnz == nnz
        assert info.bytes_out < 0.6 * x.numel() * 4 if sends else info.bytes_out == x.numel() * 4
        out = torch.full_like(x, -1.0)
        eng.swap_in(tk, out)
        torch.cuda.synchronize()
        eng.release(tk)
        assert torch.equal(out, x)
    finally:
        eng.close()
