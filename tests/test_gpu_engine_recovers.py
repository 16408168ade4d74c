"""An engine whose single-kernel compaction has given up once, on shapes whose workgroups could count for themselves: that swap is
right, and the next one is as fast as the one before."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("policy,shape", [("sparse", (64, 192, 35, 35)), ("auto", (79, 96, 28, 28)), ("sparse", (107, 200, 28, 28))])
def test_swap_out_after_a_wait_that_ran_out(policy, shape):
    import torch

    from cswap_amd import swap
    from cswap_amd._lib import lib

    L = lib()
    n = shape[0] * shape[1] * shape[2] * shape[3]
    eng = swap.SwapEngine(pinned_bytes=4 * n + (8 << 20), device_bytes=8 * n + (8 << 20), timing=True)
    try:
        process = eng.process_for(n)
        assert L.cswap_zvc_chunk_elems(n, process) % 32 != 0 and L.cswap_zvc_takes_single_pass(n, process) == 0
        gen = torch.Generator(device="cuda").manual_seed(n)
        x = torch.rand(shape, generator=gen, device="cuda") * (torch.rand(shape, generator=gen, device="cuda") >= 0.9)
        nnz = int((x != 0).sum().item())

        def out_and_back():
            ticket = eng.pre(x, swap.AUTO if policy == "auto" else swap.SPARSE)
            eng.post(ticket)
            info, took = eng.info(ticket), eng.timing(ticket).compress_us
            out = torch.full_like(x, -1.0)
            eng.swap_in(ticket, out)
            eng.release(ticket)
            torch.cuda.synchronize()
            assert info.policy == swap.SPARSE and info.nnz == nnz and torch.equal(out, x)
            return took

        out_and_back()
        before = min(out_and_back() for _ in range(3))
        L.cswap_zvc_debug_set_lookback(4, 1)
        try:
            print("forced give-up inside the engine", flush=True)
            out_and_back()
        finally:
            L.cswap_zvc_debug_set_lookback(0, 0)
        after = min(out_and_back() for _ in range(3))
        print(before, after, flush=True)
        assert after < 3.0 * before        # every workgroup counting for itself: 30 to 100 times
    finally:
        eng.close()
