"""Swapping tensors whose chunks are no whole half rows: the selector's probe and an explicit ZVC request are the compaction in
one kernel, up to 32 MiB and 256 MiB; above, and without staging room for the worst case, count and compaction apart."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("policy", ["auto", "sparse"])
@pytest.mark.parametrize("shape", [(3, 5, 29, 31), (79, 96, 28, 28), (107, 100, 28, 28), (107, 105, 28, 28), (130, 200, 28, 28)])
@pytest.mark.parametrize("room", ["worst_case", "little"])
def test_odd_chunks_out_and_back(policy, shape, room):
    import torch

    from cswap_amd import swap
    from cswap_amd._lib import lib

    n = shape[0] * shape[1] * shape[2] * shape[3]
    eng = swap.SwapEngine(pinned_bytes=8 * n + (8 << 20), device_bytes=(8 * n if room == "worst_case" else 2 * n) + (4 << 20))
    try:
        process = eng.process_for(n)
        L = lib()
        assert L.cswap_zvc_chunk_elems(n, process) % 32 != 0 and L.cswap_zvc_takes_single_pass(n, process) == 0
        gen = torch.Generator(device="cuda").manual_seed(n)
        for zeros in (0.8, 0.9):
            x = torch.rand(shape, generator=gen, device="cuda") * (torch.rand(shape, generator=gen, device="cuda") >= zeros)
            nnz = int((x != 0).sum().item())
            out = torch.full_like(x, -1.0)
            ticket = eng.pre(x, swap.AUTO if policy == "auto" else swap.SPARSE)
            info = eng.info(ticket)
            if n > 65536 or policy == "sparse":
                assert info.policy == swap.SPARSE and info.nnz == nnz
                assert info.bytes_out == 4 * process + L.cswap_zvc_mask_bytes(n, process) + 4 * nnz
            eng.post(ticket)
            eng.swap_in(ticket, out)
            eng.release(ticket)
            torch.cuda.synchronize()
            assert torch.equal(out, x)
    finally:
        eng.close()
