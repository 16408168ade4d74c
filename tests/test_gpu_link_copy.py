"""Payloads that come in on the compute stream: the copy kernel at the edges of its pieces and of its grid, and the
runtime's copy in its place beside a copy out."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine():
    from cswap_amd import swap

    e = swap.SwapEngine(pinned_bytes=256 << 20, device_bytes=256 << 20)
    yield e
    e.close()


# pieces of 16 bytes, 256 to a workgroup, 64 workgroups a turn: below and above each, and remainders of 1 to 3 words
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 1023, 1024, 1027, 65535, 65536, 65539, 200001])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_raw_payload_comes_back_at_any_element(engine, n, shift):
    import torch

    from cswap_amd import swap

    for _ in range(2):  # the second time through the same pinned block, with other values
        x = torch.randn(1, 1, 1, n, device="cuda")
        room = torch.full((n + 8,), -7.0, device="cuda")
        ticket = engine.pre(x, swap.NONE)
        engine.post(ticket)
        engine.swap_in(ticket, room[shift:shift + n])
        engine.release(ticket)
        torch.cuda.synchronize()
        assert torch.equal(room[shift:shift + n], x.view(-1))
        assert bool((room[:shift] == -7.0).all()) and bool((room[shift + n:] == -7.0).all())


@pytest.mark.parametrize("policy", ["none", "sparse", "zfp"])
def test_payload_comes_in_beside_a_copy_out(engine, policy):
    import torch

    from cswap_amd import swap

    pol = {"none": swap.NONE, "sparse": swap.SPARSE, "zfp": swap.ZFP}[policy]
    x = torch.randn(64, 64, 16, 16, device="cuda").clamp_(min=0.0)
    big = torch.randn(1, 32, 1024, 1024, device="cuda")
    alone, beside, back = torch.empty_like(x), torch.empty_like(x), torch.empty_like(big)
    for out, other in ((alone, False), (beside, True)):
        ticket = engine.pre(x, pol)
        engine.post(ticket)
        outbound = engine.pre(big, swap.NONE) if other else None
        engine.swap_in(ticket, out)
        engine.release(ticket)
        if other:
            engine.post(outbound)
            engine.swap_in(outbound, back)
            engine.release(outbound)
    torch.cuda.synchronize()
    assert torch.equal(alone, beside) and torch.equal(back, big)
    if policy != "zfp":
        assert torch.equal(alone, x)


@pytest.mark.parametrize("n", [1001, 1 << 20])
@pytest.mark.parametrize("order", ["in", "in_post", "prefetch_in", "prefetch_post_in", "prefetch_release"])
def test_raw_tensor_asked_back_behind_its_copy_out(engine, order, n):
    """A long copy out goes ahead, so that the tensor's own is still to come when it is asked back."""
    import torch

    from cswap_amd import swap

    big = torch.randn(1, 16, 1024, 1024, device="cuda")
    for _ in range(2):
        x = torch.randn(1, 1, 1, n, device="cuda")
        want, out = x.clone(), torch.empty_like(x)
        torch.cuda.synchronize()
        ahead = engine.pre(big, swap.NONE)
        ticket = engine.pre(x, swap.NONE)
        if order.startswith("prefetch"):
            engine.prefetch(ticket)
        if order == "prefetch_post_in":
            engine.post(ticket)
            x.fill_(3.0)
        if order != "prefetch_release":
            engine.swap_in(ticket, out)
        if order == "in_post":
            engine.post(ticket)
            x.fill_(3.0)
        engine.release(ticket)
        engine.post(ahead)
        engine.release(ahead)
        torch.cuda.synchronize()
        assert order == "prefetch_release" or torch.equal(out, want)


def test_raw_tensor_comes_back_into_itself(engine):
    import torch

    from cswap_amd import swap

    x = torch.randn(1, 4, 1024, 1024, device="cuda")
    want = x.clone()
    for _ in range(3):
        ticket = engine.pre(x, swap.NONE)
        engine.swap_in(ticket, x)
        engine.release(ticket)
    torch.cuda.synchronize()
    assert torch.equal(x, want)


@pytest.mark.parametrize("order", ["in", "prefetch_in", "prefetch_release"])
def test_raw_tensor_asked_back_while_another_payload_is_staged(engine, order):
    """A long copy out goes ahead of both, so the raw tensor's own copy is still to come and the other's payload
    still staged: the stream waits, and the other comes back from its staging block."""
    import torch

    from cswap_amd import swap

    big = torch.randn(1, 16, 1024, 1024, device="cuda")
    for _ in range(2):
        x = torch.randn(1, 1, 1, 200001, device="cuda")
        y = torch.randn(1, 8, 256, 256, device="cuda").clamp_(min=0.0)
        want, out, back = x.clone(), torch.empty_like(x), torch.empty_like(y)
        torch.cuda.synchronize()
        ahead = engine.pre(big, swap.NONE)
        other = engine.pre(y, swap.SPARSE)
        ticket = engine.pre(x, swap.NONE)
        if order.startswith("prefetch"):
            engine.prefetch(ticket)
        if order != "prefetch_release":
            engine.swap_in(ticket, out)
        engine.release(ticket)
        engine.swap_in(other, back)
        engine.release(other)
        engine.post(ahead)
        engine.release(ahead)
        torch.cuda.synchronize()
        assert torch.equal(back, y)
        assert order == "prefetch_release" or torch.equal(out, want)
