"""What is remembered of a tensor whose ZVC payload was sent only because the probe had made it: the selector's
own answer, raw.  From then on neither the compaction nor the host's wait for its count is paid for it."""
import pytest

pytestmark = pytest.mark.gpu

SHAPE = (64, 256, 8, 8)                                       # 4.2 MB


def half_zero(torch, seed=3):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(SHAPE, generator=gen, device="cuda")
    x[torch.rand(SHAPE, generator=gen, device="cuda") < 0.55] = 0.0
    return x


@pytest.mark.parametrize("request_name", ["AUTO", "AUTO_SPARSE"])
def test_decision_of_a_payload_sent_because_it_was_there_is_the_selectors(request_name):
    import torch

    from cswap_amd import swap

    x = half_zero(torch)
    eng = swap.SwapEngine(pinned_bytes=32 << 20, device_bytes=32 << 20)
    try:
        tk = eng.pre(x, getattr(swap, request_name))
        assert eng.info(tk).policy == swap.SPARSE and eng.decision(tk) == swap.NONE
        for explicit in (swap.NONE, swap.SPARSE, swap.ZFP):   # elsewhere the two are the same
            t2 = eng.pre(x, explicit)
            assert eng.info(t2).policy == eng.decision(t2) == explicit
            eng.release(t2)
        out = torch.full_like(x, -1.0)
        eng.swap_in(tk, out)
        torch.cuda.synchronize()
        eng.release(tk)
        assert torch.equal(out, x)
    finally:
        eng.close()


@pytest.mark.parametrize("pinned_mb,sent", [(32, [3, 2, 2, 2]), (4, [3, 3, 3, 3])])
def test_mirror_remembers_raw_and_falls_back_where_raw_has_no_room(pinned_mb, sent):
    """4 MiB of pinned memory hold the payload (2 MB) but not the tensor."""
    import torch

    from cswap_amd import swap
    from cswap_amd.execution import Execution

    x = half_zero(torch)
    eng = swap.SwapEngine(pinned_bytes=pinned_mb * 1000 * 1000, device_bytes=32 << 20)
    exe = Execution(eng)
    exe.init_(2)
    exe.policy = [-1, 0]
    try:
        tags, probes = [], []
        for _ in range(4):
            before = eng.probe_count()
            exe.preforward()
            exe.pre(x, -1); exe.post()
            exe.pre(x, 0); exe.post()
            tags.append(exe.com_and_tran(0))
            probes.append(eng.probe_count() - before)
            back = exe.fetch(0)
            torch.cuda.synchronize()
            assert torch.equal(back, x)
        assert tags == sent
        assert probes == [1 if t == swap.SPARSE else 0 for t in sent]
    finally:
        eng.close()


def test_hooks_remember_raw():
    import torch

    from cswap_amd import swap
    from cswap_amd.hooks import swap_saved_tensors

    eng = swap.SwapEngine(pinned_bytes=64 << 20, device_bytes=64 << 20)
    memo, probes, sent, gradients = {}, [], [], []
    try:
        for _ in range(3):
            w = half_zero(torch).requires_grad_()
            before = eng.probe_count()
            ctx = swap_saved_tensors(eng, policy=swap.AUTO, min_bytes=1 << 20, memo=memo)
            with ctx:
                loss = (w * 2.0).square().sum()                # the square saves 2 w: half zeros, no leaf
            probes.append(eng.probe_count() - before)
            sent.append(dict(ctx.stats["by_policy"]))
            loss.backward()
            ctx.close()
            gradients.append(w.grad)
        assert sent == [{"zvc": 1}, {"raw": 1}, {"raw": 1}] and probes == [1, 0, 0]
        assert [v[0] for v in memo.values()] == [swap.NONE]
        for g in gradients:
            assert torch.equal(g, 8.0 * half_zero(torch))
    finally:
        eng.close()


def test_cpp_mirror_remembers_raw():
    from test_gpu_execution import _build_and_run_cpp

    out = _build_and_run_cpp("cpp_made_payload_memo")
    assert out.returncode == 0, out.stdout
    assert out.stdout.split()[-9:] == ["OK", "3", "1", "2", "0", "2", "0", "2", "0"]
