"""Short ZVC chunks at any element: which sizes are expanded with the nontemporal hint, and the same bits on
either side of each line."""
import numpy as np
import pytest

MB = 1 << 20


def test_sizes_that_carry_the_hint():
    """Measured per size: ahead or level below some 28 MiB, behind from there to 128 MiB, ahead again above."""
    from cswap_amd import _lib

    hint = _lib.lib().cswap_test_zvc_packed_hint
    assert [hint(b) for b in (4, 19_000_000, 24_000_000, 28 * MB - 4)] == [1] * 4
    assert [hint(b) for b in (28 * MB, 32_000_000, 42_000_000, 87_000_000, 128 * MB - 4)] == [0] * 5
    assert [hint(b) for b in (128 * MB, 168_000_000)] == [1] * 2


@pytest.mark.gpu
@pytest.mark.parametrize("elems,process,cut", [(447, 16384, 5), (449, 16384, 0), (449, 16384, 3), (641, 16384, 1), (113, 65536, 2),
                                               (511, 65536, 7), (513, 65536, 5)])
def test_short_chunks_at_any_element_on_both_sides_of_the_lines(elems, process, cut):
    import torch

    from cswap_amd import _lib, api

    L = _lib.lib()
    n = elems * process - cut
    assert api.zvc_geometry(n, process)[0] == elems
    gen = torch.Generator(device="cuda").manual_seed(elems)
    x = torch.randn(n, generator=gen, device="cuda").clamp_(min=0.0)
    _, words, active = api.zvc_geometry(n, process)
    values = torch.zeros(n, device="cuda")
    mask = torch.zeros(words * process, dtype=torch.int32, device="cuda")
    begin = torch.zeros(process, dtype=torch.int32, device="cuda")
    nnz = torch.zeros(1, dtype=torch.int32, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert L.cswap_zvc_compress(x.data_ptr(), n, process, begin.data_ptr(), nnz.data_ptr(), values.data_ptr(), mask.data_ptr(), st) == 0
    back = torch.full((n + 8,), -1.0, device="cuda")
    assert L.cswap_zvc_expand(values.data_ptr(), mask.data_ptr(), begin.data_ptr(), n, process, back[4:].data_ptr(), st) == 0
    assert torch.equal(back[4:4 + n], x)
    assert bool((back[:4] == -1.0).all()) and bool((back[4 + n:] == -1.0).all())
    assert np.array_equal(values[:int(nnz)].cpu().numpy(), x[x != 0].cpu().numpy())
