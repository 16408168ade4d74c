"""The decoder's form with four lanes per block: up to how many blocks it takes a field, by the length of its rows, and
the same bits on both sides of each line."""
import numpy as np
import pytest

CUS, PER_WAVE = 256, 16


@pytest.mark.parametrize("side,rate,waves", [(4, 8, 11), (8, 8, 11), (4, 4, 11), (8, 32, 11), (4, 64, 11), (12, 8, 9), (16, 8, 9),
                                             (28, 8, 9), (4, 16, 9), (8, 24, 9), (8, 28, 11), (7, 8, 9)])
def test_last_size_by_the_length_of_the_rows(side, rate, waves):
    """7: rows that end inside a block; 16 to 24 bits per value: the pair form is next in line there."""
    from cswap_amd import _lib

    quad = _lib.lib().cswap_test_zfp_decode_quad
    per_slab = (-(-side // 4)) ** 2
    slabs = waves * PER_WAVE * CUS // per_slab
    assert quad(side, side, 4 * slabs, 0, 0, 64 * rate, CUS) == 1
    assert quad(side, side, 4 * (slabs + 1), 0, 0, 64 * rate, CUS) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("side,slabs,rate", [(4, 36865, 8), (4, 45056, 8), (4, 45057, 8), (8, 9217, 8), (8, 11264, 4), (8, 11265, 12), (4, 36865, 16),
                                             (4, 45056, 64)])
def test_short_rows_on_both_sides_of_the_line(side, slabs, rate):
    import torch

    import oracle
    from cswap_amd import api

    f = np.random.default_rng(slabs).standard_normal((4 * slabs, side, side)).astype(np.float32)
    want = oracle.zfp_encode3(f, 64 * rate, omp=True)
    s = api.cuda_compress(torch.from_numpy(f).cuda(), 64 * rate)
    assert np.array_equal(s.view(torch.uint8).flatten().cpu().numpy()[:want.size * 8], want.view(np.uint8))
    back = api.cuda_decompress(s, f.shape, 64 * rate)
    assert np.array_equal(back.cpu().numpy().view(np.uint32), oracle.zfp_decode3(want, f.shape, 64 * rate, omp=True).view(np.uint32))
