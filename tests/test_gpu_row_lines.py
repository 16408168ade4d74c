"""ZFP fields by the bytes of their rows: whole lines, half lines, parts of lines; the forms that store and
load them with and without the nontemporal hint, against the checker."""
import ctypes as C

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("maxbits", [256, 512, 1024])
@pytest.mark.parametrize("shape,pitch", [((64, 4, 4), 0), ((64, 8, 8), 0), ((32, 16, 16), 0), ((24, 28, 28), 0), ((20, 36, 36), 0),
                                         ((12, 48, 48), 0), ((9, 30, 32), 0), ((9, 30, 27), 28), ((9, 30, 32), 36), ((6, 9, 388), 0),
                                         ((8, 16, 383), 384), ((5, 7, 772), 0)])
def test_fields_by_their_row_length(shape, pitch, maxbits):
    import torch

    from cswap_amd import _lib

    L = _lib.lib()
    nz, ny, nx = shape
    p = pitch or nx
    rng = np.random.default_rng(nx)
    f = rng.standard_normal(shape).astype(np.float32)
    want = oracle.zfp_encode3(f, maxbits)
    wide = np.full((nz, ny, p), 7.0, np.float32)
    wide[:, :, :nx] = f
    x = torch.from_numpy(wide).cuda()
    st = torch.cuda.current_stream().cuda_stream
    back0 = oracle.zfp_decode3(want, f.shape, maxbits)
    before = (C.c_size_t * 2)()
    L.cswap_zfp_set_pair_bytes(0, 0, before)
    try:
        for limit in (0, int(before[0]), (1 << 64) - 1):     # one lane per block, as shipped, the pair form where it applies
            L.cswap_zfp_set_pair_bytes(limit, limit, None)
            s = torch.zeros(want.size * 8, dtype=torch.uint8, device="cuda")
            assert L.cswap_zfp_compress_f32(x.data_ptr(), nx, ny, nz, 1, p, p * ny, maxbits, s.data_ptr(), st) == 0
            assert np.array_equal(s.cpu().numpy().view(np.uint64), want)
            back = torch.full_like(x, 7.0)
            assert L.cswap_zfp_decompress_f32(s.data_ptr(), nx, ny, nz, 1, p, p * ny, maxbits, back.data_ptr(), st) == 0
            got = back.cpu().numpy()
            assert np.array_equal(got[:, :, :nx].copy().view(np.uint32), back0.view(np.uint32))
            assert (got[:, :, nx:] == 7.0).all()
    finally:
        L.cswap_zfp_set_pair_bytes(before[0], before[1], None)


@pytest.mark.parametrize("shape", [(8448, 64, 64), (2100000, 4, 4), (43000, 28, 28)])
def test_large_fields_by_their_row_length(shape):
    """134 MiB and more, where the hints change: the same stream and values as in pieces below that size."""
    import torch

    from cswap_amd import api

    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(shape, generator=gen, device="cuda")
    s = api.cuda_compress(x, 512)
    back = api.cuda_decompress(s, x.shape, 512)
    cut = shape[0] // 8 * 4
    for part in (slice(0, cut), slice(cut, shape[0])):
        y = x[part].contiguous()
        t = api.cuda_compress(y, 512)
        n = t.numel()
        off = 0 if part.start == 0 else s.numel() - n
        assert torch.equal(s.view(torch.uint8).flatten()[off:off + n], t.view(torch.uint8).flatten())
        assert torch.equal(back[part].view(torch.int32), api.cuda_decompress(t, y.shape, 512).view(torch.int32))
