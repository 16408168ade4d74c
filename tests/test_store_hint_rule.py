"""Which fields the ZFP decoder stores with the nontemporal hint: by where its rows start and how long they are, the
field's size and the rate.  The rule is host code; what it sends to other kernels comes out the same on the GPU."""
import numpy as np
import pytest

MIB = 1 << 20


def hint(pitch, mib, base=0, plane=None, rate=8):
    from cswap_amd import _lib

    plane = 64 * pitch if plane is None else plane
    return _lib.lib().cswap_test_zfp_store_hint(4096 + base, pitch, plane, int(mib * MIB), 64 * rate)


def test_whole_lines_always_carry_it():
    assert all(hint(p, m) for p in (128, 256, 3072) for m in (1, 30, 100, 400))


def test_rows_that_start_inside_a_line_are_no_whole_lines():
    """A view that starts 16 bytes into a line, or planes at a distance that is no multiple of a line."""
    for where in ({"base": 16}, {"plane": 64 * 128 + 16}):
        assert hint(128, 12, **where) and not hint(128, 25, **where) and not hint(128, 140, **where)
    assert hint(512, 30, base=16) and not hint(512, 48, base=16)
    assert hint(3072, 48, base=16) and not hint(3072, 190, base=16)
    assert hint(128, 30, base=64) and not hint(128, 48, base=64) and hint(128, 140, base=64)


def test_half_lines():
    assert hint(64, 34) and not hint(64, 41) and not hint(64, 105) and hint(64, 134)
    assert hint(192, 55) and not hint(192, 105) and hint(192, 134)
    assert all(hint(p, m) for p in (320, 448, 1088) for m in (10, 50, 110, 140))


def test_parts_of_lines():
    assert not any(hint(p, m, rate=r) for p in (16, 32, 48, 80) for m in (10, 30, 140) for r in (4, 8, 12))
    assert hint(144, 17) and not hint(112, 17) and not hint(144, 24)
    assert hint(112, 17, rate=16) and hint(96, 17, rate=12) and not hint(112, 24, rate=16)
    assert hint(160, 23) and not hint(160, 28) and hint(784, 23) and not hint(784, 40)
    assert hint(160, 31, rate=16) and not hint(160, 23, rate=4) and not hint(160, 40, rate=64)
    assert hint(1552, 90) and not hint(1552, 190) and hint(3088, 20)


@pytest.mark.gpu
@pytest.mark.parametrize("maxbits", [512, 1024])
@pytest.mark.parametrize("nx,ny,nz,pitch,extra,off", [(32, 32, 60, 32, 0, 4), (32, 32, 60, 32, 4, 0), (128, 12, 31, 128, 0, 16),
                                                      (30, 9, 21, 32, 0, 4), (768, 8, 12, 768, 0, 4), (24, 24, 40, 24, 0, 0),
                                                      (64, 64, 1500, 64, 0, 4), (64, 64, 2400, 64, 0, 4), (40, 40, 3700, 40, 0, 0),
                                                      (40, 40, 4800, 40, 0, 0), (16, 16, 38000, 16, 0, 0), (16, 16, 40000, 16, 0, 0)])
def test_views_and_sizes_around_the_lines_of_the_rule(nx, ny, nz, pitch, extra, off, maxbits):
    """nx, ny, nz: the field, pitch: elements from row to row, extra: elements between planes, off: where the view starts."""
    import torch

    import oracle
    from cswap_amd import _lib

    L = _lib.lib()
    plane = pitch * ny + extra
    f = np.random.default_rng(nx + nz).standard_normal((nz, ny, nx)).astype(np.float32)
    want = oracle.zfp_encode3(f, maxbits)
    back0 = oracle.zfp_decode3(want, f.shape, maxbits)
    raw = torch.full((off + nz * plane + 64,), 7.0, device="cuda")
    assert raw.data_ptr() % 128 == 0
    view = raw[off:off + nz * plane].view(nz, plane)[:, :pitch * ny].unflatten(1, (ny, pitch))[:, :, :nx]
    view.copy_(torch.from_numpy(f))
    s = torch.zeros(want.size * 8, dtype=torch.uint8, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    base = raw.data_ptr() + 4 * off
    assert L.cswap_zfp_compress_f32(base, nx, ny, nz, 1, pitch, plane, maxbits, s.data_ptr(), st) == 0
    assert np.array_equal(s.cpu().numpy().view(np.uint64), want)
    raw.fill_(7.0)
    assert L.cswap_zfp_decompress_f32(s.data_ptr(), nx, ny, nz, 1, pitch, plane, maxbits, base, st) == 0
    assert np.array_equal(view.contiguous().view(torch.int32).cpu().numpy(), back0.view(np.int32))
    view.fill_(7.0)
    assert bool((raw == 7.0).all())                            # nothing beside the field was written
