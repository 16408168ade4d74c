"""Packed fields whose rows are not made of whole lines: the decoder that stores block rows as runs through LDS."""
import os
import subprocess

import numpy as np
import pytest

import oracle

HERE = os.path.dirname(os.path.abspath(__file__))
MIB = 1 << 20


def test_every_element_is_stored_once_from_its_place(tmp_path):
    exe = str(tmp_path / "runs")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(HERE, "cpp_runs.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout


def test_route():
    from cswap_amd import _lib

    def route(nx, ny, mb, sy=0, sz=0, base=0):
        return _lib.lib().cswap_test_zfp_decode_runs(nx, ny, max(1, mb * MIB // (4 * nx * ny)), sy, sz, base)

    assert [route(28, 28, mb) for mb in (10, 100)] == [2, 2] and [route(4, 4, mb) for mb in (10, 100)] == [2, 2]
    assert [route(32, 32, mb) for mb in (10, 100)] == [0, 0]                      # whole lines
    assert [route(80, 80, 20), route(48, 48, 20), route(48, 48, 60), route(16, 16, 20)] == [0, 0, 2, 2]
    assert [route(35, 35, mb) for mb in (20, 60)] == [2, 1] and [route(7, 7, mb) for mb in (20, 60)] == [1, 1]
    assert [route(n, n, 20) for n in (17, 33, 49, 63)] == [2] * 4 and [route(n, n, 60) for n in (17, 33, 49, 63)] == [0] * 4
    assert [route(n, n, 60) for n in (2, 6, 10, 15, 13, 30, 50)] == [1, 1, 1, 1, 0, 1, 0]
    assert [route(n, n, 30) for n in (17, 33, 49, 197)] == [2, 2, 0, 0]              # lanes left over
    assert route(28, 28, 60, base=4) == 1 and route(28, 28, 60, base=8) == 1      # off 16 bytes
    assert route(28, 28, 60, sy=29) == 0 and route(28, 28, 60, sz=28 * 28 + 4) == 0 and route(28, 28, 60, sy=28, sz=28 * 28) == 2
    assert route(132, 64, 20) == 0 and route(260, 64, 20) == 0                    # lanes left over; longer than a wavefront
    assert route(4, 1 << 20, 64) == 0                                              # a plane of 2^22 elements


@pytest.mark.gpu
@pytest.mark.parametrize("maxbits", [256, 512, 1024])
@pytest.mark.parametrize("shape", [(256, 4, 4), (67, 7, 7), (33, 5, 8), (61, 1, 28), (18, 14, 14), (9, 17, 17), (5, 1030, 12),
                                   (13, 28, 28), (6, 35, 35), (3, 49, 49), (7, 197, 197), (2, 9, 254), (66, 3, 2)])
@pytest.mark.parametrize("off", [0, 1, 2])
def test_fields_against_the_checker(shape, maxbits, off):
    import ctypes as C

    import torch

    from cswap_amd import _lib

    L = _lib.lib()
    nz, ny, nx = shape
    f = np.random.default_rng(nx + ny).standard_normal(shape).astype(np.float32)
    want = oracle.zfp_encode3(f, maxbits)
    values = oracle.zfp_decode3(want, f.shape, maxbits).ravel().view(np.uint32)
    s = torch.from_numpy(want.view(np.uint8).copy()).cuda()
    st = torch.cuda.current_stream().cuda_stream
    before = (C.c_size_t * 2)()
    L.cswap_zfp_set_pair_bytes(0, 0, before)                 # one lane per block whatever the size
    try:
        raw = torch.full((f.size + 64,), 7.0, device="cuda")
        at = raw.data_ptr() + 4 * (32 + off)                 # a line's start, 4 and 8 bytes behind one
        assert at % 128 == 4 * off
        assert L.cswap_zfp_decompress_f32(s.data_ptr(), nx, ny, nz, 0, 0, 0, maxbits, at, st) == 0
        got = raw.cpu().numpy()
    finally:
        L.cswap_zfp_set_pair_bytes(before[0], before[1], None)
    assert np.array_equal(got[32 + off:32 + off + f.size].view(np.uint32), values)
    assert (got[:32 + off] == 7.0).all() and (got[32 + off + f.size:] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(9300, 35, 35), (215000, 7, 7), (54000, 14, 14), (13500, 28, 28)])
def test_large_fields_without_the_hint(shape):
    """40 MiB and more: the same values as row by row, which is how a field with a gap between planes is stored."""
    import torch

    from cswap_amd import _lib, api

    L = _lib.lib()
    nz, ny, nx = shape
    x = torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda")
    s = api.cuda_compress(x, 512)
    back = api.cuda_decompress(s, x.shape, 512)
    wide = torch.zeros((nz, ny * nx + 4), device="cuda")
    assert L.cswap_zfp_decompress_f32(s.data_ptr(), nx, ny, nz, 1, nx, ny * nx + 4, 512, wide.data_ptr(),
                                      torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(back.view(torch.int32), wide[:, :ny * nx].reshape(shape).view(torch.int32))
