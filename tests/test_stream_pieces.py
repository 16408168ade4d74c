"""The ZFP stream moved as one run of 16-byte pieces per workgroup: the piece's block, and odd word counts,
streams off 16 bytes and last workgroups that are not full, against the checker."""
import os
import subprocess

import numpy as np
import pytest

import oracle

HERE = os.path.dirname(os.path.abspath(__file__))


def test_block_of_a_piece_is_the_quotient(tmp_path):
    exe = str(tmp_path / "pieces")
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", exe, os.path.join(HERE, "cpp_stream_pieces.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("off", [0, 8])
@pytest.mark.parametrize("words", [1, 2, 3, 6, 7, 8, 12, 16, 22, 40, 64])
@pytest.mark.parametrize("shape", [(4, 4, 4), (4, 8, 252), (12, 7, 512), (40, 52, 340)])
def test_streams_of_any_whole_word_rate_and_alignment(shape, words, off):
    import torch

    from cswap_amd import _lib

    L = _lib.lib()
    nz, ny, nx = shape
    maxbits = 64 * words
    f = np.random.default_rng(words).standard_normal(shape).astype(np.float32)
    want = oracle.zfp_encode3(f, maxbits)
    x = torch.from_numpy(f).cuda()
    nbytes = want.size * 8
    raw = torch.full((nbytes + 64,), 0x5a, dtype=torch.uint8, device="cuda")
    base = raw.data_ptr() + off
    st = torch.cuda.current_stream().cuda_stream
    assert L.cswap_zfp_compress_f32(x.data_ptr(), nx, ny, nz, 0, 0, 0, maxbits, base, st) == 0
    got = raw.cpu().numpy()
    assert np.array_equal(got[off:off + nbytes].view(np.uint64), want)
    assert (got[:off] == 0x5a).all() and (got[off + nbytes:] == 0x5a).all()
    back = torch.empty_like(x)
    assert L.cswap_zfp_decompress_f32(base, nx, ny, nz, 0, 0, 0, maxbits, back.data_ptr(), st) == 0
    assert np.array_equal(back.cpu().numpy().view(np.uint32), oracle.zfp_decode3(want, f.shape, maxbits).view(np.uint32))
