"""The C-ABI library must load and export every symbol include/cswap_hip.h
declares (no compute calls: this runs without a GPU)."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_in_header():
    names = set()
    for fn in os.listdir(os.path.join(ROOT, "include")):
        if not fn.endswith(".h"):
            continue
        text = open(os.path.join(ROOT, "include", fn)).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        for m in re.finditer(r"\b([A-Za-z_][A-Za-z0-9_]*)\s*\(", text):
            name = m.group(1)
            if name.startswith("cswap_") or name in REFERENCE_NAMES:
                names.add(name)
    return names


REFERENCE_NAMES = {"PreGPUcompression", "PreAcc", "GPUcompression", "GPUdecompression", "cuda_compress",
                   "cuda_decompress", "compress", "decompress", "setRatio"}


def test_library_exports_every_declared_symbol():
    from cswap_amd import _lib

    L = _lib.lib()
    names = declared_in_header()
    assert len(names) >= 15
    for n in sorted(names):
        assert hasattr(L, n), f"{n} declared in include/ but not exported"
    for n in _lib.declared_symbols():
        assert n in names, f"{n} bound by the loader but not declared in include/"


def test_host_only_entry_points():
    from cswap_amd import _lib

    L = _lib.lib()
    assert L.cswap_abi_version() >= 1
    assert L.cswap_zfp_stream_bytes(32, 32, 4096, 512) == 4194304
    assert L.cswap_zfp_stream_capacity(2, 2, 5, 288) == ((2 * 288 + 63) // 64) * 8
    assert L.cswap_zfp_stream_bytes(2, 2, 5, 288) == (2 * 288 // 64) * 8
    assert L.cswap_zvc_mask_bytes(128 * 256 * 16 * 16, 16384) == 128 * 256 * 16 * 16 // 8
    assert (L.cswap_zvc_chunk_elems(1_000_003, 16384), L.cswap_zvc_chunk_words(1_000_003, 16384),
            L.cswap_zvc_active_chunks(1_000_003, 16384)) == (62, 2, 16130)
    assert L.cswap_strerror(-1) == b"invalid argument"


def test_argument_errors_do_not_launch():
    from cswap_amd import _lib

    L = _lib.lib()
    assert L.cswap_zfp_compress_f32(None, 4, 4, 4, 0, 0, 0, 512, None, None) == -1
    assert L.cswap_zfp_decompress_f32(None, 4, 4, 4, 0, 0, 0, 512, None, None) == -1
    assert L.cswap_zvc_count(None, 10, 16384, None, None) == -1
    assert L.cswap_probe_nnz(None, 0, None, None) == -1


def test_pipeline_kernel_grid_fits_its_scanner_on_any_part():
    """The ZVC pipeline kernel runs one data workgroup per compute unit but one, never more than
    there are tiles, and never more than the 256 tiles its one scanner wavefront serves per step:
    on a part with more compute units than that, the tiles beyond would wait for an offset that
    never comes.  The grid is computed on the host, so parts this build never runs on can be
    asked about."""
    from cswap_amd import _lib

    f = _lib.lib().cswap_test_zvc_stream_groups
    assert f(10000, 256) == 255          # MI355X
    assert f(10000, 304) == 256          # more compute units than the scanner serves per step
    assert f(10000, 1024) == 256
    assert f(100, 256) == 100            # fewer tiles than compute units
    assert f(5, 304) == 5
    assert f(10000, 2) == 1 and f(10000, 1) == 0


def test_stream_handle_without_the_private_short_cut(monkeypatch):
    """The handle of the current stream comes from torch's public interface where the short cut is
    missing, and from the short cut, asked for the current device, where it is there."""
    torch = pytest.importorskip("torch")
    from cswap_amd import api

    class Stream:
        cuda_stream = 1234

    monkeypatch.setattr(torch.cuda, "current_stream", lambda: Stream)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(api, "_raw_stream", None)
    assert api._stream() == 1234
    monkeypatch.setattr(api, "_raw_stream", lambda device: 100 + device)
    assert api._stream() == 103


def test_large_aligned_fields_keep_the_load_hint():
    """The encoder's nontemporal loads are for fields of 128 MiB and more whose rows are aligned and
    whole along x, also where blocks are cut off along y or z; every other field that is not all
    whole blocks of aligned rows takes the kernel for rows at any element."""
    from cswap_amd import _lib

    route = lambda *a: _lib.lib().cswap_test_zfp_encode_route(*a, 0)
    general, rows, hint = 0, 1, 2
    for maxbits in (256, 512, 1024):
        assert route(768, 512, 128, 0, 0, 0, maxbits) == hint            # all whole blocks, 201 MB
        assert route(768, 197, 332, 0, 0, 0, maxbits) == hint            # 197 rows: cut off along y
        assert route(4096, 512, 30, 0, 0, 0, maxbits) == hint            # along z
        assert route(768, 49, 1001, 772, 772 * 49, 0, maxbits) == hint   # along both, pitched
    assert route(768, 197, 332, 0, 0, 0, 520) == rows                    # no hinted variant at this rate
    assert route(771, 197, 332, 772, 772 * 197, 0, 512) == rows          # cut off along x
    assert route(768, 197, 332, 0, 0, 1, 512) == rows                    # rows at any element
    assert route(768, 197, 220, 0, 0, 0, 512) == rows                    # 133 MB: below the hint's size
    assert route(768, 512, 64, 0, 0, 0, 512) == general
    assert route(1, 512, 64, 0, 0, 0, 512) == general


def test_four_lanes_per_block_while_they_fit_at_once():
    """The encoder's form for the smallest fields, where the pair form does not apply: up to 22 wavefronts
    of 16 blocks per compute unit, fewer at the rates where their LDS lets fewer of them run at once
    and one lane per block does not have that limit itself."""
    from cswap_amd import _lib

    def limit(maxbits, cus=256, plane=35):
        """wavefronts per compute unit up to which a field of odd planes runs the form"""
        per_slab = ((plane + 3) // 4) ** 2
        slabs = 1
        while _lib.lib().cswap_test_zfp_encode_route(plane, plane, 4 * slabs, 0, 0, 0, maxbits, cus) == 3:
            slabs += 1
        return (slabs - 1) * per_slab / 16 / cus

    for maxbits in (128, 512, 768, 1920, 2048, 3072, 4096):
        assert 21.5 < limit(maxbits) <= 22, maxbits
    for maxbits, at_least, below in ((1024, 20, 23), (1280, 20, 22), (1536, 18, 20), (1792, 18, 20)):
        assert at_least <= limit(maxbits) < below, maxbits
        assert at_least <= limit(maxbits, cus=128) < below, maxbits
