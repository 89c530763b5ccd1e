"""The C-ABI library without a GPU: it loads, exports every symbol the header
declares, and rejects bad arguments with a status code before touching HIP."""

import ctypes
import os
import re

import pytest

from wave_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "wave_mxfp4.h")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(wave_mxfp[48]_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    names = declared_symbols()
    assert len(names) >= 12
    for name in names:
        assert hasattr(lib, name), name
    assert sorted(_lib.EXPORTS) == names


def test_abi_version_and_status_strings():
    lib = _lib.load()
    assert lib.wave_mxfp4_abi_version() == _lib.ABI_VERSION
    seen = set()
    for code in range(0, -9, -1):
        s = lib.wave_mxfp4_status_string(code).decode()
        assert s and s != "unknown status"
        seen.add(s)
    assert len(seen) == 9
    assert lib.wave_mxfp4_status_string(-99).decode() == "unknown status"


# A 16-byte aligned fake address: validation must reject the call before any
# pointer is dereferenced or any HIP call is made (there is no GPU here).
P = 0x1000


def gemm(lib, a=P, as_=P, b=P, bs=P, c=P, m=64, n=64, k=256, od=0, asl=0, bsl=0, bl=0, split=1, ws=None,
         wsb=0, variant=0):
    return lib.wave_mxfp4_gemm(a, as_, b, bs, c, m, n, k, od, asl, bsl, bl, split, ws, wsb, variant, None)


def test_gemm_argument_validation():
    lib = _lib.load()
    assert gemm(lib, a=None) == _lib.ERR_NULL_POINTER
    assert gemm(lib, as_=None) == _lib.ERR_NULL_POINTER
    assert gemm(lib, b=None) == _lib.ERR_NULL_POINTER
    assert gemm(lib, bs=None) == _lib.ERR_NULL_POINTER
    assert gemm(lib, c=None) == _lib.ERR_NULL_POINTER
    assert gemm(lib, m=-1) == _lib.ERR_BAD_SHAPE
    assert gemm(lib, n=-5) == _lib.ERR_BAD_SHAPE
    assert gemm(lib, k=-32) == _lib.ERR_BAD_SHAPE
    assert gemm(lib, k=48) == _lib.ERR_BAD_SHAPE          # K % 32 != 0
    assert gemm(lib, od=2) == _lib.ERR_BAD_ENUM
    assert gemm(lib, asl=4) == _lib.ERR_BAD_ENUM
    assert gemm(lib, bsl=3) == _lib.ERR_BAD_ENUM          # one scale per row is for A only
    assert gemm(lib, asl=3) == _lib.ERR_WORKSPACE         # ... and needs the workspace
    assert gemm(lib, asl=3, as_=P + 1, ws=P, wsb=16) == _lib.ERR_WORKSPACE
    assert gemm(lib, bsl=-1) == _lib.ERR_BAD_ENUM
    assert gemm(lib, bl=7) == _lib.ERR_BAD_ENUM
    assert gemm(lib, variant=99) == _lib.ERR_BAD_ENUM
    assert gemm(lib, bl=1, n=24) == _lib.ERR_BAD_SHAPE    # preshuffle needs N % 16 == 0
    assert gemm(lib, bl=1, k=96) == _lib.ERR_BAD_SHAPE    # and K % 64 == 0
    assert gemm(lib, a=P + 4) == _lib.ERR_MISALIGNED
    assert gemm(lib, b=P + 8) == _lib.ERR_MISALIGNED
    assert gemm(lib, as_=P + 2) == _lib.ERR_MISALIGNED
    assert gemm(lib, c=P + 8) == _lib.ERR_MISALIGNED
    assert gemm(lib, split=-1) == _lib.ERR_BAD_SPLIT
    assert gemm(lib, k=512, split=4) == _lib.ERR_BAD_SPLIT             # 128 per split < 256
    assert gemm(lib, k=768, split=2) == _lib.ERR_BAD_SPLIT             # 384 not a multiple of 256
    assert gemm(lib, m=128, k=1024, split=2, variant=3) == _lib.ERR_WORKSPACE  # no workspace given
    assert gemm(lib, m=128, k=1024, split=2, variant=3, ws=P, wsb=16) == _lib.ERR_WORKSPACE
    assert gemm(lib, m=128, variant=_lib.VARIANT_SKINNY) == _lib.ERR_UNSUPPORTED
    # empty problems are fine and touch nothing
    assert gemm(lib, m=0, a=None, as_=None, c=None) == _lib.OK
    assert gemm(lib, n=0, b=None, bs=None, c=None) == _lib.OK


def test_grouped_argument_validation():
    lib = _lib.load()

    def grouped(a=P, as_=P, b=P, bs=P, c=P, off=P, e=4, rows=256, n=64, k=256, od=1, asl=0, bsl=0, bl=0,
                variant=0):
        return lib.wave_mxfp4_gemm_grouped(a, as_, b, bs, c, off, e, rows, n, k, od, asl, bsl, bl, variant,
                                           None, 0, None)

    assert grouped(off=None) == _lib.ERR_NULL_POINTER
    assert grouped(a=None) == _lib.ERR_NULL_POINTER
    assert grouped(e=-1) == _lib.ERR_BAD_SHAPE
    assert grouped(k=40) == _lib.ERR_BAD_SHAPE
    assert grouped(od=5) == _lib.ERR_BAD_ENUM
    assert grouped(off=P + 2) == _lib.ERR_MISALIGNED
    assert grouped(variant=_lib.VARIANT_SKINNY) == _lib.ERR_UNSUPPORTED
    assert grouped(e=0) == _lib.OK
    assert grouped(rows=0, a=None, as_=None, c=None) == _lib.OK


def test_aux_argument_validation():
    lib = _lib.load()
    assert lib.wave_mxfp4_to_f32(None, P, 4, 4, None) == _lib.ERR_NULL_POINTER
    assert lib.wave_mxfp4_to_f32(P, P, -1, 4, None) == _lib.ERR_BAD_SHAPE
    assert lib.wave_mxfp4_to_f32(P, P, 0, 4, None) == _lib.OK
    assert lib.wave_mxfp4_e8m0_to_f32(P, None, 4, None) == _lib.ERR_NULL_POINTER
    assert lib.wave_mxfp4_e8m0_to_f32(P, P, -4, None) == _lib.ERR_BAD_SHAPE
    assert lib.wave_mxfp4_dequant(P, P, P, 4, 48, 0, None) == _lib.ERR_BAD_SHAPE
    assert lib.wave_mxfp4_dequant(P, P, P, 4, 64, 3, None) == _lib.ERR_BAD_ENUM
    assert lib.wave_mxfp4_scale_convert(P, 0, P + 256, 3, 4, 4, None) == _lib.ERR_BAD_ENUM
    assert lib.wave_mxfp4_scale_convert(P, 0, None, 2, 4, 4, None) == _lib.ERR_NULL_POINTER
    assert lib.wave_mxfp4_scale_convert(P, 0, P, 2, 4, 4, None) == _lib.ERR_UNSUPPORTED
    assert lib.wave_mxfp4_scale_convert(P, 0, P + 258, 2, 4, 4, None) == _lib.ERR_MISALIGNED
    assert lib.wave_mxfp4_scale_convert(P, 0, P + 256, 2, -1, 4, None) == _lib.ERR_BAD_SHAPE
    assert lib.wave_mxfp4_dequant(P, None, P, 4, 64, 0, None) == _lib.ERR_NULL_POINTER
    assert lib.wave_mxfp4_e8m0_shuffle(None, P, 4, 4, None) == _lib.ERR_NULL_POINTER
    assert lib.wave_mxfp4_b_preshuffle(P, P, 24, 32, None) == _lib.ERR_BAD_SHAPE
    assert lib.wave_mxfp4_b_preshuffle(P, P, 32, 48, None) == _lib.ERR_BAD_SHAPE
    assert lib.wave_mxfp4_b_preshuffle(P + 1, P, 32, 64, None) == _lib.ERR_MISALIGNED
    assert lib.wave_mxfp4_quantize(P, 1, P, P, 4, 48, 0, None) == _lib.ERR_BAD_SHAPE
    assert lib.wave_mxfp4_quantize(P, 3, P, P, 4, 64, 0, None) == _lib.ERR_BAD_ENUM
    assert lib.wave_mxfp4_quantize(P, 1, P, P, 4, 64, 3, None) == _lib.ERR_BAD_ENUM
    assert lib.wave_mxfp4_quantize(P, 1, None, P, 4, 64, 0, None) == _lib.ERR_NULL_POINTER
    assert lib.wave_mxfp4_quantize(P + 8, 1, P, P, 4, 64, 0, None) == _lib.ERR_MISALIGNED
    assert lib.wave_mxfp4_quantize(P, 1, P, P + 2, 4, 64, 1, None) == _lib.ERR_MISALIGNED
    assert lib.wave_mxfp4_quantize(P, 1, P, P, 0, 64, 0, None) == _lib.OK
    assert lib.wave_mxfp4_e8m0_shuffle_bytes(4093, 224) == 4096 * 224
    assert lib.wave_mxfp4_e8m0_shuffle_bytes(33, 9) == 64 * 16


def test_workspace_bytes_of_the_library_own_split_over_random_shapes():
    """The scratch query runs the library's choice of kernel and split on the host: over seeded random shapes of the
    range where it chooses by duration estimates (and around it) the partial sums it asks room for are a whole number
    of M x N f32 parts between 0 and 8, MXFP8 alike, and the answer does not depend on the call order."""
    import numpy as np

    lib = _lib.load()
    rng = np.random.default_rng(3)

    def r256(v):
        return (v + 255) // 256 * 256

    def scales(rows, k):
        return (rows + 31) // 32 * 32 * ((k // 32 + 7) // 8 * 8)

    def parts(rest, m, n):
        """The number of M x N f32 parts `rest` bytes are the (256-byte rounded) room of, or None."""
        return next((c for c in range(0, 17) if rest == (r256(c * m * n * 4) if c else 0)), None)

    seen = {}
    for _ in range(400):
        m = int(2 ** rng.uniform(0, 12.5))
        n = 4 * int(rng.integers(64, 8193))
        k = 32 * int(rng.integers(8, 513))
        for variant in (0, _lib.VARIANT_T128x128_W2x2, _lib.VARIANT_T128x256_W2x2):
            got = lib.wave_mxfp4_workspace_bytes(m, n, k, 0, variant)
            spread, relaid = r256(m * (k // 32)), r256(scales(m, k)) + r256(scales(n, k))
            # with or without room for re-laid scales (the decode kernels read them in place); the library's own
            # choice may also be the persistent kernel, which asks room for the parts of a sparse last round
            c = parts(got - spread - relaid, m, n)
            if c is None:
                c = parts(got - spread, m, n)
            if c is None and variant == 0:
                continue
            assert c is not None and c != 1 and c <= 16, (m, n, k, variant, got)
            seen[(m, n, k, variant)] = got
        if k % 256 == 0:
            got8 = lib.wave_mxfp8_workspace_bytes(m, n, k)
            c8 = parts(got8 - r256(scales(m, k)) - r256(scales(n, k)), m, n)
            assert c8 is not None and c8 != 1 and c8 <= 8, (m, n, k, got8)
    assert len(seen) > 800
    for (m, n, k, variant), got in list(seen.items())[::-1]:
        assert lib.wave_mxfp4_workspace_bytes(m, n, k, 0, variant) == got


def test_workspace_bytes():
    lib = _lib.load()
    scales = 2 * 512 * 32                     # both operands re-laid out as MFMA32
    spread = 512 * 32                         # room to spread per-row A scales over [M, K/32]
    assert lib.wave_mxfp4_workspace_bytes(512, 512, 1024, 1, 0) == scales + spread
    assert lib.wave_mxfp4_workspace_bytes(512, 512, 1024, 4, 3) == 4 * 512 * 512 * 4 + scales + spread
    assert lib.wave_mxfp4_workspace_bytes(16, 512, 1024, 1, 0) == 16 * 32      # skinny kernel: nothing else to stage
    assert lib.wave_mxfp4_workspace_bytes(512, 512, 1024, 1, _lib.VARIANT_NAIVE) == spread
    assert lib.wave_mxfp4_workspace_bytes(-1, 512, 1024, 4, 3) == 0


def test_check_maps_status_to_exceptions():
    with pytest.raises(ValueError, match="K not a multiple of 32"):
        _lib.check(_lib.ERR_BAD_SHAPE, "x")
    with pytest.raises(RuntimeError, match="HIP call failed"):
        _lib.check(_lib.ERR_HIP, "x")
    _lib.check(_lib.OK, "x")


def test_explicit_split_must_leave_no_split_empty():
    """ceil(K / splits) can be a whole number of K tiles while the last splits own none: K = 299 K tiles in 300
    splits of one K tile each.  An empty split would leave its slice of the partial sums unwritten."""
    lib = _lib.load()
    k = 299 * 256
    assert gemm(lib, m=128, k=k, split=300, variant=3, ws=P, wsb=1 << 40) == _lib.ERR_BAD_SPLIT
    assert gemm(lib, m=128, k=k, split=1000, variant=3, ws=P, wsb=1 << 40) == _lib.ERR_BAD_SPLIT
    assert gemm(lib, m=128, k=1024, split=8, variant=3, ws=P, wsb=1 << 40) == _lib.ERR_BAD_SPLIT   # 128 per split


def test_b_direct_variant_rejects_what_it_does_not_take():
    """Variant 7 (A through LDS, preshuffled B straight into registers) is refused, before anything is launched,
    for row-major B, ragged N, an odd number of K tiles, a short K, a split, or row-major scales without scratch."""
    lib = _lib.load()
    v = _lib.VARIANT_T256x256_W1x4_BDIRECT
    ok = dict(m=512, n=512, k=2048, bl=1, asl=2, bsl=2, variant=v)
    assert gemm(lib, **dict(ok, bl=0)) == _lib.ERR_UNSUPPORTED
    assert gemm(lib, **dict(ok, n=384)) == _lib.ERR_UNSUPPORTED
    assert gemm(lib, **dict(ok, k=2304)) == _lib.ERR_UNSUPPORTED      # 9 K tiles
    assert gemm(lib, **dict(ok, k=1024)) == _lib.ERR_UNSUPPORTED
    assert gemm(lib, **dict(ok, split=2)) in (_lib.ERR_UNSUPPORTED, _lib.ERR_WORKSPACE)
    assert gemm(lib, **dict(ok, asl=0)) == _lib.ERR_UNSUPPORTED       # row-major scales need the workspace


@pytest.mark.parametrize("shape", [-1, 1, 3, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("a_fmt,b_fmt", [(0, 0), (1, 0), (0, 2), (2, 1)])
@pytest.mark.parametrize("relayout", [0, 1])
def test_deep_ring_refuses_tiles_that_mxfp8_is_not_built_for(shape, a_fmt, b_fmt, relayout):
    """... before anything is launched into the caller's scratch."""
    lib = _lib.load()
    assert lib.wave_mxfp4_gemm_deep_ring(P, P, P, P, P, 64, 64, 1024, a_fmt, b_fmt, 0, _lib.SCALE_ROW_MAJOR, 0, shape, 1, relayout,
                                         P if relayout else None, 1 << 20, None) == _lib.ERR_UNSUPPORTED


@pytest.mark.parametrize("shape,most", [(0, 15), (1, 15), (2, 15), (3, 5), (4, 5), (8, 15)])
def test_deep_ring_by_name_refuses_more_staged_rows_than_it_names(shape, most):
    lib = _lib.load()
    for kt, parts in ((most + 1, 1), (2 * most + 1, 2)):
        assert lib.wave_mxfp4_gemm_deep_ring(P, P, P, P, P, 64, 64, 256 * kt, 2, 2, 0, _lib.SCALE_ROW_MAJOR, 0, shape, parts, 0, P,
                                             1 << 20, None) == _lib.ERR_UNSUPPORTED
