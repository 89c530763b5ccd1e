"""GPU: the deep-ring kernel through the library's own choice, at the sizes where it can go wrong: edges of its tile
shapes (64x64 .. 256x128) in M and N, one K tile more or less than its ring holds, uneven splits, a partial last K tile,
each way its scales come in (MFMA32 and e8m0_shuffle order in place, row-major staged by the workgroups or re-laid by
the launch in front), both layouts of B.  Against the exact oracle on a sample of rows, with the contract's bounds."""

import numpy as np
import pytest
import torch

from oracle import c_oracle
from oracle import mxfp4_oracle as orc
from wave_amd import _lib

from gpu_util import assert_close, run_gemm

pytestmark = pytest.mark.gpu

CONV = {"row": (_lib.SCALE_ROW_MAJOR, lambda s: s), "e8m0": (_lib.SCALE_E8M0_SHUFFLE, orc.e8m0_shuffle_padded),
        "mfma32": (_lib.SCALE_MFMA32, orc.mfma32_scale_layout)}


def check(m, n, k, scales, out_dtype, preshuffle=False, pad=None, **kw):
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=m * 31 + n + k, scale_lo=118, scale_hi=136)
    rows = np.unique(np.r_[0:min(m, 3), m // 2, max(0, m - 3):m])
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws, rows=rows)
    layout, conv = CONV[scales]
    w_in = orc.b_preshuffle(w_t) if preshuffle else w_t
    if preshuffle:
        kw["b_layout"] = _lib.B_PRESHUFFLE
    got = run_gemm(x, conv(xs), w_in, conv(ws), out_dtype, a_scale_layout=layout, b_scale_layout=layout, **kw)
    assert not np.isnan(got).any()
    assert_close(got[rows], ref, out_dtype, f"{m} x {n} x {k} {scales}")
    return got


@pytest.mark.parametrize("scales", ["row", "e8m0", "mfma32"])
@pytest.mark.parametrize("m", [1, 16, 63, 64, 65, 129, 255, 257, 640])
@pytest.mark.parametrize("n,k", [(1024, 1024), (1048, 1792), (2048, 2048), (1088, 2304)])
def test_small_tiles(m, n, k, scales):
    check(m, n, k, scales, torch.bfloat16 if (m + n) % 2 else torch.float32)


@pytest.mark.parametrize("scales", ["row", "e8m0", "mfma32"])
@pytest.mark.parametrize("m,n,k", [(1000, 1656, 1280), (1000, 4104, 1536), (1537, 1672, 1024), (2047, 4096, 1024),
                                   (129, 16392, 1024), (700, 3592, 3840), (333, 7944, 4096)])
def test_large_tiles(m, n, k, scales):
    check(m, n, k, scales, torch.bfloat16)
    check(m, n, k, scales, torch.float32, preshuffle=n % 16 == 0)


@pytest.mark.parametrize("scales", ["row", "mfma32"])
@pytest.mark.parametrize("m,n,k", [(16, 1024, 9472), (40, 1280, 11008), (128, 1024, 16128), (33, 2056, 8448), (200, 1024, 7424)])
def test_splits(m, n, k, scales):
    a = check(m, n, k, scales, torch.float32)
    b = check(m, n, k, scales, torch.float32, workspace=False)  # no scratch: no split, no launch in front
    assert np.abs(a - b).max() <= 4e-6 * np.abs(a).max()


@pytest.mark.parametrize("tail", [32, 96, 224])
@pytest.mark.parametrize("m,n,k", [(5, 4096, 5888), (48, 1536, 1024), (64, 1024, 12032), (300, 2048, 1536), (900, 3080, 2048)])
def test_partial_last_k_tile(m, n, k, tail):
    check(m, n, k + tail, "mfma32", torch.bfloat16)
    check(m, n, k + tail, "row", torch.float32)


def test_padding_scales_of_a_partial_last_k_tile_may_be_any_finite_value():
    m, n, k = 96, 1536, 1248
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=3, scale_lo=118, scale_hi=136)
    ks, ksp = k // 32, -(-k // 256) * 8
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws, rows=np.arange(m))

    def padded(s):  # the groups past K hold 200, not 0
        return orc.mfma32_scale_layout(np.concatenate([s, np.full((s.shape[0], ksp - ks), 200, np.uint8)], axis=1))

    got = run_gemm(x, padded(xs).reshape(-1), w_t, padded(ws).reshape(-1), torch.float32,
                   a_scale_layout=_lib.SCALE_MFMA32, b_scale_layout=_lib.SCALE_MFMA32)
    assert_close(got, ref, torch.float32, "padding scales")
