"""GPU: MXFP8 and mixed 8-bit / 4-bit operands on the deep-ring kernel through the library's own choice: every pair of
formats, edges of its tiles, odd and even counts of 128-element K tiles, row-major scales staged by the workgroups and
re-laid by the launch in front, splits.  Against the oracle on a sample of rows, with the bounds of the MXFP8 tests
(1e-4 of the largest result: the matrix core aligns the products of one instruction before it adds them)."""

import numpy as np
import pytest
import torch

import wave_amd
from oracle import mxfp8_oracle as o8
from wave_amd import _lib

from gpu_util import DEV, to_gpu

pytestmark = pytest.mark.gpu

PAIRS = [(o8.E4M3, o8.E4M3), (o8.E4M3, o8.E5M2), (o8.E4M3, o8.E2M1), (o8.E5M2, o8.E4M3), (o8.E5M2, o8.E5M2),
         (o8.E5M2, o8.E2M1), (o8.E2M1, o8.E4M3), (o8.E2M1, o8.E5M2)]
IDS = ["e4m3-e4m3", "e4m3-e5m2", "e4m3-e2m1", "e5m2-e4m3", "e5m2-e5m2", "e5m2-e2m1", "e2m1-e4m3", "e2m1-e5m2"]


def check(m, n, k, fmt, out_dtype):
    x, xs, w_t, ws = o8.make_inputs_mxfp8(m, n, k, seed=m + n + k, fmt=fmt, scale_lo=120, scale_hi=134)
    rows = np.unique(np.r_[0:min(m, 3), m // 2, max(0, m - 3):m])
    ref = np.asarray(o8.scaled_gemm_mxfp8(x[rows], w_t, xs[rows], ws, fmt), dtype=np.float64)
    gx, gxs, gw, gws = to_gpu(x, xs, w_t, ws)
    out = torch.full((m, n), float("nan"), dtype=out_dtype, device=DEV)
    wave_amd.mxfp8_gemm(gx, gxs, gw, gws, out, elem_format=fmt)
    tile = torch.full_like(out, float("nan"))
    wave_amd.mxfp8_gemm(gx, gxs, gw, gws, tile, elem_format=fmt, variant=_lib.VARIANT_T128x128_W2x2)
    torch.cuda.synchronize()
    scale = np.abs(ref).max()
    got = out.double().cpu().numpy()
    assert not np.isnan(got).any()
    tol = 1e-4 * scale + (2.0 ** -7 * np.abs(ref) if out_dtype == torch.bfloat16 else 0.0)
    assert (np.abs(got[rows] - ref) <= tol).all(), np.abs(got[rows] - ref).max() / scale
    # every element against the tile kernel: the same instructions, at most regrouped by a split; a bf16 result may
    # round to the neighbour
    full = tile.double().cpu().numpy()
    assert (np.abs(got - full) <= 2e-5 * scale + (2.0 ** -7 * np.abs(full) if out_dtype == torch.bfloat16 else 0.0)).all()


@pytest.mark.parametrize("fmt", PAIRS, ids=IDS)
@pytest.mark.parametrize("m,n,k", [(1, 1024, 1024), (63, 1032, 1152), (65, 1024, 3968), (130, 1544, 2048), (257, 2056, 1280),
                                   (600, 7176, 1024), (700, 6152, 1280)])
def test_formats(m, n, k, fmt):
    check(m, n, k, fmt, torch.float32 if m % 2 else torch.bfloat16)


@pytest.mark.parametrize("fmt", PAIRS[1:3], ids=IDS[1:3])
@pytest.mark.parametrize("m,n,k", [(64, 1024, 8192), (40, 1096, 12416), (129, 1024, 4352), (200, 1160, 16384), (1025, 1024, 5376)])
def test_splits_and_long_k(m, n, k, fmt):
    check(m, n, k, fmt, torch.float32)
