"""GPU: calls of few rows at the borders where the library's own choice goes to the deep-ring kernel, against the exact
oracle; and, on the CPU, the kernel on either side of each border."""

import numpy as np
import pytest
import torch

from oracle import c_oracle
from oracle import mxfp4_oracle as orc
from wave_amd import _lib

from gpu_util import assert_close, run_gemm
from test_gpu_deep_ring_by_name import CONV, LAYOUT
from test_launch_choice_host import QUERY, launches  # noqa: F401  (a fixture)

ROW, SHUF = _lib.B_ROW_MAJOR, _lib.B_PRESHUFFLE
# rows, the last shape (N, K tiles) on the deep ring and the first on the other side, B
BORDERS = [
    (7, (4096, 13), (4096, 14), ROW), (16, (6144, 32), (6152, 32), ROW), (3, (16384, 20), (16384, 24), ROW),
    (17, (16384, 5), (16392, 5), ROW), (9, (3080, 35), (8320, 35), ROW), (5, (4096, 9), (4096, 8), SHUF),
    (12, (6144, 29), (6144, 28), SHUF), (1, (8192, 8), (8192, 10), SHUF), (20, (16384, 20), (16400, 20), SHUF),
    (32, (12288, 40), (12320, 40), ROW), (90, (8192, 20), (8224, 20), SHUF), (70, (16384, 6), (16416, 6), ROW),
]
# the same with scales in a blocked order
BLOCKED = [
    (16, (6144, 32), (8192, 32), ROW), (2, (8192, 15), (8192, 16), ROW), (7, (12288, 16), (12288, 20), ROW),
    (1, (9216, 20), (9216, 24), SHUF), (3, (10240, 40), (10240, 48), ROW),
]
# row-major scales and a partial last K tile, which a launch in front re-lays for the deep ring (K tiles in parts of one)
TAILS = [
    (3, (4096, 5.5), (4096, 6.5), ROW), (40, (2048, 10.125), (2048, 11.125), ROW), (16, (8192, 15.125), (8192, 16.125), ROW),
    (1, (11968, 22.875), (11968, 23.125), ROW), (17, (4104, 31.5), (4096, 31.5), ROW), (8, (6144, 39.5), (6144, 38.5), ROW),
    (100, (16384, 7.5), (16392, 7.5), ROW),
]


def gemm(m, shape, b, scales):
    return ("gemm", m, shape[0], int(256 * shape[1]), _lib.OUT_BF16, scales, scales, b, 0, 0, QUERY)


@pytest.mark.parametrize("m,near,far,b,scales", [c + (_lib.SCALE_ROW_MAJOR,) for c in BORDERS] +
                         [c + (s,) for c in BLOCKED for s in (_lib.SCALE_E8M0_SHUFFLE, _lib.SCALE_MFMA32)] +
                         [c + (_lib.SCALE_ROW_MAJOR,) for c in TAILS])
def test_borders(launches, m, near, far, b, scales):  # noqa: F811
    on, off = launches([gemm(m, near, b, scales), gemm(m, far, b, scales)])
    assert on.startswith("0 |") and "deep_gemm_kernel" in on and ("to_mfma32" in on) == (near[1] % 1 != 0), on
    assert off.startswith("0 |") and "deep_gemm_kernel" not in off, off


@pytest.mark.gpu
@pytest.mark.parametrize("m,near,b", [(m, near, b) for m, near, far, b in BORDERS + TAILS] +
                         [(2, (1032, 13), ROW), (130, (12264, 5), ROW)])
def test_row_major_scales(m, near, b):
    n, k = near[0], int(256 * near[1])
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=m + n + k, scale_lo=118, scale_hi=136)
    rows = np.unique(np.r_[0, m // 2, m - 1])
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws, rows=rows)
    for out_dtype in (torch.float32, torch.bfloat16):
        got = run_gemm(x, xs, orc.b_preshuffle(w_t) if b == SHUF else w_t, ws, out_dtype, b_layout=b)
        assert_close(got[rows], ref, out_dtype, f"{m} x {n} x {k}")


@pytest.mark.gpu
@pytest.mark.parametrize("m,near,b", [(m, near, b) for m, near, far, b in BLOCKED])
@pytest.mark.parametrize("scales", ["e8m0", "mfma32"])
def test_blocked_scales(m, near, b, scales):
    n, k = near[0], int(256 * near[1])
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=m + n + k, scale_lo=118, scale_hi=136)
    rows = np.unique(np.r_[0, m // 2, m - 1])
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws, rows=rows)
    for out_dtype in (torch.float32, torch.bfloat16):
        got = run_gemm(x, CONV[scales](xs), orc.b_preshuffle(w_t) if b == SHUF else w_t, CONV[scales](ws), out_dtype,
                       a_scale_layout=LAYOUT[scales], b_scale_layout=LAYOUT[scales], b_layout=b)
        assert_close(got[rows], ref, out_dtype, f"{m} x {n} x {k}")
