"""GPU: row-major scales that the deep-ring kernel's workgroups stage themselves, at the edges of that staging: every count
of K tiles from one up (the K tile and the row of a staged piece come from a multiplication in place of a division), up to
the most that a tile shape takes; and the deeper ring that few rows against a long K run on, on both sides of its border.
Against the exact oracle on a sample of rows, with the contract's bounds."""

import numpy as np
import pytest
import torch

from oracle import c_oracle
from oracle import mxfp4_oracle as orc

from gpu_util import assert_close
from test_gpu_deep_ring_by_name import CONV, E2M1, TILES, deep_ring

pytestmark = pytest.mark.gpu

MOST = [15, 15, 15, 5, 5]  # K tiles that every build of the shape has room for


@pytest.mark.parametrize("shape,kt", [(s, kt) for s in range(5) for kt in sorted({1, 2, 3, 6, 7, 9, 13, 14, 15}) if kt <= MOST[s]])
def test_staged_rows(shape, kt):
    bm, bn = TILES[shape]
    m, n, k = bm + 7, bn + 40, 256 * kt
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=shape * 50 + kt, scale_lo=110, scale_hi=140)
    rows = np.unique(np.r_[0:2, bm - 1:bm + 1, m - 1])
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws, rows=rows)
    got = deep_ring(x, xs, w_t, ws, torch.float32, k, E2M1, E2M1, "rows", 0, shape, 1)
    assert_close(got[rows], ref, torch.float32, f"{m} x {n} x {k}")


@pytest.mark.parametrize("scales", ["mfma32", "e8m0"])
@pytest.mark.parametrize("preshuffled", [False, True], ids=["row", "preshuffled"])
@pytest.mark.parametrize("m,kt,parts", [(1, 17, 1), (16, 17, 1), (16, 16, 1), (17, 17, 1), (32, 24, 1), (33, 17, 1), (9, 39, 2)])
def test_few_rows_and_a_long_k(m, kt, parts, preshuffled, scales):
    n, k = 144, 256 * kt
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=m + kt, scale_lo=118, scale_hi=136)
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws)
    got = deep_ring(x, CONV[scales](xs), orc.b_preshuffle(w_t) if preshuffled else w_t, CONV[scales](ws), torch.float32, k, E2M1,
                    E2M1, scales, int(preshuffled), 0, parts)
    assert_close(got, ref, torch.float32, f"{m} x {n} x {k}")
