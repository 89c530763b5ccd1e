"""GPU: row-major scales that the deep-ring kernel's workgroups stage themselves, at the edges of that staging: every count
of K tiles from one up (the K tile and the row of a staged piece come from a multiplication in place of a division), up to
the most that the call by name takes; the deeper ring that few rows against a long K run on, on both sides of its border; and the
128x192 tile.
Against the exact oracle on a sample of rows, with the contract's bounds."""

import numpy as np
import pytest
import torch

from oracle import c_oracle
from oracle import mxfp4_oracle as orc

from gpu_util import assert_close, run_gemm
from test_gpu_deep_ring_by_name import CONV, E2M1, TILES, deep_ring

pytestmark = pytest.mark.gpu

MOST = [15, 15, 15, 5, 5]  # (the library's own choice stages up to 31: test_gpu_staged_rows_by_choice.py)


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


@pytest.mark.parametrize("scales,kt,parts,short,preshuffled", [("mfma32", 5, 1, 0, 0), ("mfma32", 8, 3, 64, 1), ("e8m0", 7, 2, 0, 0),
                                                               ("rows", 11, 1, 0, 0), ("rows", 1, 1, 0, 1), ("relaid", 4, 1, 32, 0)])
@pytest.mark.parametrize("m,n", [(127, 200), (129, 384), (257, 184), (40, 576)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_128x192(m, n, scales, kt, parts, short, preshuffled, out_dtype):
    k = 256 * kt - short
    n -= n % 16 if preshuffled else 0
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=m + n + kt, scale_lo=118, scale_hi=136)
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws)
    got = deep_ring(x, CONV[scales](xs), orc.b_preshuffle(w_t) if preshuffled else w_t, CONV[scales](ws), out_dtype, k, E2M1, E2M1,
                    scales, preshuffled, 8, parts)
    assert_close(got, ref, out_dtype, f"{m} x {n} x {k}")


@pytest.mark.parametrize("kt", [12, 14, 15])
@pytest.mark.parametrize("preshuffled", [0, 1])
def test_128x192_stages_up_to_15_k_tiles(kt, preshuffled):
    m, n, k = 135, 240, 256 * kt
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=kt, scale_lo=110, scale_hi=140)
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws)
    for out_dtype in (torch.float32, torch.bfloat16):
        got = deep_ring(x, xs, orc.b_preshuffle(w_t) if preshuffled else w_t, ws, out_dtype, k, E2M1, E2M1, "rows", preshuffled, 8, 1)
        assert_close(got, ref, out_dtype, f"{m} x {n} x {k}")


@pytest.mark.parametrize("m,n", [(40, 1024), (130, 2056), (250, 5000), (520, 5624)])
@pytest.mark.parametrize("kt", [16, 17, 30, 31])
def test_staged_rows_of_a_long_k(m, n, kt):
    """The library's choice of tile and parts; without scratch no launch re-lays the scales and none adds parts up."""
    k = 256 * kt
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=m + kt, scale_lo=118, scale_hi=136)
    rows = np.unique(np.r_[0:2, m // 2, m - 2:m])
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws, rows=rows)
    for kw in ({}, {"workspace": False}):
        got = run_gemm(x, xs, w_t, ws, torch.float32, **kw)
        assert_close(got[rows], ref, torch.float32, f"{m} x {n} x {k} {kw}")
