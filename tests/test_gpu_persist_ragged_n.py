"""GPU: the persistent kernels on an N that ends inside a tile (more tiles than CUs): the last columns, the columns right
past which the next row begins, f32 and bf16 C, whole and partial last K tiles, a cut last round, MXFP8; and grouped
problems of such an N with a partial last K tile (full and short tiles).  Rows against the exact oracle with the contract's
bounds; every element equal to the one-tile-per-workgroup kernel where neither splits K."""

import numpy as np
import pytest
import torch

import wave_amd
from oracle import c_oracle
from oracle import mxfp4_oracle as orc
from oracle import mxfp8_oracle as o8
from wave_amd import _lib

from gpu_util import DEV, assert_close, to_gpu

pytestmark = pytest.mark.gpu

NATIVE = {"a_scale_layout": _lib.SCALE_MFMA32, "b_scale_layout": _lib.SCALE_MFMA32}


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(4097, 4104, 1024), (4000, 4344, 1056), (2305, 7688, 1536), (4352, 4136, 4096), (4097, 4348, 768)])
def test_dense(m, n, k, out_dtype):
    if out_dtype == torch.bfloat16 and n % 8:
        n += 4
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=m + n, scale_lo=118, scale_hi=136)
    rows = np.unique(np.r_[0:2, 255:258, m // 2, m - 2:m])
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws, rows=rows)
    gx, gxs, gw, gws = to_gpu(x, orc.mfma32_scale_layout(xs), w_t, orc.mfma32_scale_layout(ws))
    guard = torch.full((m + 1, n), float("nan"), dtype=out_dtype, device=DEV)
    wave_amd.mxfp4_gemm(gx, gxs, gw, gws, guard[:m], variant=_lib.VARIANT_T256x256_W4x2, **NATIVE)
    other = torch.full((m, n), float("nan"), dtype=out_dtype, device=DEV)
    wave_amd.mxfp4_gemm(gx, gxs, gw, gws, other, variant=_lib.VARIANT_T128x128_W2x2, split_k=1, **NATIVE)
    torch.cuda.synchronize()
    assert torch.isnan(guard[m]).all()
    assert_close(guard[torch.from_numpy(rows).to(DEV)].float().cpu().numpy(), ref, out_dtype, f"{m}x{n}x{k}")
    a, b = guard[:m].double(), other.double()
    tol = (2.0 ** -7 * b.abs() if out_dtype == torch.bfloat16 else 0.0) + 2e-6 * b.abs().max()
    assert ((a - b).abs() <= tol).all()


@pytest.mark.parametrize("fmt", [(o8.E4M3, o8.E4M3), (o8.E5M2, o8.E2M1)], ids=["e4m3", "e5m2-e2m1"])
def test_mxfp8(fmt):
    m, n, k = 4100, 4136, 1024
    x, xs, w_t, ws = o8.make_inputs_mxfp8(m, n, k, seed=9, fmt=fmt, scale_lo=120, scale_hi=134)
    gx, gxs, gw, gws = to_gpu(x, xs, w_t, ws)
    out = [torch.full((m, n), float("nan"), dtype=torch.float32, device=DEV) for _ in range(2)]
    wave_amd.mxfp8_gemm(gx, gxs, gw, gws, out[0], elem_format=fmt, variant=_lib.VARIANT_T256x256_W4x2)
    wave_amd.mxfp8_gemm(gx, gxs, gw, gws, out[1], elem_format=fmt, variant=_lib.VARIANT_T128x128_W2x2, workspace=False)
    torch.cuda.synchronize()
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(2880, 2880), (2080, 1024), (2336, 1120)])
@pytest.mark.parametrize("groups", [[520, 700, 256, 0, 257, 63, 64, 65, 900, 511, 31, 1300], [1, 3000, 5, 300, 200, 777]])
def test_grouped(groups, n, k, out_dtype):
    total, e = sum(groups), len(groups)
    rng = np.random.default_rng(n + k + e)
    x = rng.integers(0, 256, size=(total, k // 2), dtype=np.uint8)
    xs = rng.integers(120, 134, size=(total, k // 32), dtype=np.uint8)
    w = rng.integers(0, 256, size=(e, n, k // 2), dtype=np.uint8)
    ws = rng.integers(120, 134, size=(e, n, k // 32), dtype=np.uint8)
    offs = np.concatenate([[0], np.cumsum(groups)]).astype(np.int32)
    gx, gw, goff = to_gpu(x, w, offs)
    gxs = torch.from_numpy(orc.mfma32_scale_layout(xs)).to(DEV)
    gws = torch.from_numpy(np.stack([orc.mfma32_scale_layout(s) for s in ws])).to(DEV)
    out = torch.full((total + 1, n), float("nan"), dtype=out_dtype, device=DEV)
    wave_amd.mxfp4_gemm_grouped(gx, gxs, gw, gws, goff, out[:total], variant=_lib.VARIANT_T256x256_W4x2, **NATIVE)
    torch.cuda.synchronize()
    assert torch.isnan(out[total]).all()
    for g in range(e):
        lo, hi = offs[g], offs[g + 1]
        if lo == hi:
            continue
        rows = np.unique(np.r_[lo, (lo + hi) // 2, hi - 1])
        ref = c_oracle.scaled_gemm_exact(x[rows], w[g], xs[rows], ws[g], rows=np.arange(len(rows)))
        assert_close(out[torch.from_numpy(rows).to(DEV)].float().cpu().numpy(), ref, out_dtype, f"group {g}")
        one = torch.empty(int(hi - lo), n, dtype=out_dtype, device=DEV)
        wave_amd.mxfp4_gemm(gx[lo:hi], torch.from_numpy(orc.mfma32_scale_layout(xs[lo:hi])).to(DEV), gw[g], gws[g], one,
                            variant=_lib.VARIANT_T128x128_W2x2, split_k=1, **NATIVE)
        assert torch.equal(out[lo:hi], one), f"group {g}"
