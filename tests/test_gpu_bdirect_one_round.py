"""GPU: the B-direct kernel on 256x256 tiles as the library's own choice for one round of them and less than that (workgroups
without a tile), against the exact oracle on a sample of rows; and, on the CPU, that the calls do reach it."""

import numpy as np
import pytest
import torch

from oracle import c_oracle
from oracle import mxfp4_oracle as orc
from wave_amd import _lib

from gpu_util import assert_close, run_gemm
from test_gpu_deep_ring_by_name import CONV, LAYOUT
from test_launch_choice_host import QUERY, launches  # noqa: F401  (a fixture)

SHAPES = [(500, 16640, 1536), (257, 22784, 2048), (3000, 2816, 1536), (33 * 256, 1024, 1536)]  # 130, 178, 132 and 132 tiles


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("scales,scratch", [("rows", True), ("e8m0", True), ("e8m0", False), ("mfma32", False)])
def test_one_round(m, n, k, scales, scratch):
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=m + k, scale_lo=118, scale_hi=136)
    rows = np.unique(np.r_[0, 255, 256, m - 1])
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws, rows=rows)
    layout, conv = LAYOUT[scales], CONV[scales]
    for out_dtype in (torch.float32, torch.bfloat16):
        got = run_gemm(x, conv(xs), orc.b_preshuffle(w_t), conv(ws), out_dtype, a_scale_layout=layout, b_scale_layout=layout,
                       b_layout=_lib.B_PRESHUFFLE, **({} if scratch else {"workspace": False}))
        assert_close(got[rows], ref, out_dtype, f"{m} x {n} x {k}")


@pytest.mark.parametrize("m,n,k", SHAPES + [(890, 22272, 8704)])
def test_the_library_takes_it(launches, m, n, k):  # noqa: F811
    for layout in (_lib.SCALE_ROW_MAJOR, _lib.SCALE_E8M0_SHUFFLE, _lib.SCALE_MFMA32, _lib.SCALE_PER_ROW):
        b_scale = _lib.SCALE_ROW_MAJOR if layout == _lib.SCALE_PER_ROW else layout
        line, = launches([("gemm", m, n, k, _lib.OUT_BF16, layout, b_scale, _lib.B_PRESHUFFLE, 0, 0, QUERY)])
        assert line.startswith("0 |") and "asym_gemm_kernel" in line, line
    for n2, k2, b in ((n, k, _lib.B_ROW_MAJOR), (n - 16, k, _lib.B_PRESHUFFLE), (n, k + 256, _lib.B_PRESHUFFLE)):
        line, = launches([("gemm", m, n2, k2, _lib.OUT_BF16, 2, 2, b, 0, 0, QUERY)])
        assert line.startswith("0 |") and "asym_gemm_kernel" not in line, line
