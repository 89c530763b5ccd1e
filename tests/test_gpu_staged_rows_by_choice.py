"""GPU: row-major scales of more K tiles than the call by name stages (16 to 31 on 64x64, 64x128 and 128x128 tiles, the last of
them on a ring of three; 12 to 15 on 128x192), through the library's own choice, against the exact oracle on a sample of rows;
and, on the CPU, that each of these calls stages them on the tile it is here for."""

import re

import numpy as np
import pytest
import torch

from oracle import c_oracle
from oracle import mxfp4_oracle as orc
from wave_amd import _lib

from gpu_util import assert_close, run_gemm
from test_launch_choice_host import launches  # noqa: F401  (a fixture)

NO_SCRATCH = -2  # (no launch can re-lay the scales, and none adds parts up)
TILES = {"64, 64": (130, 2064), "64, 128": (135, 5552), "128, 128": (260, 6768), "128, 192": (525, 6640)}  # tile: M, N
CASES = [(tile, kt) for tile in TILES for kt in ((12, 14, 15) if tile == "128, 192" else (16, 17, 30, 31))]


@pytest.mark.parametrize("tile,kt", CASES)
@pytest.mark.parametrize("b", [_lib.B_ROW_MAJOR, _lib.B_PRESHUFFLE])
def test_the_library_stages_them(launches, tile, kt, b):  # noqa: F811
    m, n = TILES[tile]
    for out in (_lib.OUT_F32, _lib.OUT_BF16):
        line, = launches([("gemm", m, n, 256 * kt, out, 0, 0, b, 0, 0, NO_SCRATCH)])
        assert re.fullmatch(rf"0 \| \S+ \S+deep_gemm_kernel<\S+DeepCfg<{tile}, .*?>, 2, 4, 4> <\d+,1,1>", line.replace("(anonymous namespace)", "")), line


@pytest.mark.gpu
@pytest.mark.parametrize("tile,kt", CASES)
@pytest.mark.parametrize("b", [_lib.B_ROW_MAJOR, _lib.B_PRESHUFFLE], ids=["row", "preshuffled"])
def test_staged_rows(tile, kt, b):
    (m, n), k = TILES[tile], 256 * kt
    x, xs, w_t, ws = orc.make_inputs(m, n, k, seed=m + kt + b, scale_lo=110, scale_hi=140)
    rows = np.unique(np.r_[0:2, 63:65, m - 2:m])
    ref = c_oracle.scaled_gemm_exact(x, w_t, xs, ws, rows=rows)
    for out_dtype in (torch.float32, torch.bfloat16):
        got = run_gemm(x, xs, orc.b_preshuffle(w_t) if b == _lib.B_PRESHUFFLE else w_t, ws, out_dtype, b_layout=b, workspace=False)
        assert_close(got[rows], ref, out_dtype, f"{m} x {n} x {k}")
