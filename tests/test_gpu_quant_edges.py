"""GPU, bit-exact against the oracle: the quantiser's lanes beyond the last row, the last scale group and the ids of a gathered
batch (they load the nearest row there is and count as zeros), and the sizes at which its loads and stores change policy."""

import numpy as np
import pytest
import torch

import wave_amd
from oracle import quant_oracle as qo
from wave_amd import _lib

from gpu_util import DEV
from test_gpu_quant import layout_of, make_x

pytestmark = pytest.mark.gpu

LAYOUTS = [_lib.SCALE_ROW_MAJOR, _lib.SCALE_E8M0_SHUFFLE, _lib.SCALE_MFMA32]


@pytest.mark.parametrize("dtype", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("src_rows,rows,k,div", [(1, 1, 32, 1), (3, 33, 288, 2), (40, 31, 512, 1), (65, 130, 992, 2)])
def test_gathered_rows(src_rows, rows, k, div, layout, dtype):
    x, xf = make_x(src_rows, k, rows + k, dtype)
    ids = np.random.default_rng(rows).integers(0, src_rows * div + div, rows).astype(np.int32)  # some beyond the last row
    ids[-1] = src_rows * div - 1
    if rows > 4:
        ids[:3] = (src_rows * div, -1, np.iinfo(np.int32).max)
    q, s = wave_amd.quantize_mxfp4_rows(x, torch.from_numpy(ids).to(DEV), div, scale_layout=layout)
    torch.cuda.synchronize()
    at = ids.astype(np.int64) // div
    known = (ids >= 0) & (at < src_rows)
    want_q, want_s = qo.quantize_mxfp4(np.where(known[:, None], xf[np.where(known, at, 0)], np.float32(0)))
    assert np.array_equal(q.cpu().numpy(), want_q)
    assert np.array_equal(s.cpu().numpy().reshape(-1), layout_of(want_s, layout).reshape(-1)[: s.numel()])


@pytest.mark.parametrize("layout", LAYOUTS)
def test_no_source_row(layout):
    rows, k = 37, 96
    groups = (rows, k // 32) if layout == _lib.SCALE_ROW_MAJOR else (64, 8)
    q = torch.full((rows + 1, k // 2), 0x5A, dtype=torch.uint8, device=DEV)
    s = torch.full((groups[0] * groups[1] + 16,), 0x5A, dtype=torch.uint8, device=DEV)
    ids, x = torch.zeros(rows, dtype=torch.int32, device=DEV), torch.zeros(16, dtype=torch.bfloat16, device=DEV)
    _lib.check(_lib.load().wave_mxfp4_quantize_rows(x.data_ptr(), _lib.IN_BF16, 0, ids.data_ptr(), 1, q.data_ptr(), s.data_ptr(), rows,
                                                    k, layout, torch.cuda.current_stream().cuda_stream), "quantize_rows")
    torch.cuda.synchronize()
    n = groups[0] * groups[1]
    assert (q[:rows] == 0).all() and (q[rows] == 0x5A).all() and (s[:n] == 0).all() and (s[n:] == 0x5A).all()


@pytest.mark.parametrize("dtype,rows", [("bf16", 1535), ("bf16", 1536), ("bf16", 2047), ("f16", 2048), ("f32", 2049)])
def test_sizes_where_the_policies_change(rows, dtype):
    """8192 columns: 6 MB of codes from 1536 rows on, 32 MB of 16-bit elements from 2048."""
    x, xf = make_x(rows, 8192, rows, dtype)
    q, s = wave_amd.quantize_mxfp4(x, scale_layout=_lib.SCALE_MFMA32)
    torch.cuda.synchronize()
    want_q, want_s = qo.quantize_mxfp4(xf)
    assert np.array_equal(q.cpu().numpy(), want_q)
    assert np.array_equal(s.cpu().numpy().reshape(-1), layout_of(want_s, _lib.SCALE_MFMA32).reshape(-1)[: s.numel()])
