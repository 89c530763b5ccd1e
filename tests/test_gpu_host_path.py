"""GPU: the native call path (csrc/wave_host.cpp) against the wrappers' own checks and allocations: what it serves gives
the bits of a call with an explicit scratch, what it does not serve falls through to the wrapper, per stream and with
scratch that has to grow."""

import pytest
import torch

import wave_amd
from oracle import mxfp4_oracle as orc
from wave_amd import _lib

from gpu_util import DEV, to_gpu

pytestmark = pytest.mark.gpu


def operands(m, n, k, seed):
    return to_gpu(*orc.make_inputs(m, n, k, seed=seed, scale_lo=120, scale_hi=130))


@pytest.mark.parametrize("m,n,k", [(1, 256, 512), (200, 136, 512), (384, 1024, 8192)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_native_call_equals_explicit_scratch(m, n, k, dt):
    x, xs, w, ws = operands(m, n, k, m)
    want = torch.empty(m, n, dtype=dt, device=DEV)
    scratch = torch.empty(wave_amd.workspace_bytes(m, n, k), dtype=torch.uint8, device=DEV)
    wave_amd.mxfp4_gemm(x, xs, w, ws, want, workspace=scratch)
    streams = [torch.cuda.current_stream(), torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [torch.empty_like(want) for _ in streams]
    torch.cuda.synchronize()
    for s, o in zip(streams, outs):   # each stream grows a scratch of its own at its first call
        with torch.cuda.stream(s):
            wave_amd.mxfp4_gemm(x, xs, w, ws, o)
            wave_amd.mxfp4_gemm(x, xs, w, ws, o)
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs)


def test_native_path_declines_what_the_wrapper_handles():
    host = _lib.load_host()
    m, n, k = 64, 256, 512
    x, xs, w, ws = operands(m, n, k, 3)
    out = torch.empty(m, n, dtype=torch.bfloat16, device=DEV)
    opts = (0, 0, 0, 0, 0)
    assert host.gemm(x, xs, w, ws, out, *opts)
    strided = torch.cat([x, x], dim=1)[:, :k // 2]
    declined = [(strided, xs, w, ws, out), (x, xs, w, ws, out.to(torch.float16)), (x.cpu(), xs, w, ws, out),
                (x, xs[:-1], w, ws, out), (x, xs, w[:, :-16], ws, out), (x, xs, w, ws, out[:-1]), (x.float(), xs, w, ws, out),
                (None, xs, w, ws, out)]
    assert not any(host.gemm(*a, *opts) for a in declined)
    again = torch.empty_like(out)
    wave_amd.mxfp4_gemm(strided, xs, w, ws, again)   # copied by the wrapper, as before
    wave_amd.mxfp4_gemm(x, xs, w, ws, out)
    assert torch.equal(out, again)
    for bad in declined[1:]:
        with pytest.raises((ValueError, AttributeError)):
            wave_amd.mxfp4_gemm(*bad)
    act = torch.randn(m, k, device=DEV, dtype=torch.bfloat16)
    q, s = wave_amd.quantize_mxfp4(act)
    q2, s2 = wave_amd.quantize_mxfp4(act.t().contiguous().t())
    assert torch.equal(q, q2) and torch.equal(s, s2) and host.quantize(act.t(), 0) is None
    with pytest.raises(ValueError):
        wave_amd.quantize_mxfp4(act[:, :48])


