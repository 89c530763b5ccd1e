"""GPU: the alignment kernel at the edges of how it ranks the entries - the table length up to which a wave keeps its
places in registers (16 waves x 16 steps x 64 entries = 16384), counts of experts around powers of two (one ballot per
bit of the id), a last step of one entry, ids outside the range (skipped).  Integer work: bit-exact."""

import numpy as np
import pytest
import torch

import wave_amd

from gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1025, 16383, 16384, 16385, 40001])
@pytest.mark.parametrize("experts", [1, 2, 31, 32, 33, 1024])
def test_align_places(n, experts):
    rng = np.random.default_rng(n * 7 + experts)
    ids = rng.integers(0, experts, size=n)
    ids[rng.random(n) < 0.05] = -1
    ids[rng.random(n) < 0.05] = experts
    valid = (ids >= 0) & (ids < experts)
    order = np.flatnonzero(valid)[np.argsort(ids[valid], kind="stable")]
    offsets = np.concatenate([[0], np.cumsum(np.bincount(ids[valid], minlength=experts))])
    want = np.full(n, n)
    want[: len(order)] = order

    def buf(size):
        return torch.full((size,), -7, dtype=torch.int32, device=DEV)

    sorted_ids, expert_ids, total, off = buf(n), buf(n), buf(1), buf(experts + 1)
    wave_amd.moe_align_block_size(torch.from_numpy(ids.astype(np.int32)).to(DEV), experts, 1, sorted_ids, expert_ids, total, off)
    torch.cuda.synchronize()
    assert total.item() == len(order)
    assert np.array_equal(off.cpu().numpy(), offsets)
    assert np.array_equal(sorted_ids.cpu().numpy(), want)
    assert np.array_equal(expert_ids.cpu().numpy()[: len(order)], ids[order])
