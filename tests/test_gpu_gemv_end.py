"""Weights that end with their allocation: the last block's dwords stay
inside it (a dword-aligned Q4_1 block is five dwords, not the six that a
block at an odd half-word spans)."""
from __future__ import annotations

import numpy as np
import pytest

from gguf2bin_amd import attn, hip
from oracle import orc
from test_gpu_matmul import SHAPE, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [orc.T_Q4_1, orc.T_Q4_0, orc.T_Q8_0])
@pytest.mark.parametrize("n,d", [(4096, 16), (1024, 64), (96, 5)])
def test_matrix_at_the_end_of_its_allocation(gpu_device, t, n, d):
    rng = np.random.default_rng(n + d + t)
    w = orc.random_weights(rng, t, n, d)
    x = rng.standard_normal(n).astype(np.float32)
    size = 2 << 20  # a whole number of pages of every size
    buf = hip.DeviceBuffer(size)
    at = size - w.nbytes
    buf.upload(w, at)
    with attn.Context(SHAPE) as ctx:
        xd, od = hip.to_device(x), hip.DeviceBuffer(4 * d)
        ctx.matmul(od.ptr, xd.ptr, buf.ptr + at, t, n, d)
        ctx.sync()
        check(od.download(np.float32, d), x, w, t, n, d, f"type {t} n {n} d {d}")
