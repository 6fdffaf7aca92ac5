"""GEMVs with x in registers (k_gemv_rows) at the edges of its forms: lanes
per row from 1 to 64 with and without idle lanes, one and two blocks per lane,
one and two wave-steps at a time, last rows and steps past the end - the bar
of every GEMV, and nothing stored past the last row."""
from __future__ import annotations

import numpy as np
import pytest

from gguf2bin_amd import attn, hip
from oracle import orc
from test_gpu_matmul import SHAPE, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [orc.T_Q8_0, orc.T_Q4_0, orc.T_Q4_1])
@pytest.mark.parametrize("n", [32, 96, 128, 576, 1024, 2016, 2080, 4096])
def test_gemv_rows_edges(gpu_device, t, n):
    rng = np.random.default_rng(n + t)
    x = rng.standard_normal(n).astype(np.float32)
    x[n // 2] *= 1e3
    with attn.Context(SHAPE) as ctx:
        xd = hip.to_device(x)
        for d in (1, 7, 2049, 13001):
            w = orc.random_weights(rng, t, n, d)
            wd = ctx.weights_upload(w)
            try:
                od = hip.to_device(np.full(d + 8, 7.5, np.float32))
                print(f"[gemv] type={t} n={n} d={d}", flush=True)
                ctx.matmul(od.ptr, xd.ptr, wd, t, n, d)
                ctx.sync()
                out = od.download(np.float32, d + 8)
            finally:
                ctx.weights_free(wd)
            check(out[:d], x, w, t, n, d, f"n={n} d={d}")
            assert np.all(out[d:] == 7.5)
