"""A NaN or an Inf in x of a weight product reaches every output that sums it,
in the forms that hold x as integer digit planes (Q8_0 over many rows; 1024
elements per row on the matrix cores, weights at both alignments) as in the
others."""
from __future__ import annotations

import numpy as np
import pytest

from gguf2bin_amd import attn, hip
from oracle import orc
from test_gpu_matmul import SHAPE, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,n,d,offset", [
    (orc.T_Q8_0, 2048, 32768, 0),  # digit planes on the VALU
    (orc.T_Q8_0, 1024, 32769, 0),  # matrix cores, weights through LDS
    (orc.T_Q4_0, 1024, 32769, 0),
    (orc.T_Q4_1, 1024, 32769, 0),
    (orc.T_Q8_0, 1024, 32769, 4),  # matrix cores, weights straight to registers
    (orc.T_Q4_0, 1024, 32769, 4),
    (orc.T_Q4_1, 1024, 32769, 4),
    (orc.T_Q8_0, 1024, 300, 0),    # x in registers
    (orc.T_Q4_1, 8192, 70, 0),     # a row over four waves
])
def test_non_finite_x(gpu_device, t, n, d, offset):
    rng = np.random.default_rng(n + d + t)
    w = orc.random_weights(rng, t, n, d)
    clean = rng.standard_normal(n).astype(np.float32)
    print(f"[gemv] type={t} n={n} d={d} offset={offset}", flush=True)
    with attn.Context(SHAPE) as ctx:
        wd = ctx.weights_upload(np.concatenate([np.zeros(offset, np.uint8), w]))
        try:
            for bad in (None, np.nan, np.inf):
                x = clean.copy()
                if bad is not None:
                    x[n // 2 + 3] = bad
                xd, od = hip.to_device(x), hip.DeviceBuffer(d * 4)
                ctx.matmul(od.ptr, xd.ptr, wd + offset, t, n, d)
                ctx.sync()
                out = od.download(np.float32, d)
                if bad is None:
                    check(out, x, w, t, n, d, "finite x")
                else:
                    # (an infinite x times the weight's sign; NaN where the
                    # weight is 0 or the form's block unit is NaN)
                    lost = np.isnan(out) if np.isnan(bad) else ~np.isfinite(out)
                    assert lost.all(), f"{bad}: {np.count_nonzero(~lost)} of {d} outputs finite"
        finally:
            ctx.weights_free(wd)
