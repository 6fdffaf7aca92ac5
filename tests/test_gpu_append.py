"""kv_append_rows: runs of rows through k_append_run (16-byte aligned
operands, head_dim 64 / 128 / 256) and row by row through k_append_rows
(anything else): cache bytes equal to the oracle's, nothing written outside
the run."""
from __future__ import annotations

import numpy as np
import pytest

from gguf2bin_amd import attn, hip
from helpers import normed
from oracle import orc
from test_gpu_parity import DevSeq, ashape

pytestmark = pytest.mark.gpu

# rows of 1024, 192, 64, 4096 and 512 floats: 2, 10, 32, 1 and 4 rows per
# workgroup; Q8_0 rows of 68 and 204 bytes leave in 4-byte pieces
SHAPES = {
    "8x128_neox": (16, 8, 128, orc.ARCH_QWEN3),
    "3x64_llama": (9, 3, 64, orc.ARCH_LLAMA),
    "1x64_neox": (2, 1, 64, orc.ARCH_QWEN3),
    "32x128_llama": (32, 32, 128, orc.ARCH_LLAMA),
    "2x256_neox": (4, 2, 256, orc.ARCH_QWEN3),
}


def special(rows, rng):
    """Values at the quantiser's edges among ordinary ones."""
    x = rng.standard_normal(rows).astype(np.float32)
    flat = x.reshape(-1)
    at = rng.permutation(flat.size)[:max(8, flat.size // 50)]
    flat[at] = rng.choice(np.array([0, -0.0, np.nan, np.inf, -np.inf, 1e38, -3e-39, 1e-45, 127.5,
                                    63.5, -0.5], np.float32), at.size)
    return x


@pytest.mark.parametrize("exp", [-140, -100, -91, -89, -20, 0, 60, 99, 101, 110])
def test_append_quotients_at_half_steps(gpu_device, exp):
    """Quotients x / d at and a few ulps beside every half step of the
    quantiser, for d from subnormals to 2^110 and every kind of mantissa: the
    bytes of the division and of lroundf."""
    o = orc.Shape(1, 16, 8, 128, 1e5, orc.ARCH_QWEN3, True)
    rng = np.random.default_rng(exp + 200)
    rows = 64
    n_blk = rows * o.nkv // 32
    with np.errstate(over="ignore", under="ignore"):
        amax = np.ldexp(rng.uniform(1, 2, n_blk), exp + 6).astype(np.float32)
        d = (amax / np.float32(127)).astype(np.float32)
        half = (rng.integers(-127, 127, (n_blk, 32)) + 0.5).astype(np.float32)
        x = (half * d[:, None]).astype(np.float32)
        x = (x.view(np.int32) + rng.integers(-2, 3, x.shape, dtype=np.int32)).view(np.float32)
        x = np.clip(x, -amax[:, None], amax[:, None])
    x[:, 5] = amax
    v = np.ascontiguousarray(x.reshape(rows, o.nkv))
    k = rng.standard_normal(v.shape).astype(np.float32)
    with attn.Context(ashape(o)) as ctx:
        seq = DevSeq(ctx, o, rows)
        okc, ovc = orc.alloc_kv(o, rows)
        try:
            seq.prefill(0, k, v)
            orc.kv_prefill(o, rows, 0, 0, okc, ovc, k, v)
            kc, vc = seq.download()
        finally:
            seq.free()
    assert np.array_equal(vc, ovc)
    assert np.array_equal(kc, okc)


@pytest.mark.parametrize("q8", [True, False])
@pytest.mark.parametrize("name", sorted(SHAPES))
def test_append_rows_vs_oracle(gpu_device, name, q8):
    nh, nkv, hd, arch = SHAPES[name]
    o = orc.Shape(2, nh, nkv, hd, 1e5, arch, q8)
    rng = np.random.default_rng(3)
    cap = 300
    for norm in (None, (1 + 0.25 * rng.standard_normal((2, hd))).astype(np.float32)):
        for misalign in (0, 4):
            with attn.Context(ashape(o)) as ctx:
                if norm is not None:
                    for L in range(2):
                        ctx.set_qk_norm(L, None, norm[L], 1e-6)
                seq = DevSeq(ctx, o, cap)
                okc, ovc = orc.alloc_kv(o, cap)
                try:
                    for L, pos0, n in ((0, 0, 1), (0, 5, 2), (0, 7, 3), (0, 20, 11), (1, 1, 257),
                                       (1, 299, 1)):
                        k, v = (rng.standard_normal((n, o.nkv)).astype(np.float32)
                                for _ in range(2))
                        if n > 3 and norm is None:
                            v = special(v.shape, rng)
                        kd, vd = (hip.DeviceBuffer(k.nbytes + 16) for _ in range(2))
                        kd.upload(k, misalign)
                        vd.upload(v, misalign)
                        print(f"[append] {name} q8={q8} norm={norm is not None} at={misalign} "
                              f"L={L} pos0={pos0} n={n}", flush=True)
                        ctx.kv_append_rows(seq.k, seq.v, cap, L, pos0, n, kd.ptr + misalign,
                                           vd.ptr + misalign)
                        ctx.sync()
                        kn = normed(k, None if norm is None else norm[L], nkv, hd, 1e-6)
                        orc.kv_prefill(o, cap, L, pos0, okc, ovc, kn, v)
                    kc, vc = seq.download()
                finally:
                    seq.free()
            assert np.array_equal(kc, okc), "K bytes"
            assert np.array_equal(vc, ovc), "V bytes"
