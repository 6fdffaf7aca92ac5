"""A NaN or an Inf in q: the reference's fp32 scores of that head are not
finite and neither is its softmax (/root/reference/src/l5_model.c:520-562), so
the head's whole output is NaN, and no other head is touched.  Every decode
kernel, those that hold q as integer digit planes (Q8_0 rows) among them, one
split and several, with and without QK-RMSNorm (whose factor spreads the value
over the head), one sequence with such heads beside a clean one."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import normed
from oracle import orc
from test_gpu_parity import DevSeq, ashape

from gguf2bin_amd import attn, hip

pytestmark = pytest.mark.gpu

QWEN3 = (16, 8, 128, orc.ARCH_QWEN3)
CASES = {
    # name: (n_heads, n_kv_heads, head_dim, arch), q8, g2b_ctx_tune_kernel, g2b_ctx_tune or None
    "wide_q8": (QWEN3, True, 4, None),
    "wide_f32": (QWEN3, False, 4, None),
    "wide_q8_llama_hd64": ((9, 3, 64, orc.ARCH_LLAMA), True, 4, None),
    "wide_q8_group8": ((16, 2, 128, orc.ARCH_QWEN3), True, 0, None),
    "wide_q8_hd256": ((4, 1, 256, orc.ARCH_LLAMA), True, 0, None),
    "short_or_layer_q8": (QWEN3, True, 1, None),
    "layer_q8_staged": (QWEN3, True, 1, (64, 0, 2, -1)),
    "layer_q8_half_blocks": ((32, 8, 128, orc.ARCH_LLAMA), True, 1, (64, 0, 0, -1)),
    "layer_q8_hd64": ((6, 2, 64, orc.ARCH_QWEN3), True, 1, (64, 0, -1, -1)),
    "layer_q8_queue": (QWEN3, True, 1, (0, 0, 2, 1)),
    "layer_f32": (QWEN3, False, 1, (64, 0, 0, -1)),
    "tiles_g4": ((32, 8, 128, orc.ARCH_LLAMA), True, 2, (64, 0, 0, -1)),
    "tiles_g3_queue": ((24, 8, 128, orc.ARCH_QWEN3), True, 2, (0, 0, 0, 16)),
}


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("poss", [[40], [40, 700]], ids=str)
@pytest.mark.parametrize("name", sorted(CASES))
def test_head_of_a_non_finite_q_is_nan(gpu_device, name, poss, norm):
    (nh, nkv, hd, arch), q8, kernel, tune = CASES[name]
    o = orc.Shape(1, nh, nkv, hd, 1e5, arch, q8)
    n, eps = len(poss), 1e-6
    caps = [p // 8 * 8 + 8 for p in poss]
    qn = 1 + 0.25 * orc.normal(5, hd) if norm else None
    kn = 1 + 0.25 * orc.normal(6, hd) if norm else None
    q = orc.normal(11, n * o.nq).reshape(n, o.nq)
    k = orc.normal(12, n * o.nkv).reshape(n, o.nkv)
    v = orc.normal(13, n * o.nkv).reshape(n, o.nkv)
    bad = {1: np.nan, nh - 1: np.inf}  # head -> the value of one of its channels
    dirty = q.copy()
    for h, x in bad.items():
        dirty[0, h * hd + hd // 2 + 5] = x
    print(f"[nonfinite] {name} {poss} norm={norm}", flush=True)
    outs, ref = [], None
    with attn.Context(ashape(o)) as ctx:
        ctx.tune_kernel(kernel)
        if tune:
            ctx.tune(*tune)
        if norm:
            ctx.set_qk_norm(0, qn, kn, eps)
        seqs = [DevSeq(ctx, o, c) for c in caps]
        try:
            for i, p in enumerate(poss):
                kp = orc.normal(100 + i, p * o.nkv).reshape(p, o.nkv)
                vp = orc.normal(200 + i, p * o.nkv).reshape(p, o.nkv)
                seqs[i].prefill(0, kp, vp)
                if i == 0:
                    kc, vc = orc.alloc_kv(o, caps[0])
                    orc.kv_prefill(o, caps[0], 0, 0, kc, vc, normed(kp, kn, nkv, hd, eps), vp)
                    ref, _ = orc.attn_layer(o, caps[0], 0, p, kc, vc,
                                            normed(dirty[0], qn, nh, hd, eps),
                                            normed(k[0], kn, nkv, hd, eps), v[0])
            ctx.batch_begin([(p, c, s.k, s.v) for p, c, s in zip(poss, caps, seqs)])
            kd, vd = hip.to_device(k), hip.to_device(v)
            for x in (q, dirty):
                qd = hip.to_device(x)
                ctx.attn_layers(0, 1, qd.ptr, kd.ptr, vd.ptr)
                ctx.sync()
                outs.append(qd.download(np.float32, x.size).reshape(n, nh, hd))
        finally:
            for s in seqs:
                s.free()
    clean, got = outs
    assert np.isfinite(clean).all()
    ref = ref.reshape(nh, hd)
    for i in range(n):
        for h in range(nh):
            if i == 0 and h in bad:
                assert np.isnan(ref[h]).all()
                assert np.isnan(got[i, h]).all(), f"head {h} ({bad[h]}): {got[i, h, :4]}"
            elif "queue" in name or name == "layer_f32":
                # The queue merges pieces in the order of their claims, and an
                # infinite fp32 score has its whole wave rescale: p and the
                # sums of the wave's other heads are rounded at another
                # reference, a few 2^-24 of values whose |v| is below 5.
                assert np.allclose(got[i, h], clean[i, h], rtol=0, atol=1e-5), f"head {h}"
            else:
                assert np.array_equal(got[i, h].view(np.uint32), clean[i, h].view(np.uint32)), \
                    f"head {h}"
