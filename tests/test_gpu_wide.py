"""k_wide: the shapes k_layer does not take (wide GQA groups, KV heads whose
rows no lane layout of k_layer covers, head_dim 256), against the oracle -
K/V bytes bit for bit, outputs and softmax weights within the bars of every
decode test."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import orc
from test_gpu_parity import run_batch_case

pytestmark = pytest.mark.gpu

# n_heads, n_kv_heads, head_dim, arch, q8: every instance (both formats, head
# sizes 64, 128 and 256, one, two and four sets of four heads, full and ragged
# groups of 1 to 16), one to twenty KV heads (a workgroup each), rows that are
# not whole 16-byte pieces (136 and 68 bytes)
SHAPES = {
    "g5_hd64_q8": (10, 2, 64, orc.ARCH_LLAMA, True),
    "g7_hd64_f32": (14, 2, 64, orc.ARCH_QWEN3, False),
    "g8_hd128_q8": (16, 2, 128, orc.ARCH_QWEN3, True),
    "g8_hd128_f32": (16, 2, 128, orc.ARCH_LLAMA, False),
    "mqa16_hd128_q8": (16, 1, 128, orc.ARCH_QWEN3, True),
    "g9_3kv_hd128_f32": (27, 3, 128, orc.ARCH_QWEN3, False),
    "mha20_hd128_q8": (20, 20, 128, orc.ARCH_LLAMA, True),
    "g6_hd256_q8": (12, 2, 256, orc.ARCH_QWEN3, True),
    "g2_hd256_f32": (8, 4, 256, orc.ARCH_LLAMA, False),
    "mqa16_hd64_q8": (16, 1, 64, orc.ARCH_LLAMA, True),
    "g12_hd64_f32": (24, 2, 64, orc.ARCH_QWEN3, False),
    "g4_hd256_q8": (8, 2, 256, orc.ARCH_LLAMA, True),
    "g16_hd256_q8": (32, 2, 256, orc.ARCH_QWEN3, True),
    "g8_hd256_f32": (16, 2, 256, orc.ARCH_QWEN3, False),
    "g9_hd256_f32": (9, 1, 256, orc.ARCH_LLAMA, False),
}
# positions at the edges of a tile (16), of a round of four waves' tiles (64)
# and of splits, from the first position on
POS = [0, 1, 15, 16, 17, 63, 64, 150]


@pytest.mark.parametrize("name", sorted(SHAPES))
@pytest.mark.parametrize("split,att,norm", [(0, True, False), (0, False, True), (16, False, False),
                                            (37, True, True)])
def test_wide_vs_oracle(gpu_device, name, split, att, norm):
    nh, nkv, hd, arch, q8 = SHAPES[name]
    o = orc.Shape(2, nh, nkv, hd, 1e5, arch, q8)
    norms = None
    if norm:
        norms = ((1 + 0.25 * orc.normal(5, 2 * hd)).reshape(2, hd),
                 (1 + 0.25 * orc.normal(6, 2 * hd)).reshape(2, hd), 1e-6)
    print(f"[wide] {name} split={split} att={att} norm={norm}", flush=True)
    for poss, fused in ((POS, True), ([1], False), ([700], False)):
        sched = {}
        run_batch_case(o, [p + 1 + (p % 3) for p in poss], poss, seed=91 + split, fused=fused,
                       want_att=att, norms=norms, tune=(split, 0, 0, 0) if split else None,
                       sched=sched)
        assert sched["kernel"] == "k_wide", sched
        assert not split or sched["split_len"] == min(split, max(poss) + 1), sched


@pytest.mark.parametrize("name", ["g8_hd128_q8", "mha20_hd128_q8", "g9_3kv_hd128_f32",
                                  "g16_hd256_q8", "g9_hd256_f32", "mqa16_hd64_q8"])
def test_wide_ragged_batch(gpu_device, name):
    """20 sequences of 1 to 2500 positions: the splits of a batch, of every
    length down to none, and partials of several rounds in the combine."""
    nh, nkv, hd, arch, q8 = SHAPES[name]
    o = orc.Shape(1, nh, nkv, hd, 1e5, arch, q8)
    poss = [(2499 * i * i) // 361 for i in range(20)]
    print(f"[wide] ragged batch {name}", flush=True)
    sched = {}
    run_batch_case(o, [p + 1 for p in poss], poss, seed=23, fused=False, want_att=False,
                   sched=sched)
    assert sched["kernel"] == "k_wide", sched


def test_wide_outlier_q(gpu_device):
    """One channel of every head and 32-element block 10^2 times the others
    (what the digit planes must not lose).  Scores reach |s| ~ 250 log2
    units; a few fp32 roundings of one (2^-24 |s| each) move a weight, and the
    output with it, by up to ~6e-5: within the 1e-4 bar."""
    for name in ("g8_hd128_q8", "g8_hd128_f32"):
        nh, nkv, hd, arch, q8 = SHAPES[name]
        o = orc.Shape(2, nh, nkv, hd, 1e6, arch, q8)
        gain = np.ones((nh, hd), np.float32)
        gain[:, 7::32] = 1e2
        run_batch_case(o, [400], [390], seed=17, fused=False, q_gain=gain.reshape(-1),
                       w_as_accurate_as_ref=True)
