"""k_wide on shapes that k_layer also serves (g2b_ctx_tune_kernel(4)), against
the oracle: the whole context in one split up to 128 positions, splits and a
combine from 129 on, one sequence and a ragged batch, with the softmax weights
and the QK norms."""
from __future__ import annotations

import pytest

from oracle import orc
from test_gpu_parity import run_batch_case

pytestmark = pytest.mark.gpu

SHAPES = {
    "qwen3_q8": (16, 8, 128, orc.ARCH_QWEN3, True),
    "qwen3_f32": (16, 8, 128, orc.ARCH_QWEN3, False),
    "smollm2_q8": (9, 3, 64, orc.ARCH_LLAMA, True),
    "smollm2_f32": (9, 3, 64, orc.ARCH_LLAMA, False),
    "llama3_q8": (32, 8, 128, orc.ARCH_LLAMA, True),
}


@pytest.mark.parametrize("name", sorted(SHAPES))
@pytest.mark.parametrize("poss", [[0], [126], [127], [128], [129], [1000], [5, 127, 40],
                                  [128, 3, 64, 300]], ids=str)
@pytest.mark.parametrize("att,norm", [(False, False), (True, True)])
def test_vs_oracle(gpu_device, name, poss, att, norm):
    nh, nkv, hd, arch, q8 = SHAPES[name]
    o = orc.Shape(2, nh, nkv, hd, 1e5, arch, q8)
    norms = None
    if norm:
        norms = ((1 + 0.25 * orc.normal(5, 2 * hd)).reshape(2, hd),
                 (1 + 0.25 * orc.normal(6, 2 * hd)).reshape(2, hd), 1e-6)
    print(f"[wide] {name} {poss} att={att}", flush=True)
    # (rows of 204 bytes: whole capacities of eight rows keep caches aligned)
    caps = [(p // 8 + 1) * 8 for p in poss]
    sched = {}
    run_batch_case(o, caps, poss, seed=61, fused=len(poss) > 1, want_att=att, norms=norms, kernel=4,
                   sched=sched)
    assert sched["kernel"] == "k_wide" and sched["variant"].startswith("k_wide<"), sched
    whole = max(poss) < 128
    assert (sched["max_splits"] == 1) == whole, sched
    # (the weights are normalised by the combine)
    assert sched["output_in_kernel"] == (whole and not att), sched
