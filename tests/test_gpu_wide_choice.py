"""Which calls of k_layer's shapes the automatic choice gives to k_wide, and in
how many splits, on both sides of each line of the rule, against the oracle."""
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
    "mha_f32": (8, 8, 64, orc.ARCH_LLAMA, False),
}
# shape, positions, weights output, kernel[, layers in the one call[, splits]]
CASES = [
    ("qwen3_q8", [127], False, "k_wide"),
    ("qwen3_q8", [700], False, "k_wide"),
    ("qwen3_q8", [700], True, "k_layer"),  # the weights output
    ("smollm2_q8", [0, 127, 64], False, "k_wide"),
    ("smollm2_q8", [511, 128, 4], False, "k_wide"),
    # 2 x 4096 bytes a position: 2048 positions are the 16 MiB of a batch
    ("qwen3_f32", [1023, 1023], False, "k_wide"),
    ("qwen3_f32", [1024, 1023], False, "k_layer"),
    ("qwen3_f32", [8191], False, "k_wide"),
    ("qwen3_f32", [8192], False, "k_wide"),
    ("llama3_q8", [16383], False, "k_wide"),
    ("llama3_q8", [16384], False, "k_tiles"),
    # rows of 204 bytes, more than 64 units below k_layer's shortest split (160):
    # the whole context in one split that writes the output
    ("smollm2_q8", [159] + [40] * 64, False, "k_wide", 1, 1),
    ("smollm2_q8", [159] + [40] * 63, False, "k_wide", 1, 3),
    ("smollm2_q8", [160] + [40] * 64, False, "k_wide", 1, 3),
    ("smollm2_q8", [128, 159, 7, 40, 97], False, "k_wide", 14, 1),
    ("smollm2_f32", [159] + [40] * 64, False, "k_wide", 1, 3),
    # rows of 204 bytes: nine to twelve splits become eight or fewer (whole tiles
    # of 16) once sixteen per unit are more than three workgroups per CU
    ("smollm2_q8", [640] * 16, False, "k_wide", 1, 11),
    ("smollm2_q8", [640] * 17, False, "k_wide", 1, 7),
    ("smollm2_q8", [800] * 24, False, "k_wide", 1, 8),
    ("smollm2_q8", [703], False, "k_wide", 28, 8),
    ("smollm2_f32", [640] * 17, False, "k_wide", 1, 11),
    # one F32 q head of 64 per KV head, below 512 positions: two splits become one
    ("mha_f32", [303] * 20 + [150] * 44, False, "k_wide", 1, 1),
    ("mha_f32", [511] + [300] * 63, False, "k_wide", 1, 1),
    ("mha_f32", [303] + [15] * 20, False, "k_wide", 1, 5),
    # rows of 4 KB, F32: 163840 KB of positions below 128 in one call are the line
    ("qwen3_f32", [127] * 5, False, "k_wide", 32),
    ("qwen3_f32", [127] * 5 + [0], False, "k_short", 32),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(
    [c[0], f"{len(c[1])}x{max(c[1])}", *map(str, c[2:])]))
def test_choice(gpu_device, case):
    (name, poss, att, kernel), layers = case[:4], case[4] if len(case) > 4 else 1
    splits = case[5] if len(case) > 5 else None
    nh, nkv, hd, arch, q8 = SHAPES[name]
    o = orc.Shape(layers, nh, nkv, hd, 1e5, arch, q8)
    # (rows of 204 bytes: whole capacities of eight rows keep caches aligned)
    caps = [(p // 8 + 1) * 8 for p in poss]
    print(f"[choice] {name} {poss} att={att} layers={layers}", flush=True)
    sched = {}
    run_batch_case(o, caps, poss, seed=71, fused=layers > 1, want_att=att, sched=sched)
    assert sched["kernel"] == kernel and sched["variant"].startswith(kernel + "<"), sched
    if splits:
        assert sched["max_splits"] == splits, sched
        assert sched["output_in_kernel"] == (splits == 1), sched
