"""The combine of static splits at the edges of its forms, against the oracle:
partials that just fill or just pass one, two, four and eight rounds of a
workgroup's rows, head sizes 64, 128 and 256, a workgroup per quarter of a
head's dims (up to 256 heads) and per head (more), with and without the
softmax weights."""
from __future__ import annotations

import pytest

from oracle import orc
from test_gpu_parity import run_batch_case

pytestmark = pytest.mark.gpu

SPLIT = 8  # positions per split


@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("rounds,extra", [(1, 0), (1, 1), (2, 0), (2, 1), (4, 1), (8, 0), (8, 1)])
def test_few_heads(gpu_device, hd, rounds, extra):
    parts = 4096 // hd * rounds + extra
    o = orc.Shape(1, 8, 4, hd, 1e5, orc.ARCH_QWEN3, False)
    print(f"[combine] hd={hd} partials={parts}", flush=True)
    pos = parts * SPLIT - 3
    sched = {}
    run_batch_case(o, [pos + 1, 30], [pos, 20], seed=41 + rounds, fused=False,
                   want_att=rounds == 1, tune=(SPLIT, 0, 0, 0), sched=sched)
    # (past 512 splits the schedule lengthens them to 9 positions)
    assert sched["max_splits"] == (parts if parts <= 512 else -(-(pos + 1) // 9)), sched


@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("n_seq,att", [(32, False), (33, True), (33, False), (129, False)])
def test_many_heads(gpu_device, hd, n_seq, att):
    o = orc.Shape(1, 8, 4, hd, 1e5, orc.ARCH_QWEN3, False)
    print(f"[combine] hd={hd} heads={8 * n_seq}", flush=True)
    parts = 4096 // hd
    poss = [(parts * SPLIT - 1) * (i + 1) // n_seq for i in range(n_seq)]
    sched = {}
    run_batch_case(o, [p + 1 for p in poss], poss, seed=51, fused=False, want_att=att,
                   tune=(SPLIT, 0, 0, -1), sched=sched)
    assert sched["max_splits"] == parts and not sched["output_in_kernel"], sched
