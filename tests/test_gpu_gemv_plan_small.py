"""Grouped W8A16 GEMV plans that move few bytes (one round of loads per wave)
against the CPU oracle: every row-length class (one slab of 1024 weights, two,
three to five, more), its first and last K, rows past a wave's task, with the
descriptors in the kernel arguments (at most eight) and in a device table."""
import pytest

import refcases as rc
from helpers import bf16_out, check_close, to_dev, words

pytestmark = pytest.mark.gpu

# (N, K): K at the edges of the slab classes, N at the edges of a block's rows
SHAPES = [(1, 64), (15, 1024), (17, 1088), (9, 2048), (3, 2112), (5, 4096), (4, 4160), (7, 5120),
          (2, 5184), (6, 8960), (1, 10304)]


@pytest.mark.parametrize("count", [1, 8, 9, 11])
def test_small_plan_matches_oracle(hip, orc, dev, count):
    import torch
    rng = rc.philox(900 + count)
    calls, expected = [], []
    for i, (n, k) in enumerate((SHAPES + SHAPES)[11 - count:11]):
        q, s = rc.w8a16_synthetic(rng, n, k)
        x = rc.bf16_normal(rng, (k,))
        b = rc.bf16_normal(rng, (n,)) if i % 2 else None
        expected.append(orc.w8a16_reference(q, s, 64, b, x)[0][0])
        calls.append((to_dev(q, dev), to_dev(s, dev), 64, None if b is None else to_dev(b, dev),
                      to_dev(x, dev), bf16_out((n,), dev), n, k))
    plan = hip.W8A16GemvPlan(calls)
    try:
        plan.launch()
        torch.cuda.synchronize()
        for c, e in zip(calls, expected):
            check_close(words(c[5]), e, what=f"plan {c[6]}x{c[7]}")
    finally:
        plan.close()
