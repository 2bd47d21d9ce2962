"""The timeline launch of a plan of 256 tokens or more that runs on the ring
kernel: the plan's own outputs bit for bit, and one entry per unit."""
import numpy as np
import pytest

import refcases as rc
from helpers import bf16_out, to_dev, words

pytestmark = pytest.mark.gpu

# tokens and (out_features, in_features): a layer at hidden 896 (descriptors in
# the kernel's arguments, down in parts), nine GEMMs (descriptors in a table)
PLANS = ((700, tuple((n, k) for _, n, k, _ in rc.QWEN_LINEARS)),
         (300, ((1536, 1536), (256, 1536), (256, 1536), (1536, 1536), (8960, 1536), (8960, 1536),
                (1536, 8960), (100, 192), (70, 64))))


@pytest.mark.parametrize("w8", (True, False), ids=("w8a16", "bf16"))
@pytest.mark.parametrize("plan", PLANS, ids=lambda p: f"{p[0]}x{len(p[1])}")
def test_ring_plan_timeline_is_the_plans(hip, dev, plan, w8):
    import torch
    m, shapes = plan
    print(f"ring timeline m={m} w8={w8}", flush=True)
    rng = rc.philox(m + w8)
    calls = []
    for n, k in shapes:
        x = to_dev(rc.bf16_normal(rng, (m, k)), dev)
        if w8:
            q, s = rc.w8a16_synthetic(rng, n, k)
            weight = (to_dev(q, dev), to_dev(s, dev), 64)
        else:
            weight = (to_dev(rc.bf16_normal(rng, (n, k), 0.02), dev),)
        calls.append((*weight, None, x, bf16_out((m, n), dev), m, n, k))
    p = hip.GemmPlan(calls)
    try:
        p.launch()
        torch.cuda.synchronize()
        expected = [words(c[-4]) for c in calls]
        units = p.workgroups()
        stamps = torch.zeros(p.TIMELINE_WORDS * units, dtype=torch.int64, device=dev)
        for _ in range(2):
            for c in calls:
                c[-4].zero_()
            p.launch_timeline(stamps)
            torch.cuda.synchronize()
            for c, e in zip(calls, expected):
                np.testing.assert_array_equal(words(c[-4]), e)
        st = stamps.cpu().numpy().reshape(units, p.TIMELINE_WORDS)
        np.testing.assert_array_equal(st[:, 6] & 0xFFFF, np.arange(units))
        assert np.all(st[:, 0] <= st[:, 1]) and np.all(st[:, 1] <= st[:, 2])
        assert np.all(st[:, 2] <= st[:, 3]) and np.all(st[:, 7] > 0)
        assert set(((st[:, 6] >> 24) & 0xFF).tolist()) <= {0, 1}
        stages = (st[:, 6] >> 16) & 0xFF
        assert stages.min() > 0 and stages.max() <= max(k for _, k in shapes) // 64
        # every stage of every output tile once: 64 x 64 or 128 x 64 tiles
        work = [sum((m + t - 1) // t * ((n + 63) // 64) * (k // 64) for n, k in shapes)
                for t in (64, 128)]
        assert int(stages.sum()) in work
        p.launch()  # the counters are back at zero
        torch.cuda.synchronize()
        for c, e in zip(calls, expected):
            np.testing.assert_array_equal(words(c[-4]), e)
        with pytest.raises(hip.InferError):  # too few entries
            p.launch_timeline(stamps[: p.TIMELINE_WORDS * (units - 1)])
    finally:
        p.close()
