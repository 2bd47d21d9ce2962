"""The prefill GEMM whose operands are loaded straight into an LDS ring, at
the edges of its tiles, K groups and K parts.

Bar, per output: the FP32 sum of K exact products is within K 2^-24 sum|x w|
of the exact one in any order (every partial sum rounds to 2^-24 of at most
the sum of magnitudes), plus the group scaling's fused multiply-add per group,
which the same bound covers, the bias add and the rounding to BF16 (2^-8,
2^-9 to nearest plus what the FP32 error moves across a tie).
"""
import numpy as np
import pytest
import torch

import refcases as rc
from helpers import bf16_out, to_dev, words

pytestmark = pytest.mark.gpu

# tokens, out_features, in_features: one stage (idle K groups), odd N, N and M
# past a tile by one, one K group longer than the other, every tile of the
# size rule, K parts of unequal length, a part of K for the 64 x 32 and the
# 64 x 64 tile
SIZES = ((129, 33, 64), (130, 1025, 128), (257, 130, 192), (513, 1030, 320), (1001, 896, 896),
         (1000, 2560, 192), (1025, 3001, 128), (1500, 3601, 128),
         (200, 70, 1088), (137, 897, 4864), (333, 600, 3136), (700, 300, 3072), (1030, 260, 8960))


@pytest.mark.parametrize("w8", (True, False), ids=("w8a16", "bf16"))
@pytest.mark.parametrize("mnk", SIZES, ids=lambda c: "x".join(map(str, c)))
def test_ring_gemm_edges(hip, dev, mnk, w8):
    m, n, k = mnk
    rng = rc.philox(m + n + k)
    x = rc.bf16_normal(rng, (m, k))
    b = rc.bf16_normal(rng, (n,))
    if w8:
        q, s = rc.w8a16_synthetic(rng, n, k)
        w = q.astype(np.float64) * np.repeat(rc.bf16_values(s).astype(np.float64), 64, axis=1)
        args = (to_dev(q, dev), to_dev(s, dev), 64, to_dev(b, dev), to_dev(x, dev))
        run, run_ws = hip.gemm_w8a16, hip.gemm_w8a16_ws
    else:
        wb = rc.bf16_normal(rng, (n, k), 0.02)
        w = rc.bf16_values(wb).astype(np.float64)
        args = (to_dev(wb, dev), to_dev(b, dev), to_dev(x, dev))
        run, run_ws = hip.gemm_bf16, hip.gemm_bf16_ws
    xv = rc.bf16_values(x).astype(np.float64)
    exp = xv @ w.T + rc.bf16_values(b)
    tol = 2.0**-8 * np.abs(exp) + 1.01 * k * 2.0**-24 * (np.abs(xv) @ np.abs(w).T + 1.0)
    ws_bytes = hip.gemm_workspace_bytes(m, n, k)
    ws = torch.zeros(max(ws_bytes, 16), dtype=torch.uint8, device=dev)
    guard = 64
    buf = torch.full((m * n + 2 * guard,), 0x7FC1, dtype=torch.int16, device=dev)
    first = {}
    for call in ("plain", "ws", "ws", "unaligned"):
        buf.fill_(0x7FC1)
        at = guard + (1 if call == "unaligned" else 0)  # rows of any alignment
        y = buf[at:at + m * n].view(torch.bfloat16)
        if call == "ws":
            run_ws(*args, y, m, n, k, ws)
        else:
            run(*args, y, m, n, k)
        got = words(y).reshape(m, n)
        err = np.abs(rc.bf16_values(got) - exp)
        assert np.all(err <= tol), (call, float(np.max(err - tol)))
        np.testing.assert_array_equal(first.setdefault(call, got), got)  # every launch alike
        assert torch.all(buf[:at] == 0x7FC1) and torch.all(buf[at + m * n:] == 0x7FC1)
    np.testing.assert_array_equal(first["plain"], first["unaligned"])


# tokens, then each GEMM's out_features and in_features: short and long K in
# one launch, descriptors in the kernel's arguments (up to 8) and in a table, a
# plan of 256 tokens or more whose wide-tile launch would not fit the CUs
PLANS = ((3, ((130, 64), (33, 4864))),
         (100, ((130, 64), (896, 896), (896, 4864), (70, 192)) + ((65, 128),) * 5),
         (257, ((4864, 896),) * 8 + ((100, 1536),)))


@pytest.mark.parametrize("w8", (True, False), ids=("w8a16", "bf16"))
@pytest.mark.parametrize("plan", PLANS, ids=lambda p: f"{p[0]}x{len(p[1])}")
def test_ring_plan_edges(hip, dev, plan, w8):
    m, shapes = plan
    rng = rc.philox(m + w8)
    calls, expected = [], []
    for n, k in shapes:
        x = rc.bf16_normal(rng, (m, k))
        b = rc.bf16_normal(rng, (n,))
        if w8:
            q, s = rc.w8a16_synthetic(rng, n, k)
            w = q.astype(np.float64) * np.repeat(rc.bf16_values(s).astype(np.float64), 64, axis=1)
            weight = (to_dev(q, dev), to_dev(s, dev), 64)
        else:
            wb = rc.bf16_normal(rng, (n, k), 0.02)
            w = rc.bf16_values(wb).astype(np.float64)
            weight = (to_dev(wb, dev),)
        calls.append((*weight, to_dev(b, dev), to_dev(x, dev), bf16_out((m, n), dev), m, n, k))
        xv = rc.bf16_values(x).astype(np.float64)
        exp = xv @ w.T + rc.bf16_values(b)
        expected.append((exp, 2.0**-8 * np.abs(exp)
                         + 1.01 * k * 2.0**-24 * (np.abs(xv) @ np.abs(w).T + 1.0)))
    p = hip.GemmPlan(calls)
    try:
        first = None
        for _ in range(2):
            p.launch()
            torch.cuda.synchronize()
            got = [words(c[-4]) for c in calls]
            for g, (exp, tol) in zip(got, expected):
                assert np.all(np.abs(rc.bf16_values(g) - exp) <= tol)
            first = first or got
            for g, f in zip(got, first):
                np.testing.assert_array_equal(g, f)
    finally:
        p.close()
