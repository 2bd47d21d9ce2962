"""Gate|up pairs with K past 1024 (where calls of few rows run on another
kernel than the pair) against 64-bit sums: one, two and more tiles of rows and
columns, K groups of unequal length, biases.

Bar, per output silu(g) u: g and u are BF16 values off the exact sums by dg =
2^-8 |g| + K 2^-24 sum|x w| (du alike), and silu has a slope of at most 1.1;
so 1.1 dg (|u| + du) + |silu(g)| du, plus 2^-8 of the output for its own
rounding and the short SiLU's few FP32 ulps."""
import numpy as np
import pytest
import torch

import model_hip
import refcases as rc
from helpers import to_dev, words

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w8", (True, False), ids=("w8a16", "bf16"))
@pytest.mark.parametrize("tih", ((2, 100, 1088), (17, 4864, 1536), (33, 1000, 1600),
                                 (64, 72, 4864), (65, 2100, 1216), (300, 520, 2112),
                                 (1030, 900, 1536)), ids=lambda c: "x".join(map(str, c)))
def test_gate_up_long_k(hip, dev, tih, w8):
    t, inter, hidden = tih
    print(f"gate|up long K w8={w8} {t}x{inter}x{hidden}", flush=True)
    rng = rc.philox(t + inter + hidden + w8)
    x = rc.bf16_normal(rng, (t, hidden))
    xv = rc.bf16_values(x).astype(np.float64)
    args, sums = [], []
    for _ in range(2):
        b = rc.bf16_normal(rng, (inter,), 0.5)
        if w8:
            q, s = rc.w8a16_synthetic(rng, inter, hidden)
            w = q.astype(np.float64) * np.repeat(rc.bf16_values(s).astype(np.float64), 64, axis=1)
            args += [to_dev(q, dev), to_dev(s, dev), to_dev(b, dev)]
        else:
            wb = rc.bf16_normal(rng, (inter, hidden), 0.02)
            w = rc.bf16_values(wb).astype(np.float64)
            args += [to_dev(wb, dev), to_dev(b, dev)]
        v = xv @ w.T + rc.bf16_values(b)
        sums.append((v, 2.0**-8 * np.abs(v)
                     + 1.01 * hidden * 2.0**-24 * (np.abs(xv) @ np.abs(w).T + 1.0)))
    (g, dg), (u, du) = sums
    silu = g / (1.0 + np.exp(-g))
    tol = 1.1 * dg * (np.abs(u) + du) + np.abs(silu) * du + 2.0**-8 * np.abs(silu * u)
    y = torch.full((t, inter), float("nan"), dtype=torch.bfloat16, device=dev)
    if w8:
        model_hip.gemm_gate_up_silu_w8a16(*args, 64, to_dev(x, dev), y, t, inter, hidden)
    else:
        model_hip.gemm_gate_up_silu_bf16(*args, to_dev(x, dev), y, t, inter, hidden)
    err = np.abs(rc.bf16_values(words(y).reshape(t, inter)) - silu * u)
    assert np.all(err <= tol), float(np.max(err - tol))
