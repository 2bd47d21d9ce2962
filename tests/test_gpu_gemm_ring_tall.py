"""Tall GEMMs (many rows, few columns, K past 1024) on both sides of the rule
that gives them the ring's wider tile.  The bar is the ring kernel's: K 2^-24
sum|x w| for the FP32 sum in any order, plus the BF16 rounding."""
import numpy as np
import pytest
import torch

import refcases as rc
from helpers import to_dev, words

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w8", (True, False), ids=("w8a16", "bf16"))
@pytest.mark.parametrize("mnk", ((1280, 256, 1536), (1281, 256, 1536), (1999, 250, 1536),
                                 (2048, 256, 2560), (2000, 192, 1088)), ids=lambda c: "x".join(map(str, c)))
def test_tall_gemm(hip, dev, mnk, w8):
    m, n, k = mnk
    print(f"tall w8={w8} {m}x{n}x{k}", flush=True)
    rng = rc.philox(m + n + k)
    x, b = rc.bf16_normal(rng, (m, k)), rc.bf16_normal(rng, (n,))
    if w8:
        q, s = rc.w8a16_synthetic(rng, n, k)
        w = q.astype(np.float64) * np.repeat(rc.bf16_values(s).astype(np.float64), 64, axis=1)
        args, run = (to_dev(q, dev), to_dev(s, dev), 64, to_dev(b, dev), to_dev(x, dev)), \
            hip.gemm_w8a16
    else:
        wb = rc.bf16_normal(rng, (n, k), 0.02)
        w = rc.bf16_values(wb).astype(np.float64)
        args, run = (to_dev(wb, dev), to_dev(b, dev), to_dev(x, dev)), hip.gemm_bf16
    xv = rc.bf16_values(x).astype(np.float64)
    exp = xv @ w.T + rc.bf16_values(b)
    tol = 2.0**-8 * np.abs(exp) + 1.01 * k * 2.0**-24 * (np.abs(xv) @ np.abs(w).T + 1.0)
    y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
    run(*args, y, m, n, k)
    assert np.all(np.abs(rc.bf16_values(words(y).reshape(m, n)) - exp) <= tol)
