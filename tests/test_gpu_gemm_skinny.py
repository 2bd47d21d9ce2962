"""The skinny kernel (32 weight rows for 32 tokens a workgroup, eight waves over
K) at the shapes that reach it: K past 1024, few tokens.  Both of its int8
forms (up to a workgroup per CU, and more: over 8192 outputs), ragged N and
M, waves with no groups, one round of loads and several.

Bar, per output, as for the ring kernel: the FP32 sum of K exact products
within K 2^-24 sum|x w| of the exact one in any order, plus the BF16 rounding.
"""
import numpy as np
import pytest
import torch

import refcases as rc
from helpers import to_dev, words

pytestmark = pytest.mark.gpu

# tokens, out_features, in_features
SIZES = ((2, 33, 1088), (17, 256, 1536), (32, 896, 4864), (5, 2048, 2560), (31, 70, 8960))
W8_SIZES = SIZES + ((2, 8193, 1088), (17, 8960, 1536), (32, 8225, 2112), (64, 2048, 1536),
                    (33, 100, 4864), (100, 1000, 1152))


@pytest.mark.parametrize("w8,mnk", [(True, c) for c in W8_SIZES] + [(False, c) for c in SIZES],
                         ids=lambda c: "x".join(map(str, c)) if isinstance(c, tuple) else
                         ("w8a16" if c else "bf16"))
def test_skinny_sizes(hip, dev, w8, mnk):
    m, n, k = mnk
    print(f"skinny w8={w8} {m}x{n}x{k}", flush=True)
    rng = rc.philox(m + n + k + w8)
    x, b = rc.bf16_normal(rng, (m, k)), rc.bf16_normal(rng, (n,))
    if w8:
        q, s = rc.w8a16_synthetic(rng, n, k)
        w = q.astype(np.float64) * np.repeat(rc.bf16_values(s).astype(np.float64), 64, axis=1)
        args = (to_dev(q, dev), to_dev(s, dev), 64, to_dev(b, dev), to_dev(x, dev))
        run = hip.gemm_w8a16
    else:
        wb = rc.bf16_normal(rng, (n, k), 0.02)
        w = rc.bf16_values(wb).astype(np.float64)
        args, run = (to_dev(wb, dev), to_dev(b, dev), to_dev(x, dev)), hip.gemm_bf16
    xv = rc.bf16_values(x).astype(np.float64)
    exp = xv @ w.T + rc.bf16_values(b)
    tol = 2.0**-8 * np.abs(exp) + 1.01 * k * 2.0**-24 * (np.abs(xv) @ np.abs(w).T + 1.0)
    guard = 64
    buf = torch.full((m * n + 2 * guard,), 0x7FC1, dtype=torch.int16, device=dev)
    y = buf[guard:guard + m * n].view(torch.bfloat16)
    run(*args, y, m, n, k)
    err = np.abs(rc.bf16_values(words(y).reshape(m, n)) - exp)
    assert np.all(err <= tol), float(np.max(err - tol))
    assert torch.all(buf[:guard] == 0x7FC1) and torch.all(buf[guard + m * n:] == 0x7FC1)
