"""BF16 GEMMs of one to two 64 x 64 tiles per CU with K whole: the ring's four
slots (K a multiple of the ring and one, two and three stages past it, fewer
stages than slots, ragged M and N, groups) and, past 11/8 tiles per CU at K
over 4096, the register tile.  The bar is the ring kernel's: K 2^-24 sum|x w|
for the FP32 sum in any order, plus the BF16 rounding."""
import numpy as np
import pytest
import torch

import refcases as rc
from helpers import bf16_out, to_dev, words

pytestmark = pytest.mark.gpu

# tokens, out_features, in_features (t64 = 264 .. 512 of 256 CUs)
SIZES = ((65, 8450, 1088), (129, 6000, 1152), (257, 4100, 1216), (300, 4090, 1280),
         (200, 4864, 896), (130, 5600, 64), (66, 8500, 192), (1100, 961, 2112),
         (700, 1536, 4160), (1000, 1473, 4160))


def _expected(x, w, b):
    xv, wv = (rc.bf16_values(a).astype(np.float64) for a in (x, w))
    exp = xv @ wv.T + rc.bf16_values(b)
    k = x.shape[1]
    return exp, (2.0**-8 * np.abs(exp)
                 + 1.01 * k * 2.0**-24 * (np.abs(xv) @ np.abs(wv).T + 1.0))


@pytest.mark.parametrize("mnk", SIZES, ids=lambda c: "x".join(map(str, c)))
def test_deep_tile_sizes(hip, dev, mnk):
    m, n, k = mnk
    print(f"deep tile {m}x{n}x{k}", flush=True)
    rng = rc.philox(m + n + k)
    x, w, b = rc.bf16_normal(rng, (m, k)), rc.bf16_normal(rng, (n, k), 0.02), rc.bf16_normal(
        rng, (n,))
    exp, tol = _expected(x, w, b)
    guard = 64
    buf = torch.full((m * n + 2 * guard,), 0x7FC1, dtype=torch.int16, device=dev)
    y = buf[guard:guard + m * n].view(torch.bfloat16)
    hip.gemm_bf16(to_dev(w, dev), to_dev(b, dev), to_dev(x, dev), y, m, n, k)
    err = np.abs(rc.bf16_values(words(y).reshape(m, n)) - exp)
    assert np.all(err <= tol), float(np.max(err - tol))
    assert torch.all(buf[:guard] == 0x7FC1) and torch.all(buf[guard + m * n:] == 0x7FC1)


def test_deep_tile_group(hip, dev):
    """Three GEMMs of one launch, one of them past the slots by a stage."""
    m, calls, bars = 100, [], []
    rng = rc.philox(9)
    for n, k in ((8000, 1088), (900, 1088), (70, 1152)):
        x, w, b = rc.bf16_normal(rng, (m, k)), rc.bf16_normal(rng, (n, k), 0.02), rc.bf16_normal(
            rng, (n,))
        bars.append(_expected(x, w, b))
        calls.append((to_dev(w, dev), to_dev(b, dev), to_dev(x, dev), bf16_out((m, n), dev), m, n,
                      k))
    plan = hip.GemmPlan(calls)
    try:
        plan.launch()
        torch.cuda.synchronize()
        for c, (exp, tol) in zip(calls, bars):
            assert np.all(np.abs(rc.bf16_values(words(c[3])) - exp) <= tol)
    finally:
        plan.close()
