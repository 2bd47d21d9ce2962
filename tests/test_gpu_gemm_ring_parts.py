"""W8A16 GEMMs of long K split over two or three workgroups per CU: unequal last
parts, the fewest stages of the rule, ragged M and N, and a workspace too
small for the parts (the call then runs whole).  The bar is the ring kernel's:
K 2^-24 sum|x w| for the FP32 sum in any order, plus the BF16 rounding."""
import numpy as np
import pytest
import torch

import refcases as rc
from helpers import to_dev, words

pytestmark = pytest.mark.gpu

# tokens, out_features, in_features; 64 x 64 tiles and parts of 256 CUs:
# 86 in 5, 110 in 4, 130 in 3, 196 in 2, 256 in 2, 192 in 4 (parts of 35 stages)
SIZES = ((65, 2750, 2560), (300, 1400, 2624), (600, 830, 4864), (850, 890, 4864),
         (1001, 1000, 5120), (512, 1500, 8960))


@pytest.mark.parametrize("mnk", SIZES, ids=lambda c: "x".join(map(str, c)))
def test_parts_per_cu(hip, dev, mnk):
    m, n, k = mnk
    print(f"parts {m}x{n}x{k}", flush=True)
    rng = rc.philox(m + n + k)
    x, b = rc.bf16_normal(rng, (m, k)), rc.bf16_normal(rng, (n,))
    q, s = rc.w8a16_synthetic(rng, n, k)
    w = q.astype(np.float64) * np.repeat(rc.bf16_values(s).astype(np.float64), 64, axis=1)
    args = (to_dev(q, dev), to_dev(s, dev), 64, to_dev(b, dev), to_dev(x, dev))
    xv = rc.bf16_values(x).astype(np.float64)
    exp = xv @ w.T + rc.bf16_values(b)
    tol = 2.0**-8 * np.abs(exp) + 1.01 * k * 2.0**-24 * (np.abs(xv) @ np.abs(w).T + 1.0)
    full = torch.zeros(hip.gemm_workspace_bytes(m, n, k), dtype=torch.uint8, device=dev)
    first = None
    for ws in (full, full, full[-(full.numel() * 3 // 4) // 256 * 256:]):
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
        try:
            hip.gemm_w8a16_ws(*args, y, m, n, k, ws)
        except hip.InferError:  # less than the shape's need: refused, nothing written
            assert ws.numel() < full.numel() and torch.isnan(y.float()).all()
            continue
        got = words(y).reshape(m, n)
        assert np.all(np.abs(rc.bf16_values(got) - exp) <= tol)
        if ws.numel() == full.numel():
            np.testing.assert_array_equal(first if first is not None else got, got)
            first = got
    assert not full[:4096].any()  # the counters are back at zero
