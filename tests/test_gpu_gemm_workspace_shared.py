"""One workspace, sized for the largest of the Linears that share it: a call
split on the 256 x 128 tile, whose partial tiles fill nearly all of it, and
then one whose parts are counted in its first words.  Every call's outputs
are those it gives on a zeroed workspace of its own."""
import pytest

import refcases as rc
from helpers import to_dev

pytestmark = pytest.mark.gpu

# (w8, tokens, out_features, in_features): wide tiles in two parts (67 MB of
# partials), then 384 ring tiles in parts (more counters than the 256 bytes of
# alignment leave room for), then few tokens in many parts
CALLS = ((True, 2000, 4096, 1024), (False, 1001, 1536, 8960), (True, 33, 896, 4864))


def test_largest_workspace_serves_every_linear(hip, dev):
    import torch
    rng = rc.philox(77)
    runs = []
    for w8, m, n, k in CALLS:
        x = to_dev(rc.bf16_normal(rng, (m, k)), dev)
        if w8:
            q, s = rc.w8a16_synthetic(rng, n, k)
            args, run = (to_dev(q, dev), to_dev(s, dev), 64, None, x), hip.gemm_w8a16_ws
        else:
            args, run = (to_dev(rc.bf16_normal(rng, (n, k), 0.02), dev), None, x), hip.gemm_bf16_ws
        need = hip.gemm_workspace_bytes(m, n, k)
        assert need > 0
        own = torch.zeros(need, dtype=torch.uint8, device=dev)
        first = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
        run(*args, first, m, n, k, own)
        assert torch.isfinite(first.float()).all()
        runs.append((run, args, (m, n, k), need, first))
    shared = torch.zeros(max(r[3] for r in runs), dtype=torch.uint8, device=dev)
    for run, args, (m, n, k), _, first in runs + runs:
        print(f"shared workspace {m}x{n}x{k}", flush=True)
        y = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
        run(*args, y, m, n, k, shared)
        assert torch.equal(y.view(torch.int16), first.view(torch.int16)), (m, n, k)


def test_workspace_without_room_for_counters_is_left_alone(hip, dev):
    """A workspace that holds the wide tile's partials but not the counters
    behind them is accepted as ever, and its first words stay zero."""
    import torch
    m, n, k = CALLS[0][1:]
    rng = rc.philox(78)
    q, s = rc.w8a16_synthetic(rng, n, k)
    args = (to_dev(q, dev), to_dev(s, dev), 64, None, to_dev(rc.bf16_normal(rng, (m, k)), dev))
    tight = 256 * 2 * 256 * 128 * 4 + 256  # 256 tiles, two parts
    ws = torch.zeros(tight, dtype=torch.uint8, device=dev)
    y, plain = (torch.full((m, n), float("nan"), dtype=torch.bfloat16, device=dev)
                for _ in range(2))
    hip.gemm_w8a16_ws(*args, y, m, n, k, ws)
    hip.gemm_w8a16(*args, plain, m, n, k)
    assert not ws[:4096].any()
    a, b = y.float(), plain.float()
    assert ((a - b).abs() <= torch.clamp(0.01 * b.abs(), min=1 / 64)).all()
