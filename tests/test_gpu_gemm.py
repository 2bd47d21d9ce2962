"""GPU parity of the MFMA prefill GEMMs (W8A16 and BF16) through the C ABI.

Oracle: the CPU FP32 path (cpu_ops.cpp linear_fp32_batch, 108-123, restated
in oracle/) on the same bytes; for W8A16 on the exactly dequantised weights
q * s.  Bar, per output: |a - e| <= max(1e-2 |e|, 1e-3 rms(e)) (the BASELINE
north star) and at least 95 % of the BF16 words identical to bf16(e) (the
MFMA sums in FP32 like the oracle, in another order).  Dequantisation is
checked bitwise: with one-hot activation rows the GEMM returns
bf16(q[n, j] * s[n, j / 64]) exactly.
"""
import numpy as np
import pytest

import refcases as rc
from helpers import bf16_out, check_close, to_dev, words

pytestmark = pytest.mark.gpu

TILES = range(6)  # infer_hip_gemm_tile_count()
RAGGED = ((33, 100, 128), (130, 70, 192), (2, 128, 64), (200, 260, 1024), (65, 33, 4864))


def test_tile_count_matches(hip):
    assert hip.gemm_tile_count() == len(TILES) == len(hip.GEMM_TILES)


@pytest.mark.parametrize("m", (32, 128, 512))
@pytest.mark.parametrize("shape", rc.QWEN_LINEARS, ids=lambda s: s[0])
def test_config3_w8a16_gemm_synthetic(hip, orc, dev, m, shape):
    # Config 3: q ~ U{-127..127}, s = bf16(|N(0,.02)|/127), X = bf16(N(0,1)),
    # seed 3.
    name, n, k, _ = shape
    rng = rc.philox(3 + 100 * m + rc.QWEN_LINEARS.index(shape))
    q, s = rc.w8a16_synthetic(rng, n, k)
    x = rc.bf16_normal(rng, (m, k))
    exp = orc.linear_fp32_batch(orc.dequant_w8a16(q, s), None, rc.bf16_values(x))
    y = bf16_out((m, n), dev)
    hip.gemm_w8a16(to_dev(q, dev), to_dev(s, dev), 64, None, to_dev(x, dev), y, m, n, k)
    stats = check_close(words(y), exp, what=f"gemm_w8a16 {name} M={m}")
    assert stats["bit_identical"] > 0.95, stats


@pytest.mark.parametrize("m", (32, 128, 512))
@pytest.mark.parametrize("shape", rc.QWEN_LINEARS, ids=lambda s: s[0])
def test_config3_bf16_gemm_synthetic(hip, orc, dev, m, shape):
    # Config 3, W16A16 comparison: W = bf16(N(0, 0.02)), X = bf16(N(0,1)).
    name, n, k, _ = shape
    rng = rc.philox(3 + 100 * m + 10 * rc.QWEN_LINEARS.index(shape))
    w = rc.bf16_normal(rng, (n, k), 0.02)
    x = rc.bf16_normal(rng, (m, k))
    exp = orc.linear_fp32_batch(rc.bf16_values(w), None, rc.bf16_values(x))
    y = bf16_out((m, n), dev)
    hip.gemm_bf16(to_dev(w, dev), None, to_dev(x, dev), y, m, n, k)
    stats = check_close(words(y), exp, what=f"gemm_bf16 {name} M={m}")
    assert stats["bit_identical"] > 0.95, stats


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("mnk", RAGGED, ids=lambda c: "x".join(map(str, c)))
def test_every_tile_on_ragged_shapes(hip, orc, dev, tile, mnk):
    # M and N not multiples of any tile; bias on.
    m, n, k = mnk
    rng = rc.philox(70 + tile)
    q, s = rc.w8a16_synthetic(rng, n, k)
    x = rc.bf16_normal(rng, (m, k))
    b = rc.bf16_normal(rng, (n,))
    exp, _ = orc.w8a16_reference(q, s, 64, b, x)
    y = bf16_out((m, n), dev)
    hip.gemm_w8a16_tile(to_dev(q, dev), to_dev(s, dev), 64, to_dev(b, dev), to_dev(x, dev),
                        y, m, n, k, tile)
    check_close(words(y), exp, what=f"w8a16 tile {tile}")

    w = rc.bf16_normal(rng, (n, k), 0.02)
    expb = orc.bf16_linear_reference(w, b, x)
    yb = bf16_out((m, n), dev)
    hip.gemm_bf16_tile(to_dev(w, dev), to_dev(b, dev), to_dev(x, dev), yb, m, n, k, tile)
    check_close(words(yb), expb, what=f"bf16 tile {tile}")


@pytest.mark.parametrize("tile", TILES)
def test_gemm_dequant_is_bit_exact(hip, dev, tile):
    # Row i of X is e_{j_i}: Y[i, n] = bf16(q[n, j_i] * s[n, j_i / 64]) with
    # no rounding before the final BF16 one, for every chunk slot, group
    # edge and lane half of the staged columns.
    n, k = 160, 1216
    rng = rc.philox(90 + tile)
    q, s = rc.w8a16_synthetic(rng, n, k)
    q[0, :] = 127
    q[1, :] = -127
    cols = sorted({0, 1, 7, 8, 15, 16, 31, 32, 33, 63, 64, 65, 127, 128, 600, 1151, 1152,
                   1200, 1215})
    x = np.zeros((len(cols), k), np.uint16)
    for i, j in enumerate(cols):
        x[i, j] = 0x3F80  # BF16 1.0
    y = bf16_out((len(cols), n), dev)
    hip.gemm_w8a16_tile(to_dev(q, dev), to_dev(s, dev), 64, None, to_dev(x, dev), y,
                        len(cols), n, k, tile)
    got = words(y)
    for i, j in enumerate(cols):
        expect = rc.bf16_words((q[:, j].astype(np.float32)
                                * rc.bf16_values(s[:, j // 64])).astype(np.float32))
        np.testing.assert_array_equal(got[i], expect, err_msg=f"column {j}")


def test_gemm_row_matches_gemv(hip, orc, dev):
    # tools/linear_benchmark.cpp:533-542 / test_cuda.cpp:604-608: the GEMM's
    # row 0 agrees with the GEMV on the same row, within the reference bound.
    m, n, k = 128, 4864, 896
    rng = rc.philox(99)
    q, s = rc.w8a16_synthetic(rng, n, k)
    x = rc.bf16_normal(rng, (m, k))
    dq, ds, dx = to_dev(q, dev), to_dev(s, dev), to_dev(x, dev)
    y = bf16_out((m, n), dev)
    hip.gemm_w8a16(dq, ds, 64, None, dx, y, m, n, k)
    y1 = bf16_out((n,), dev)
    hip.gemv_w8a16(dq, ds, 64, None, to_dev(x[0], dev), y1, n, k)
    g, v = rc.bf16_values(words(y)[0]), rc.bf16_values(words(y1))
    assert np.all(np.abs(g - v) <= np.maximum(1.0 / 64, 0.01 * np.abs(v)))


# ------------------------------------------------------ grouped GEMM plan --

@pytest.mark.parametrize("m", (130, 300))
@pytest.mark.parametrize("w8", (True, False), ids=("w8a16", "bf16"))
def test_gemm_plan_matches_single_calls(hip, orc, dev, w8, m):
    # The seven Qwen Linears at M = 130 or 300 (ragged last M tiles; plans
    # with every M >= 256 use the 8-wave 256 x 128 tile, others 64 x 64)
    # plus ragged-N descriptors with bias, in one launch.  At M = 130 the
    # shortest reduction (K = 192, 3 stages) makes the plan split every K >=
    # 576 into parts of 8 stages: split-K hand-offs through arrival counters
    # (up to 10 parts for K = 4864).  At M = 300 the wide-tile plan raises
    # the part length until its units fit the CUs, and split tiles (down and
    # the K = 2048 ragged one, which has a bias) go through the separate
    # reduction launch.  Each output equals the oracle, agrees with the
    # single call (same tile; split tiles add their parts in another order)
    # within the reference's GEMV-vs-GEMM bound max(1/64, 1 %)
    # (test_cuda.cpp:604-608), and is bit-identical across launches (the
    # parts are summed in a fixed order whichever finishes last).
    import torch
    rng = rc.philox(110 + w8 + m)
    tile = 5 if m >= 256 else 3  # the plan's tile, for the single calls
    calls, expected, singles = [], [], []
    extra = (("ragged", 70, 192, True), ("ragged_long", 70, 2048, True))
    for (name, n, k, bias) in rc.QWEN_LINEARS + extra:
        x = rc.bf16_normal(rng, (m, k))
        b = rc.bf16_normal(rng, (n,)) if bias else None
        dx, db = to_dev(x, dev), (to_dev(b, dev) if bias else None)
        y, y1 = bf16_out((m, n), dev), bf16_out((m, n), dev)
        if w8:
            q, s = rc.w8a16_synthetic(rng, n, k)
            exp, _ = orc.w8a16_reference(q, s, 64, b, x)
            dq, ds = to_dev(q, dev), to_dev(s, dev)
            calls.append((dq, ds, 64, db, dx, y, m, n, k))
            hip.gemm_w8a16_tile(dq, ds, 64, db, dx, y1, m, n, k, tile)
        else:
            w = rc.bf16_normal(rng, (n, k), 0.02)
            exp = orc.bf16_linear_reference(w, b, x)
            dw = to_dev(w, dev)
            calls.append((dw, db, dx, y, m, n, k))
            hip.gemm_bf16_tile(dw, db, dx, y1, m, n, k, tile)
        expected.append(exp)
        singles.append(y1)
    plan = hip.GemmPlan(calls)
    try:
        assert plan.flops == sum(2.0 * c[-3] * c[-2] * c[-1] for c in calls)
        first = None
        for _ in range(3):  # later launches rewrite the same outputs
            plan.launch()
            torch.cuda.synchronize()
            got = [words(c[5] if w8 else c[3]) for c in calls]
            for g, e, y1 in zip(got, expected, singles):
                check_close(g, e, what="gemm plan")
                a, b1 = rc.bf16_values(g), rc.bf16_values(words(y1))
                assert np.all(np.abs(a - b1) <= np.maximum(1.0 / 64, 0.01 * np.abs(b1)))
            if first is None:
                first = got
            for g, f in zip(got, first):
                np.testing.assert_array_equal(g, f)
        if tile != 5:
            with pytest.raises(hip.InferError):  # the timeline is the wide tile's
                plan.workgroups()
            return
        # The timeline launch computes the same outputs and stamps every
        # workgroup: each logical unit once, its four times in order.
        wg = plan.workgroups()
        words_per = hip.GemmPlan.TIMELINE_WORDS
        stamps = torch.zeros(words_per * wg, dtype=torch.int64, device=dev)
        for c in calls:
            (c[5] if w8 else c[3]).zero_()
        plan.launch_timeline(stamps)
        torch.cuda.synchronize()
        for g, f in zip([words(c[5] if w8 else c[3]) for c in calls], first):
            np.testing.assert_array_equal(g, f)
        st = stamps.cpu().numpy().reshape(wg, words_per)
        assert sorted((st[:, 6] & 0xFFFF).tolist()) == list(range(wg))
        assert np.all(st[:, 0] <= st[:, 1]) and np.all(st[:, 1] <= st[:, 2])
        assert np.all(st[:, 2] <= st[:, 3]) and np.all(st[:, 7] > 0)
        kinds = set(((st[:, 6] >> 24) & 0xFF).tolist())
        assert kinds == {0, 1}  # whole tiles and split parts
        assert np.all((st[:, 6] >> 16) & 0xFF > 0)
        parts = ((st[:, 6] >> 24) & 0xFF) == 1
        if np.any(st[parts, 8] != 0):  # hand-off inside the launch: its times in order
            h = st[parts]
            assert np.all(h[:, 2] <= h[:, 8]) and np.all(h[:, 8] <= h[:, 9])
            assert np.all(h[:, 9] <= h[:, 10]) and np.all(h[:, 10] <= h[:, 3])
        with pytest.raises(hip.InferError):  # too few slots
            plan.launch_timeline(stamps[: words_per * (wg - 1)])
    finally:
        plan.close()


def test_gemm_plan_rejects_unsupported_descriptors(hip, dev):
    q = to_dev(np.zeros((4, 70), np.int8), dev)
    s = to_dev(np.zeros((4, 2), np.uint16), dev)
    x = to_dev(np.zeros((2, 70), np.uint16), dev)
    y = bf16_out((2, 4), dev)
    with pytest.raises(hip.InferError):  # K % 64 != 0
        hip.GemmPlan([(q, s, 64, None, x, y, 2, 4, 70)])
    q64 = to_dev(np.zeros((4, 64), np.int8), dev)
    x64 = to_dev(np.zeros((2, 64), np.uint16), dev)
    w64 = to_dev(np.zeros((4, 64), np.uint16), dev)
    with pytest.raises(hip.InferError):  # group size
        hip.GemmPlan([(q64, s, 32, None, x64, y, 2, 4, 64)])
    with pytest.raises(hip.InferError):  # one token is a GEMV
        hip.GemmPlan([(q64, s, 64, None, x64, y, 1, 4, 64)])
    with pytest.raises(hip.InferError):  # mixed weight types
        hip.GemmPlan([(q64, s, 64, None, x64, y, 2, 4, 64), (w64, None, x64, y, 2, 4, 64)])


@pytest.mark.parametrize("w8", [True, False], ids=["w8a16", "bf16"])
def test_lone_gemm_with_workspace_splits_long_k(hip, orc, dev, w8):
    """infer_hip_gemm_*_ws: down_proj (K = 4864) at M = 2 .. 512 splits K
    over the workspace; every call sharing one workspace (sized for M <= 512,
    zeroed once) meets the oracle bar, a shape that never splits needs none,
    and a workspace smaller than a call needs is rejected."""
    import torch
    n, k = 896, 4864
    need = hip.gemm_workspace_bytes(512, n, k)
    assert need > 0
    assert hip.gemm_workspace_bytes(512, 896, 896) == 0      # 14 stages: never split
    assert hip.gemm_workspace_bytes(1, n, k) == 0            # one token: the GEMV
    ws = torch.zeros(need // 4 + 1, dtype=torch.int32, device=dev)
    rng = rc.philox(4864 + w8)
    if w8:
        q, s = rc.w8a16_synthetic(rng, n, k)
        wd, sd = to_dev(q, dev), to_dev(s, dev)
        weights = orc.dequant_w8a16(q, s)
    else:
        w = rc.bf16_normal(rng, (n, k), 0.02)
        wd = to_dev(w, dev)
        weights = rc.bf16_values(w)
    b = rc.bf16_normal(rng, (n,))
    for m in (2, 32, 128, 512, 65):
        print(f"gemm ws w8={w8} M={m}", flush=True)
        x = rc.bf16_normal(rng, (m, k))
        exp = orc.linear_fp32_batch(weights, rc.bf16_values(b), rc.bf16_values(x))
        y = bf16_out((m, n), dev)
        if w8:
            hip.gemm_w8a16_ws(wd, sd, 64, to_dev(b, dev), to_dev(x, dev), y, m, n, k, ws)
        else:
            hip.gemm_bf16_ws(wd, to_dev(b, dev), to_dev(x, dev), y, m, n, k, ws)
        stats = check_close(words(y), exp, what=f"gemm ws w8={w8} M={m}")
        assert stats["bit_identical"] > 0.95, stats
    # A workspace too small for the call's shape is rejected.
    small = ws[:4]
    x = to_dev(rc.bf16_normal(rng, (128, k)), dev)
    with pytest.raises(hip.InferError) as err:
        if w8:
            hip.gemm_w8a16_ws(wd, sd, 64, None, x, bf16_out((128, n), dev), 128, n, k, small)
        else:
            hip.gemm_bf16_ws(wd, None, x, bf16_out((128, n), dev), 128, n, k, small)
    assert err.value.status == hip.INVALID_ARGUMENT and "workspace" in str(err.value)


# ---------------------------------------------------- GEMMs of few tokens --
#
# Lone calls (automatic tile) of few tokens run the ring kernel, or past K =
# 1024 the skinny kernel: each workgroup streams 32 weight rows once, its eight
# waves splitting K and summing their accumulators in LDS
# (tests/test_gpu_gemm_skinny.py has that kernel's own sizes).  Their MFMA
# fragments per group are the 64 x 64 tile's, so with exact sums they agree
# with the tile bit for bit; otherwise only the association of the sums
# differs.  Plans never take the skinny kernel.

def test_skinny_gemm_dequant_is_bit_exact(hip, dev):
    """One-hot activation rows (19 tokens) through the automatic path: Y[i,
    n] = bf16(q[n, j_i] s[n, j_i / 64]) exactly, for every chunk slot, lane
    half, group edge and wave of the K split (K = 1216: 19 groups over 8
    waves of 3, the last wave with none)."""
    n, k = 160, 1216
    rng = rc.philox(91)
    q, s = rc.w8a16_synthetic(rng, n, k)
    q[0, :] = 127
    q[1, :] = -127
    cols = sorted({0, 1, 7, 8, 15, 16, 31, 32, 33, 63, 64, 65, 127, 128, 600, 1151, 1152,
                   1200, 1215})
    x = np.zeros((len(cols), k), np.uint16)
    for i, j in enumerate(cols):
        x[i, j] = 0x3F80  # BF16 1.0
    y = bf16_out((len(cols), n), dev)
    hip.gemm_w8a16(to_dev(q, dev), to_dev(s, dev), 64, None, to_dev(x, dev), y, len(cols), n, k)
    got = words(y)
    w = rc.bf16_words((rng.integers(-127, 128, size=(n, k)) / 64.0).astype(np.float32))
    yb = bf16_out((len(cols), n), dev)
    hip.gemm_bf16(to_dev(w, dev), None, to_dev(x, dev), yb, len(cols), n, k)
    gotb = words(yb)
    for i, j in enumerate(cols):
        expect = rc.bf16_words((q[:, j].astype(np.float32)
                                * rc.bf16_values(s[:, j // 64])).astype(np.float32))
        np.testing.assert_array_equal(got[i], expect, err_msg=f"w8a16 column {j}")
        np.testing.assert_array_equal(gotb[i], w[:, j], err_msg=f"bf16 column {j}")


SKINNY_SHAPES = ((2, 100, 128), (17, 33, 192), (32, 70, 4864), (32, 4864, 896), (5, 896, 896),
                 (31, 257, 1024),
                 # more rows than a token tile of 32; the skinny kernel at K = 4864
                 (64, 896, 896), (100, 130, 1024), (128, 896, 4864), (77, 1000, 128))


@pytest.mark.parametrize("mnk", SKINNY_SHAPES, ids=lambda c: "x".join(map(str, c)))
@pytest.mark.parametrize("w8", [True, False], ids=["w8a16", "bf16"])
def test_skinny_gemm_matches_oracle_and_tile(hip, orc, dev, mnk, w8):
    """Ragged M and N, bias on, K from 2 to 76 groups (the ring kernel up to 16,
    the skinny kernel past them): the oracle's bar, and the 64 x 64 tile's
    result within the reference's GEMV-vs-GEMM bound max(1/64, 1 %)."""
    m, n, k = mnk
    print(f"skinny w8={w8} {m}x{n}x{k}", flush=True)
    rng = rc.philox(1000 + m + n + k + w8)
    x = rc.bf16_normal(rng, (m, k))
    b = rc.bf16_normal(rng, (n,))
    dx, db = to_dev(x, dev), to_dev(b, dev)
    y, yt = bf16_out((m, n), dev), bf16_out((m, n), dev)
    if w8:
        q, s = rc.w8a16_synthetic(rng, n, k)
        exp, _ = orc.w8a16_reference(q, s, 64, b, x)
        dq, ds = to_dev(q, dev), to_dev(s, dev)
        hip.gemm_w8a16(dq, ds, 64, db, dx, y, m, n, k)
        hip.gemm_w8a16_tile(dq, ds, 64, db, dx, yt, m, n, k, 3)
    else:
        w = rc.bf16_normal(rng, (n, k), 0.02)
        exp = orc.bf16_linear_reference(w, b, x)
        dw = to_dev(w, dev)
        hip.gemm_bf16(dw, db, dx, y, m, n, k)
        hip.gemm_bf16_tile(dw, db, dx, yt, m, n, k, 3)
    got = words(y)
    stats = check_close(got, exp, what=f"skinny w8={w8} {m}x{n}x{k}")
    assert stats["bit_identical"] > 0.95, stats
    a, t = rc.bf16_values(got), rc.bf16_values(words(yt))
    assert np.all(np.abs(a - t) <= np.maximum(1.0 / 64, 0.01 * np.abs(t)))


def test_gemm_plan_skinny_token_tiles(hip, orc, dev):
    """A plan of the five narrow Linears (q, k, v, o, down) at M = 100 tokens:
    one ring launch, down split over K into parts — against the oracle, and
    bit-identical across launches."""
    import torch
    m = 100
    rng = rc.philox(2500)
    calls, expected = [], []
    for (name, n, k, bias) in rc.QWEN_LINEARS:
        if n > 1024:
            continue
        x = rc.bf16_normal(rng, (m, k))
        b = rc.bf16_normal(rng, (n,)) if bias else None
        q, s = rc.w8a16_synthetic(rng, n, k)
        exp, _ = orc.w8a16_reference(q, s, 64, b, x)
        calls.append((to_dev(q, dev), to_dev(s, dev), 64, to_dev(b, dev) if bias else None,
                      to_dev(x, dev), bf16_out((m, n), dev), m, n, k))
        expected.append(exp)
    plan = hip.GemmPlan(calls)
    try:
        first = None
        for _ in range(3):
            plan.launch()
            torch.cuda.synchronize()
            got = [words(c[5]) for c in calls]
            for g, e in zip(got, expected):
                stats = check_close(g, e, what="skinny plan, token tiles")
                assert stats["bit_identical"] > 0.95, stats
            if first is None:
                first = got
            for g, f in zip(got, first):
                np.testing.assert_array_equal(g, f)
    finally:
        plan.close()


@pytest.mark.parametrize("w8", [True, False], ids=["w8a16", "bf16"])
def test_gemm_plan_skinny_matches_single_calls(hip, orc, dev, w8):
    """Config 3's seven Linears at M = 24 as one plan: one ring launch of seven
    descriptors (down in parts), against the oracle and the single calls
    (down on the skinny kernel: another association of the same partial
    sums), and bit-identical across launches."""
    import torch
    m = 24
    rng = rc.philox(2400 + w8)
    calls, expected, singles = [], [], []
    for (name, n, k, bias) in rc.QWEN_LINEARS:
        x = rc.bf16_normal(rng, (m, k))
        b = rc.bf16_normal(rng, (n,)) if bias else None
        dx, db = to_dev(x, dev), (to_dev(b, dev) if bias else None)
        y, y1 = bf16_out((m, n), dev), bf16_out((m, n), dev)
        if w8:
            q, s = rc.w8a16_synthetic(rng, n, k)
            exp, _ = orc.w8a16_reference(q, s, 64, b, x)
            dq, ds = to_dev(q, dev), to_dev(s, dev)
            calls.append((dq, ds, 64, db, dx, y, m, n, k))
            hip.gemm_w8a16(dq, ds, 64, db, dx, y1, m, n, k)
        else:
            w = rc.bf16_normal(rng, (n, k), 0.02)
            exp = orc.bf16_linear_reference(w, b, x)
            dw = to_dev(w, dev)
            calls.append((dw, db, dx, y, m, n, k))
            hip.gemm_bf16(dw, db, dx, y1, m, n, k)
        expected.append(exp)
        singles.append(y1)
    plan = hip.GemmPlan(calls)
    try:
        first = None
        for _ in range(3):
            plan.launch()
            torch.cuda.synchronize()
            got = [words(c[5] if w8 else c[3]) for c in calls]
            for g, e, y1 in zip(got, expected, singles):
                check_close(g, e, what="skinny plan")
                a, b1 = rc.bf16_values(g), rc.bf16_values(words(y1))
                assert np.all(np.abs(a - b1) <= np.maximum(1.0 / 64, 0.01 * np.abs(b1)))
            if first is None:
                first = got
            for g, f in zip(got, first):
                np.testing.assert_array_equal(g, f)
    finally:
        plan.close()
