"""Prefill attention over more query blocks of 32 than one grid dimension
holds (65535): every row is written, the first block and those around the
wrap with the values of their own positions."""
import pytest

pytestmark = pytest.mark.gpu


def test_query_blocks_past_one_grid_dimension(hip, dev):
    import model_hip
    import torch
    tokens, hd = 65535 * 32 + 33, 64
    q = torch.zeros((tokens, 1, hd), dtype=torch.bfloat16, device=dev)  # equal weights
    k = torch.zeros((1, tokens, hd), dtype=torch.bfloat16, device=dev)
    v = torch.ones((1, tokens, hd), dtype=torch.bfloat16, device=dev)
    v[0, :, 0] = (torch.arange(tokens, device=dev) % 2).to(torch.bfloat16)
    out = torch.full_like(q, float("nan"))
    print(f"attention {tokens} tokens", flush=True)
    model_hip.attention_prefill_bf16(q, k, v, out, tokens, 1, 1, hd, tokens)
    # row t: the mean of 0, 1, 0, 1, ... over t + 1 positions; ones elsewhere.
    # FP32 sums of equal weights, their sum off by 2^-24 a term in the worst
    # order (a wave adds 2^16 blocks), and the BF16 rounding
    t = torch.arange(tokens, device=dev)
    mean = ((t + 1) // 2).double() / (t + 1).double()
    tol = 2.0**-9 + 2.0**-8 + 2.0**-7
    assert (out[:, 0, 1:].double() - 1).abs().max() <= tol
    assert (out[:, 0, 0].double() - mean).abs().max() <= tol
