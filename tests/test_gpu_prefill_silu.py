"""The SiLU of the prefill's gate|up at prompt lengths whose epilogue divides
(g / (1 + e^-g) in FP32, as a launch of its own does): at g = -88 the
reciprocal of 1 + e^88 is subnormal, and a flushed one would drop every MLP
output of this model, whose up_proj is 2^120."""
import numpy as np
import pytest

import model_hip
import refcases as rc
import synthetic as S

pytestmark = pytest.mark.gpu

CFG = S.ModelConfig(hidden_size=64, intermediate_size=192, num_layers=1, num_heads=1,
                    num_kv_heads=1, vocab_size=256)
G, LOG2_U = -88.0, 120


def _model_tensors(precision):
    """Attention adds nothing, the MLP's input is all ones, and every gate is
    G, every up 2^120; down adds the same value to the odd elements."""
    t = S.random_model(CFG, precision, seed=3)
    rng = np.random.default_rng(5)
    embed = np.sign(rng.standard_normal((CFG.vocab_size, CFG.hidden_size))).astype(np.float32)
    embed[0] = 1.0  # the prompt's token
    t["model.embed_tokens.weight"] = rc.bf16_words(embed)
    h, inter = CFG.hidden_size, CFG.intermediate_size
    for name in list(t):
        if "layernorm" in name or name == "model.norm.weight":
            t[name] = rc.bf16_words(np.ones(h, np.float32))
        elif name.endswith(".bias"):
            t[name] = np.zeros_like(t[name])
    odd = np.arange(h)[:, None] % 2
    mats = {"mlp.gate_proj": (np.full((inter, h), -88), 2.0**-6),
            "mlp.up_proj": (np.full((inter, h), 64), 2.0**(LOG2_U - 12)),
            "mlp.down_proj": (np.broadcast_to(odd, (h, inter)), 2.0**-6),
            "self_attn.o_proj": (np.zeros((h, h)), 1.0)}
    for short, (q, scale) in mats.items():
        name = f"model.layers.0.{short}.weight"
        if precision == "w8a16":
            t[name] = np.ascontiguousarray(q, dtype=np.int8)
            t[name + ".scale"] = rc.bf16_words(
                np.full((q.shape[0], q.shape[1] // 64), scale, np.float32))
        else:
            t[name] = rc.bf16_words((np.asarray(q, np.float64) * scale).astype(np.float32))
    mlp = G * np.exp(G) * 2.0**LOG2_U  # e^88 + 1 = e^88 to 38 digits
    x = 1.0 + np.arange(h) % 2 * (inter * mlp * 2.0**-6)
    return t, embed.astype(np.float64) @ (x / np.sqrt(np.mean(x * x) + CFG.rms_norm_eps))


# the first, one inside and the last length of the range at this model's shape
@pytest.mark.parametrize("precision,tokens", [
    ("w8a16", 129), ("w8a16", 200), ("w8a16", 300), ("w16a16", 33), ("w16a16", 100),
    ("w16a16", 257)])
def test_prefill_silu_keeps_tiny_values(dev, precision, tokens):
    t, expected = _model_tensors(precision)
    m = model_hip.Qwen2Model(CFG, t, precision, max_sequence_length=512)
    print(f"prefill silu {precision} tokens={tokens}", flush=True)
    m.prefill([0] * tokens)
    got = np.asarray(m.last_logits_host(), np.float64)
    m.close()
    # four BF16 roundings (MLP output, down's sum, residual, norm) and the
    # logits' own, each 2^-9 of the elements' magnitudes, which sum to at most
    # the logit's 64 terms
    bound = 5 * 2.0**-8 * np.abs(expected).max()
    assert np.abs(got - expected).max() <= bound
