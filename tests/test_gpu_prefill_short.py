"""Short prompts whose q|k|v leaves the RoPE and the KV-cache store to the
attention launch (up to 64 tokens) and the first that does not, against the
CPU FP32 model oracle: the logits, and decode steps on the cache they leave.
K of q|k|v up to 1024 runs on the ring kernel, 1088 to 2048 with int8 weights
on the skinny kernel, three Linears to a launch, gate|up pairs on the ring at
any K."""
import pytest

import model_hip
import synthetic as S
from test_gpu_model import check_step, oracle_model, prompt, teacher_forced

pytestmark = pytest.mark.gpu

CFGS = {
    "h192": S.ModelConfig(hidden_size=192, intermediate_size=320, num_layers=2, num_heads=3,
                          num_kv_heads=1, vocab_size=512),
    "h1088": S.ModelConfig(hidden_size=1088, intermediate_size=192, num_layers=1, num_heads=17,
                           num_kv_heads=1, vocab_size=512),
    "h1536_hd128": S.ModelConfig(hidden_size=1536, intermediate_size=1152, num_layers=1,
                                 num_heads=12, num_kv_heads=2, vocab_size=512),
}
STD = {"h192": 0.12, "h1088": 0.05, "h1536_hd128": 0.04}
_models = {}


def _weights(name, precision):
    key = (name, precision)
    if key not in _models:
        t = S.random_model(CFGS[name], precision, seed=41, std=STD[name])
        _models[key] = (t, S.dequantized_fp32(t, CFGS[name]))
    return _models[key]


@pytest.mark.parametrize("precision", ["w8a16", "w16a16"])
@pytest.mark.parametrize("tokens", [2, 17, 33, 64, 65])
@pytest.mark.parametrize("name", list(CFGS))
def test_short_prompt_and_decode(orc, dev, name, tokens, precision):
    cfg = CFGS[name]
    t, fp32 = _weights(name, precision)
    print(f"short prompt {name} {precision} tokens={tokens}", flush=True)
    g = model_hip.Qwen2Model(cfg, t, precision, max_sequence_length=96, use_graph=False)
    o = oracle_model(orc, cfg, fp32, 96)
    teacher_forced(g, o, prompt(tokens, cfg.vocab_size, seed=tokens), 3, 0.9995, name)
    g.close()
    o.close()
