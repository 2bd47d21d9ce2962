"""The decode step's attention in parts over KV capacities past one tile per
wave of four parts (eight parts, eight waves, tiles in a loop; head_dim 64 and
128), teacher-forced across the edges of a tile and of a part against the CPU
FP32 model oracle."""
import pytest

import model_hip
import synthetic as S
from test_gpu_model import oracle_model, prompt, teacher_forced

pytestmark = pytest.mark.gpu

HD64 = S.ModelConfig(hidden_size=192, intermediate_size=256, num_layers=1, num_heads=3,
                     num_kv_heads=1, vocab_size=512)
HD128 = S.ModelConfig(hidden_size=256, intermediate_size=256, num_layers=1, num_heads=2,
                      num_kv_heads=2, vocab_size=512)


# (config, max_seq, first position): part lengths 256 and 512, then 1024 in a
# loop of two 512-position rounds; head_dim 128: 256 (one tile per wave), and
# 512 in a loop
@pytest.mark.parametrize("cfg,max_seq,start", [
    (HD64, 1025, 254), (HD64, 2048, 2044), (HD64, 4096, 1022), (HD64, 4100, 510),
    (HD64, 4100, 1022), (HD128, 1024, 1020), (HD128, 2048, 254), (HD128, 2049, 254),
    (HD128, 2049, 510)], ids=lambda v: v if isinstance(v, int) else f"hd{v.head_dim}")
def test_parts_form_matches_oracle(orc, dev, cfg, max_seq, start):
    t = S.random_model(cfg, "w8a16", seed=31, std=0.12)
    fp32 = S.dequantized_fp32(t, cfg)
    g = model_hip.Qwen2Model(cfg, t, "w8a16", max_sequence_length=max_seq, use_graph=True)
    o = oracle_model(orc, cfg, fp32, max_seq)
    print(f"parts form hd={cfg.head_dim} max_seq={max_seq} start={start}", flush=True)
    teacher_forced(g, o, prompt(start, cfg.vocab_size, seed=32), 4, 0.9995, "parts")
    g.close()
    o.close()
