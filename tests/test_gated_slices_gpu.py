"""A gated feed-forward of 17 to 64 rows whose product is cut along K: the activation kernel adds the slices."""
import pytest
import torch

import hector_engine_amd as he
from hector_engine_amd.config.qwen2 import Qwen2Config
from hector_engine_amd.kernels import ops
from tests.helpers import rand_ids

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [17, 32, 33, 64])
def test_a_gated_product_cut_along_k_runs_between_17_and_64_rows(rows):
    config = Qwen2Config.from_dict(dict(architectures=["Qwen2ForCausalLM"], num_hidden_layers=2, hidden_size=896,
                                        num_attention_heads=14, num_key_value_heads=2, head_dim=64, intermediate_size=1024,
                                        vocab_size=500, rope_theta=10000.0, rms_norm_eps=1e-6, max_position_embeddings=256,
                                        tie_word_embeddings=True))
    assert ops.gemm_rows_plan(rows, 2 * 1024, 896)[1] > 1          # the case this is about
    ids = rand_ids(500, rows, 3)
    logits = {}
    for dtype in ("bfloat16", "float32"):
        engine = he.Engine(config=config, seed=1, dtype=dtype, max_tokens=256)
        logits[dtype] = engine.step([he.StepEntry(engine.acquire(), ids, list(range(rows)))]).clone()
    want = logits["float32"]
    assert (logits["bfloat16"] - want).abs().max().item() <= 0.02 * want.abs().max().item()
