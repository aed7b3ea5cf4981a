"""gqa_attention's QKV launch with the rotation and the KV store in it, and
the two launches that narrow projections keep, against the oracle."""
import numpy as np
import pytest

from helpers import rel_l2, upload_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("hidden,heads,kv", [(64, 28, 4), (2880, 24, 4), (3136, 28, 4), (4160, 32, 8), (192, 64, 8)])
def test_gqa_attention_widths(gpu, oracle, hidden, heads, kv, offset):
    """2304, 2048 (two launches), 2304 and 3072, 5120 QKV rows over inputs below,
    at and past the 3072 columns held in registers. Sums of at most 4160 fp32
    products in another order than the oracle's: 1e-5, as for the 20B widths."""
    import torch
    import picchio_amd as pa
    cfg = pa.gptoss_cfg(n_layers=2, n_experts=4, ctx_len=160, vocab=256, hidden=hidden, n_heads=heads, n_kv_heads=kv,
                        moe_inter=128)
    model = oracle.model_build(cfg, 31, 0)
    eng = pa.Engine(cfg)
    try:
        upload_model(eng, oracle, model, cfg)
        oracle.model_reset_kv(model)
        rng = np.random.default_rng(hidden)
        od = eng.empty(hidden, torch.float32)
        for pos in range(132):
            for layer in (0, 1):
                x = rng.standard_normal(hidden).astype(np.float32)
                ref = np.empty(hidden, np.float32)
                oracle.gqa_attention(model, layer, x, pos, ref)
                buf = eng.to_dev(np.concatenate([np.zeros(offset, np.float32), x]))
                eng.gqa_attention(layer, buf[offset:], pos, od)
                assert rel_l2(eng.to_host(od), ref) < 1e-5, (pos, layer)
    finally:
        eng.close()
        oracle.model_free(model)
