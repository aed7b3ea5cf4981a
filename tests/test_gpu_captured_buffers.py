"""A captured batched MoE replays to the eager bits after calls that needed
larger buffers (the kernels of the graph address the ones it was captured
with)."""
import numpy as np
import pytest

from helpers import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu


def test_captured_moe_after_a_longer_prompt(gpu):
    import picchio_amd as pa
    import torch
    cfg = pa.gptoss_cfg(n_layers=2, n_experts=8, hidden=256, moe_inter=512, n_heads=8, n_kv_heads=2, ctx_len=1024,
                        vocab=512)
    T, D, K = 64, cfg.hidden, cfg.topk
    rng = np.random.default_rng(4)
    with pa.Engine(cfg) as eng:
        eng.build_synthetic(5, 7)
        xd = eng.to_dev(rng.standard_normal((T, D)).astype(np.float32))
        ref, out = eng.empty((T, D), torch.float32), eng.empty((T, D), torch.float32)
        sel, w = eng.empty((T, K), torch.int32), eng.empty((T, K), torch.float32)
        eng.moe_forward_batch(0, xd, ref, sel, w)
        ref_h, sel_h, w_h = eng.to_host(ref).copy(), eng.to_host(sel).copy(), eng.to_host(w).copy()
        eng.capture_begin()
        eng.moe_forward_batch(0, xd, out, sel, w)
        g = eng.capture_end()
        for n in (0, 300, 900):
            if n:
                eng.prefill_tokens(rng.integers(0, 512, n).astype(np.int32))
                big = eng.to_dev(rng.standard_normal((n, D)).astype(np.float32))
                eng.moe_forward_batch(1, big, eng.empty((n, D), torch.float32))
            out.zero_(), sel.zero_(), w.zero_()
            torch.cuda.synchronize()
            eng.graph_launch(g)
            got = eng.to_host(out)
            assert bits_equal(got, ref_h), (n, first_mismatch(got, ref_h))
            assert np.array_equal(eng.to_host(sel), sel_h) and bits_equal(eng.to_host(w), w_h), n
        eng.graph_destroy(g)
