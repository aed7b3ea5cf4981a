"""The prompt path's rows: the in-order router sums (k_router_seq4) bit for
bit, and a prompt's chunks run through the layers together against the same
prompt chunk by chunk."""
import numpy as np
import pytest

from helpers import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,D,T", [(4, 192, 1), (5, 64, 130), (16, 320, 17), (32, 2880, 9), (33, 192, 8), (64, 448, 5),
                                   (100, 192, 3), (128, 2880, 5)])
def test_router_rows_bitexact(gpu, E, D, T):
    import picchio_amd as pa
    import torch
    cfg = pa.gptoss_cfg(n_layers=1, n_experts=E, hidden=D, moe_inter=128, n_heads=2, n_kv_heads=1, topk=2, ctx_len=16,
                        vocab=64)
    rng = np.random.default_rng(E + D)
    r, b = rng.standard_normal((E, D)).astype(np.float32), rng.standard_normal(E).astype(np.float32)
    x = rng.standard_normal((T, D)).astype(np.float32)
    ref = np.repeat(b[None], T, 0)
    for c in range(D):
        ref = ref + x[:, c:c + 1] * r[None, :, c]          # float32: product rounded, then added
    with pa.Engine(cfg) as eng:
        eng.build_synthetic(3, 1)
        eng.store_router(0, r, b)
        trace, out = eng.empty(T * E, torch.float32), eng.empty((T, D), torch.float32)
        eng.set_router_trace(trace)
        eng.moe_forward_batch(0, eng.to_dev(x), out)
        got = eng.to_host(trace).reshape(T, E)
        eng.set_router_trace(None)
    assert bits_equal(got, ref), first_mismatch(got, ref)


@pytest.mark.parametrize("n", [2, 64, 65, 130, 600])
def test_prompt_chunks_together_match_chunk_by_chunk(gpu, n):
    """With the router trace on, every pass over the layers is one chunk of 64
    tokens; without it up to 512 tokens. Same KV rows, same next token."""
    import picchio_amd as pa
    import torch
    cfg = pa.gptoss_cfg(n_layers=2, n_experts=8, hidden=256, moe_inter=512, n_heads=8, n_kv_heads=2, ctx_len=640,
                        vocab=512)
    ids = np.random.default_rng(n).integers(0, 512, n).astype(np.int32)
    got = []
    with pa.Engine(cfg) as eng:
        eng.build_synthetic(5, 7)
        trace, lg = eng.empty(16, torch.float32), eng.empty(512, torch.float32)
        for traced in (True, False):
            for sampled in (False, True):
                eng.set_sampling(0.9 if sampled else 0.0, 0.95, 50, 1.1 if sampled else 1.0, 77)
                eng.set_router_trace(trace if traced else None)
                nxt = eng.prefill_tokens(ids)
                eng.set_router_trace(None)
                rng, hist = eng.sampler_state()
                eng.set_sampling(0.0, 1.0, 0, 1.0, 1)
                eng.forward_token(7, n, lg)                # reads every KV row
                got.append((nxt, rng, hist.tolist(), eng.to_host(lg).copy()))
    for a, b in ((got[0], got[2]), (got[1], got[3])):
        assert a[0] == b[0] and a[1:3] == b[1:3]
        assert bits_equal(a[3], b[3]), first_mismatch(a[3], b[3])
