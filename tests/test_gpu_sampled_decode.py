"""Draws spread over the device inside the decode step (a vocabulary of 16,384
and more: the draw reads the step's logits, updates the decode state and
leaves no array behind), eagerly after a prompt and replayed from a captured
step, against the oracle's logits drawn by the oracle's sampler. The logits
agree to fp32 noise, so a draw differs only within that of a boundary."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup(gpu, oracle):
    import picchio_amd as pa
    from helpers import upload_model
    cfg = pa.gptoss_cfg(n_layers=2, n_experts=4, topk=2, hidden=256, moe_inter=256, n_heads=4, n_kv_heads=2,
                        ctx_len=256, vocab=20011)
    model = oracle.model_build(cfg, 91, 0)
    eng = pa.Engine(cfg)
    upload_model(eng, oracle, model, cfg)
    yield cfg, model, eng
    eng.set_sampling(0.0, 1.0, 0, 1.0, 0)
    eng.close()
    oracle.model_free(model)


def _params(st, t, p, k):
    C.c_float.from_buffer(st, 0).value = t
    C.c_float.from_buffer(st, 4).value = p
    C.c_int32.from_buffer(st, 8).value = k


# temperature, top_p, top_k, penalty: candidates gathered over the device; more
# than its LDS holds (the 4096th largest's bucket takes them past 4096), so one
# workgroup draws; the ordered sums with and without a cut
CASES = [(0.8, 0.95, 40, 1.0), (0.8, 0.9, 40, 1.3), (0.7, 1.0, 4096, 1.2), (0.7, 0.9, 6000, 1.0), (1.0, 0.9, 0, 1.0),
         (1.0, 0.8, 0, 1.2), (1.0, 1.0, 0, 1.0), (0.9, 1.0, 0, 1.2)]


@pytest.mark.parametrize("case", CASES)
def test_generate_matches_oracle(setup, oracle, monkeypatch, case):
    cfg, model, eng = setup
    monkeypatch.setenv("PREFILL_BATCH", "64")
    prompt = np.random.default_rng(2).integers(0, cfg.vocab, 70).astype(np.int32)
    st, n = oracle.sampler(*case, 77), 10
    if case[3] > 1.0:
        oracle.sampler_push_history(st, prompt, cfg.vocab)
    oracle.model_reset_kv(model)
    lg, ref = np.empty(cfg.vocab, np.float32), []
    for pos, tok in enumerate(prompt):
        oracle.forward_token(model, int(tok), pos, lg.ctypes.data)
        if pos in (63, 69):
            ref = [oracle.sample_logits(st, lg.copy())]
    for i in range(n - 1):
        oracle.forward_token(model, ref[-1], len(prompt) + i, lg.ctypes.data)
        ref.append(oracle.sample_logits(st, lg.copy()))
    eng.set_sampling(*case, 77)
    assert [int(v) for v in eng.generate(prompt, n)] == ref
    rng, hist = eng.sampler_state()
    rng_ref, hist_ref = oracle.sampler_state(st)
    assert rng == rng_ref and np.array_equal(hist, hist_ref)


@pytest.mark.parametrize("rep", [1.0, 1.25])
def test_replay_follows_turn_settings(setup, oracle, rep):
    """The settings change between replays of a captured step (kinds of draw,
    the cut, greedy and back), with eager work between the replays; rng and
    history carry on."""
    cfg, model, eng = setup
    turns = [(0.8, 0.9, 40), (0.8, 1.0, 50), (1.0, 0.9, 0), (1.0, 1.0, 0), (0.9, 0.9, 5000), (0.0, 1.0, 0),
             (0.8, 0.9, 40), (1.0, 0.8, 0), (0.8, 0.9, 0), (0.7, 0.9, 100)]
    st = oracle.sampler(*turns[0], rep, 5)
    eng.set_sampling(*turns[0], rep, 5)
    oracle.model_reset_kv(model)
    lg, tok, pos, steps = np.empty(cfg.vocab, np.float32), 11, 0, 4
    for turn in turns:
        eng.set_turn_sampling(*turn)
        _params(st, *turn)
        first, ref = tok, []
        for i in range(steps):
            oracle.forward_token(model, tok, pos + i, lg.ctypes.data)
            tok = oracle.sample_logits(st, lg.copy())
            ref.append(tok)
        got = [int(v) for v in eng.decode_replay(first, pos, steps)]
        assert got == ref, (turn, got, ref)
        pos += steps
        rng, hist = eng.sampler_state()
        if turn[0] == 0 and rep == 1.0:                # (the step's own argmax, which keeps no history: nothing reads it)
            C.c_int32.from_buffer(st, 24).value = len(hist)
        rng_ref, hist_ref = oracle.sampler_state(st)
        assert rng == rng_ref and np.array_equal(hist, hist_ref), turn
