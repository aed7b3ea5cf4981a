"""The coalesced INT4 quantizer (power-of-two groups) byte for byte the
convert.py restatement: float4 and scalar columns, ragged last groups, odd
widths, zero groups, ties; rows of whole groups taken as one row, a row over
several waves, several spans per wave; non-finite weights' neighbours."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("O,I,gs", [(1, 68, 64), (5, 1441, 64), (9, 2880, 32), (7, 1025, 4), (3, 4096, 256), (6, 130, 128),
                                    (130, 1030, 64), (4, 66, 16)])
def test_quantizer_rows_byteexact(gpu, oracle, O, I, gs, offset):
    import picchio_amd as pa
    import torch
    rng = np.random.default_rng(O + I + gs)
    w = (rng.standard_normal((O, I)) * 0.02).astype(np.float32)
    w[0, :gs] = 0.0                                        # the 1e-8 scale floor
    w[-1, -3:] = np.array([0.25, -0.25, 0.125], np.float32)
    w[-1, gs:2 * gs] = np.round(w[-1, gs:2 * gs] * 64) / 64  # ties
    q4, s = oracle.quant_gs(w, gs)
    with pa.Engine(pa.gptoss_cfg(n_layers=1, n_experts=4, ctx_len=16, vocab=64)) as eng:
        buf = eng.to_dev(np.concatenate([np.zeros(offset, np.float32), w.ravel()]))
        ng = (I + gs - 1) // gs
        pd, sd = eng.empty((O, (I + 1) // 2), torch.uint8), eng.empty((O, ng), torch.float32)
        eng.quantize_int4_gs(buf[offset:], O, I, gs, pd, sd)
        p, sc = eng.to_host(pd), eng.to_host(sd)
    assert np.array_equal(sc.view(np.uint32), np.ascontiguousarray(s, np.float32).reshape(O, ng).view(np.uint32))
    assert np.array_equal(p, q4.reshape(p.shape))


@pytest.mark.parametrize("O,I,gs", [(3, 100003, 8), (2, 70000, 64), (1, 262144, 4), (12000, 2880, 64), (9001, 1001, 16),
                                    (5, 4100, 256), (70001, 64, 4), (40001, 128, 64)])
def test_quantizer_spans_byteexact(gpu, oracle, O, I, gs):
    import picchio_amd as pa
    import torch
    w = (np.random.default_rng(O + I + gs).standard_normal((O, I)) * 0.02).astype(np.float32)
    q4, s = oracle.quant_gs(w, gs)
    with pa.Engine(pa.gptoss_cfg(n_layers=1, n_experts=4, ctx_len=16, vocab=64)) as eng:
        ng = (I + gs - 1) // gs
        pd, sd = eng.empty((O, (I + 1) // 2), torch.uint8), eng.empty((O, ng), torch.float32)
        eng.quantize_int4_gs(eng.to_dev(w), O, I, gs, pd, sd)
        p, sc = eng.to_host(pd), eng.to_host(sd)
    assert np.array_equal(sc.view(np.uint32), np.ascontiguousarray(s, np.float32).reshape(O, ng).view(np.uint32))
    assert np.array_equal(p, q4.reshape(p.shape))


@pytest.mark.parametrize("O,I,gs", [(4, 256, 64), (5, 1441, 16)])
def test_quantizer_non_finite_stays_in_its_group(gpu, oracle, O, I, gs):
    import picchio_amd as pa
    import torch
    w = (np.random.default_rng(O).standard_normal((O, I)) * 0.02).astype(np.float32)
    q4, s = oracle.quant_gs(w, gs)
    bad = w.copy()
    bad[1, gs + 3], bad[1, 2 * gs + 1], bad[2, 0] = np.inf, np.nan, -np.inf
    with pa.Engine(pa.gptoss_cfg(n_layers=1, n_experts=4, ctx_len=16, vocab=64)) as eng:
        ng = (I + gs - 1) // gs
        pd, sd = eng.empty((O, (I + 1) // 2), torch.uint8), eng.empty((O, ng), torch.float32)
        eng.quantize_int4_gs(eng.to_dev(bad), O, I, gs, pd, sd)
        p, sc = eng.to_host(pd), eng.to_host(sd)
    keep = np.ones((O, ng), bool)
    keep[1, 1:3], keep[2, 0] = False, False
    cols = np.repeat(keep, gs, 1)[:, :I:2][:, :p.shape[1]]
    assert np.array_equal(sc[keep], np.ascontiguousarray(s, np.float32).reshape(O, ng)[keep])
    assert np.array_equal(p[cols], q4.reshape(p.shape)[cols])
