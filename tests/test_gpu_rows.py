"""The INT4 GEMV of several input rows on the fp32 matrix instructions
(k_i4_rows): bit-identical to matmul_i4_gs (quant.h:259-319) at the edges of
its tiles (8 input rows, 64 matrix rows, spans of 48 groups), and to the
per-pair kernels inside the batched MoE."""
import numpy as np
import pytest

from helpers import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu


def _rand(shape, seed, scale=1.0):
    return (np.random.default_rng(seed).standard_normal(shape) * scale).astype(np.float32)


@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("O,I,S", [(64, 64, 257), (130, 128, 87), (200, 3136, 65), (70, 6208, 131), (4000, 128, 5),
                                   (2880, 2880, 17), (720, 2880, 31)])
def test_i4_rows_matmul_bitexact(gpu, oracle, O, I, S, offset):
    """offset 1: input rows that are not 16-byte aligned take the per-row kernel."""
    import picchio_amd as pa
    import torch
    q4, s = oracle.quant_gs(_rand((O, I), 5 + O + I, 0.02), 64)
    x = _rand((S, I), 9 + S)
    # the chains hold q/16: exact while a sum's last bit, at least 2^-24 of the
    # smallest term x/16, stays above the least denormal 2^-149 (|x| > 2^-121)
    x[0, ::7] *= 1e-30
    y_ref = oracle.mm_i4_gs(x, q4, s, O, I, 64)
    with pa.Engine(pa.gptoss_cfg(n_layers=1, n_experts=4, ctx_len=16, vocab=64)) as eng:
        qt = eng.qt_upload(pa.FMT_INT4, q4, s, O, I, 64)
        buf = eng.to_dev(np.concatenate([np.zeros(offset, np.float32), x.ravel()]))
        yd = eng.empty((S, O), torch.float32)
        eng.matmul_qt(yd, buf[offset:], qt, S)
        y = eng.to_host(yd)
        eng.qt_free(qt)
    assert bits_equal(y, y_ref), first_mismatch(y, y_ref)


@pytest.mark.parametrize("T", [23, 24, 70, 255, 256, 300])
def test_i4_rows_moe_matches_single_tokens(gpu, T):
    """With one expert per token the batch's expert order does not matter:
    every row of the grouped launch has the bits of the token's own call."""
    import picchio_amd as pa
    import torch
    cfg = pa.gptoss_cfg(n_layers=1, n_experts=8, topk=1, ctx_len=16, vocab=64)
    with pa.Engine(cfg) as eng:
        eng.build_synthetic(11, 1)
        xd = eng.to_dev(_rand((T, cfg.hidden), 3 + T))
        out = eng.empty((T, cfg.hidden), torch.float32)
        one = eng.empty((T, cfg.hidden), torch.float32)
        eng.moe_forward_batch(0, xd, out)
        for t in range(T):
            eng.moe_forward_batch(0, xd[t:t + 1], one[t:t + 1])
        a, b = eng.to_host(out), eng.to_host(one)
    assert bits_equal(a, b), first_mismatch(a, b)


@pytest.mark.parametrize("n", [1, 2, 3])
def test_i4_few_row_blocks_match_many(gpu, n):
    """gate_up and down of a few experts (halves and quarters of row blocks:
    k_i4_gemv_part) against the same experts among 32 in one launch."""
    import picchio_amd as pa
    import torch
    cfg = pa.gptoss_cfg(n_layers=1, n_experts=32, ctx_len=16, vocab=64)
    half = cfg.moe_inter // 2
    with pa.Engine(cfg) as eng:
        eng.build_synthetic(11, 1)
        xd = eng.to_dev(_rand((cfg.hidden,), 3))
        got = []
        for ids in (np.arange(n, dtype=np.int32), np.arange(32, dtype=np.int32)):
            act, eo = eng.empty((len(ids), half), torch.float32), eng.empty((len(ids), cfg.hidden), torch.float32)
            eng.expert_gate_up(0, eng.to_dev(ids), xd, act)
            eng.expert_down(0, eng.to_dev(ids), act, eo)
            got.append((eng.to_host(act)[:n], eng.to_host(eo)[:n]))
    for a, b in zip(*got):
        assert bits_equal(a, b), first_mismatch(a, b)


@pytest.mark.parametrize("O,I,S", [(130, 128, 1), (200, 3136, 3), (70, 6208, 131), (12000, 2880, 1), (33000, 192, 1), (5000, 8192, 1),
                                   (700, 8192, 33), (2880, 2880, 1), (5120, 2880, 17)])
def test_i4_row_scales_in_tiles_bound(gpu, oracle, O, I, S):
    """A scale per row in the tile layout (halves and quarters of row blocks,
    whole ones, the streaming launch, several rows), against the exact sum
    over the stored integers. The order is free: at most D roundings lie
    between a product and its output, D = 8 in a group's chain + 3 in its
    tree, ceil(NG / 4) in a fold chain or 12 + NG / 12 in the rows kernel, + 4
    for the product, the last sums and the scale."""
    import picchio_amd as pa
    import torch
    w = _rand((O, I), 7 + O + I, 0.02)
    q4, s = oracle.quant_gs(w, 0)
    s = np.asarray(s, np.float32).reshape(-1)
    x = _rand((S, I), 13 + S)
    s[0] = np.float32(2.0 ** 125)                 # 16 x the scale alone would overflow
    x *= np.float32(2.0 ** -10)
    b = np.asarray(q4).reshape(O, I // 2)
    q = np.empty((O, I), np.float64)
    q[:, 0::2], q[:, 1::2] = (b & 15).astype(np.float64) - 8, (b >> 4).astype(np.float64) - 8
    with pa.Engine(pa.gptoss_cfg(n_layers=1, n_experts=4, ctx_len=16, vocab=64)) as eng:
        qt = eng.qt_upload(pa.FMT_INT4, q4, s, O, I, 0)
        yd = eng.empty((S, O), torch.float32)
        eng.matmul_qt(yd, eng.to_dev(x), qt, S)
        y = eng.to_host(yd).reshape(S, O).astype(np.float64)
        eng.qt_free(qt)
    sd, xd, ng = s.astype(np.float64), x.astype(np.float64), I // 64
    exact = (xd @ q.T) * sd
    depth = 8 + 3 + max(-(-ng // 4), 12 + ng // 12) + 4
    bound = (np.abs(xd) @ np.abs(q).T) * sd * depth * 2.0 ** -24
    assert (np.abs(y - exact) <= bound).all()


@pytest.mark.parametrize("O,I,S", [(130, 128, 1), (5000, 8192, 1), (12000, 2880, 1), (33000, 192, 1), (700, 8192, 33)])
def test_i4_row_scale_applies_to_the_whole_sum(gpu, O, I, S):
    """Groups that would overflow times the row's scale but cancel (halves and
    quarters of row blocks, whole ones, the streaming launch, several rows).
    Every sum is a small integer over 16 and every scale a power of two, so the
    result is exact."""
    import picchio_amd as pa
    import torch
    q4 = np.full((O, I // 2), 0xff, np.uint8)          # every weight 7
    s = np.full(O, 2.0 ** 125, np.float32)
    s[1::3] = np.float32(2.0 ** -140)
    x = np.zeros((S, I), np.float32)
    x[:, :64], x[:, -64:] = 16.0, -16.0                # +-7168 per group, times 2^125
    x[:, 5] += 0.125 * (1 + np.arange(S) % 8)
    with pa.Engine(pa.gptoss_cfg(n_layers=1, n_experts=4, ctx_len=16, vocab=64)) as eng:
        qt = eng.qt_upload(pa.FMT_INT4, q4, s, O, I, 0)
        yd = eng.empty((S, O), torch.float32)
        eng.matmul_qt(yd, eng.to_dev(x), qt, S)
        y = eng.to_host(yd).reshape(S, O)
        eng.qt_free(qt)
    ref = (x.astype(np.float64).sum(1)[:, None] * 7 * s.astype(np.float64)).astype(np.float32)
    assert bits_equal(y, ref), first_mismatch(y, ref)


def test_i4_upload_in_pieces(gpu, oracle):
    """A tensor larger than the upload's staging (32 MiB: 113 row blocks of 8192
    gs64 columns, 127 with a scale per row), the last piece ragged."""
    import picchio_amd as pa
    import torch
    O, I = 9001, 8192
    rng = np.random.default_rng(3)
    q4 = rng.integers(0, 256, (O, I // 2)).astype(np.uint8)
    x = rng.standard_normal((1, I)).astype(np.float32)
    w = np.empty((O, I), np.float32)
    w[:, 0::2], w[:, 1::2] = (q4 & 15).astype(np.float32) - 8, (q4 >> 4).astype(np.float32) - 8
    sums = (w.astype(np.float64).reshape(O, I // 64, 64) * x[0].astype(np.float64).reshape(1, I // 64, 64)).sum(2)
    size = (np.abs(w) * np.abs(x[0])).sum(1).astype(np.float64)
    with pa.Engine(pa.gptoss_cfg(n_layers=1, n_experts=4, ctx_len=16, vocab=64)) as eng:
        xd, yd = eng.to_dev(x), eng.empty((1, O), torch.float32)
        for gs, ng in ((64, I // 64), (0, 1)):
            s = (rng.random((O, ng)) + 0.5).astype(np.float32)
            qt = eng.qt_upload(pa.FMT_INT4, q4, s, O, I, gs)
            eng.matmul_qt(yd, xd, qt, 1)
            y = eng.to_host(yd).reshape(O)
            eng.qt_free(qt)
            if gs:
                ref = oracle.mm_i4_gs(x, q4, s, O, I, 64).reshape(O)
                assert bits_equal(y, ref), first_mismatch(y, ref)
            else:                                       # (20 roundings at most of sums of these terms)
                assert (np.abs(y - sums.sum(1) * s[:, 0]) <= 20 * 2.0 ** -24 * size * s[:, 0]).all()


@pytest.mark.parametrize("O,I,S", [(64, 64, 513), (130, 128, 175), (200, 3136, 129), (70, 6208, 257), (4000, 128, 9)])
def test_i4_rows_edges_bitexact(gpu, oracle, O, I, S):
    """The shapes above with rows enough for k_i4_rows whatever their groups
    fill, and a scale per row beside (order free: against the exact sum)."""
    import picchio_amd as pa
    import torch
    q4, s = oracle.quant_gs(_rand((O, I), 5 + O + I, 0.02), 64)
    x = _rand((S, I), 9 + S)
    y_ref = oracle.mm_i4_gs(x, q4, s, O, I, 64)
    b = np.asarray(q4).reshape(O, I // 2)
    q = np.empty((O, I), np.float64)
    q[:, 0::2], q[:, 1::2] = (b & 15).astype(np.float64) - 8, (b >> 4).astype(np.float64) - 8
    rs = (np.random.default_rng(1).random(O) + 0.5).astype(np.float32)
    with pa.Engine(pa.gptoss_cfg(n_layers=1, n_experts=4, ctx_len=16, vocab=64)) as eng:
        xd, yd = eng.to_dev(x), eng.empty((S, O), torch.float32)
        got = []
        for gs, sc in ((64, s), (0, rs)):
            qt = eng.qt_upload(pa.FMT_INT4, q4, sc, O, I, gs)
            eng.matmul_qt(yd, xd, qt, S)
            got.append(eng.to_host(yd).copy())
            eng.qt_free(qt)
    assert bits_equal(got[0], y_ref), first_mismatch(got[0], y_ref)
    # a product and its sum: 8 in a chain + 3 in its tree, 4 of a wave's 12
    # groups pairwise, 4 waves per span, the scale
    xd64, depth = x.astype(np.float64), 8 + 3 + 4 + 4 * (-(-I // 3072)) + 1
    exact = (xd64 @ q.T) * rs
    bound = (np.abs(xd64) @ np.abs(q).T) * rs * depth * 2.0 ** -24
    assert (np.abs(got[1] - exact) <= bound).all()
