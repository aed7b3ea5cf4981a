"""matmul_f32 and matmul_q8 of any number of rows (k_gemm_chain8), bit for
bit the oracle's restatement of quant.h:117-186: one and two rows (v_fma),
tiles of 16 and 64 rows (matrix instructions), many int8 outputs of few
rows (k_gemv_chain8_q8), ragged rows, outputs and columns, and operands
whose alignment takes the scalar loads."""
import numpy as np
import pytest

from helpers import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("O,I,S", [(1, 8, 1), (17, 136, 1), (33, 1444, 2), (5, 7, 3), (17, 1441, 16), (300, 2880, 16),
                                   (48, 272, 17), (31, 64, 33), (160, 2880, 64), (16390, 144, 65), (7, 4096, 129), (65700, 48, 1),
                                   (65700, 144, 3), (4096, 48, 130), (49090, 80, 2)])
def test_chain8_bitexact(gpu, oracle, O, I, S, offset):
    import picchio_amd as pa
    import torch
    rng = np.random.default_rng(O + I + S)
    x = rng.standard_normal((S, I)).astype(np.float32)
    x[:, ::5] *= 1e-25                     # with small weights: denormal products and sums
    w = rng.standard_normal((O, I)).astype(np.float32)
    w[:, ::3] *= 1e-17
    w[0] *= 1e-20
    q = rng.integers(-127, 128, (O, I)).astype(np.int8)
    sc = (rng.random(O) + 0.5).astype(np.float32)
    with pa.Engine(pa.gptoss_cfg(n_layers=1, n_experts=4, ctx_len=16, vocab=64)) as eng:
        buf = eng.to_dev(np.concatenate([np.zeros(offset, np.float32), x.ravel()]))
        for fmt, data, scales in ((pa.FMT_F32, w, None), (pa.FMT_INT8, q, sc)):
            ref = np.empty((S, O), np.float32)
            if fmt == pa.FMT_F32:
                oracle.matmul_f32(ref, x, w, S, I, O)
            else:
                oracle.matmul_q8(ref, x, q, sc, S, I, O)
            qt = eng.qt_upload(fmt, data, scales, O, I)
            yd = eng.empty((S, O), torch.float32)
            eng.matmul_qt(yd, buf[offset:], qt, S)
            y = eng.to_host(yd)
            eng.qt_free(qt)
            assert bits_equal(y, ref), (fmt, first_mismatch(y, ref))
