"""Which launches matmul_f32 and matmul_q8 take, on the host side alone
(hip_host): tiles of 16 rows, of 64 rows, or a wave per 64 int8 outputs, on 256
CUs."""
import pytest

from hip_host import run


@pytest.mark.parametrize("O,last,first", [(5120, 96, 97), (1000, 480, 481), (2880, 160, 161), (16000, 32, 33),
                                          # (one round of 64 x 64 tiles, then two)
                                          (8192, 48, 49), (8256, 96, 97), (64, 512, None)])
def test_rows_in_64_x_64_tiles(O, last, first):
    run(f"""
h = engine(small(n_layers=1, vocab=64, ctx_len=64), synthetic=False)
O, I, first = {O}, 32, {first}
w = np.zeros((O, I), np.float32)
t, qt = pa.PkQtHost(pa.FMT_F32, w.ctypes.data, None, O, I, 0), vp()
pa.check(L.pk_qt_upload(h, C.byref(t), C.byref(qt)))
for S, tiled in [({last}, False)] + [(S, True) for S in (first, 600) if first]:
    x, y = dev(S * I), dev(S * O)
    hh.hh_clear()
    pa.check(L.pk_matmul_qt(h, y, x, qt, S))
    n = launches()
    assert len(n) == 1 and n[0].startswith("k_gemm_chain8_tile<") == tiled, (S, n)
""")


@pytest.mark.parametrize("O,wave", [(49088, False), (49089, True), (201088, True)])
def test_int8_outputs_by_the_wave(O, wave):
    run(f"""
h = engine(small(n_layers=1, vocab=64, ctx_len=64), synthetic=False)
O, I = {O}, 48
q, s = np.zeros((O, I), np.int8), np.ones(O, np.float32)
t, qt = pa.PkQtHost(pa.FMT_INT8, q.ctypes.data, s.ctypes.data, O, I, 0), vp()
pa.check(L.pk_qt_upload(h, C.byref(t), C.byref(qt)))
for S in (1, 4, 5):
    x, y = dev(S * I), dev(S * O)
    hh.hh_clear()
    pa.check(L.pk_matmul_qt(h, y, x, qt, S))
    n = launches()
    assert len(n) == 1 and n[0].startswith("k_gemv_chain8_q8<") == ({wave} and S <= 4), (S, n)
""")
