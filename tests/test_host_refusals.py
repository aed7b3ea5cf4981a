"""What the library refuses, it refuses for every number of rows: the checks
of the launches, on the host side alone (hip_host)."""
import pytest

from hip_host import run


@pytest.mark.parametrize("gs", [64, 0])
def test_int4_columns_above_8192(gs):
    """gs64 tiles hold rows of at most 128 groups, for one row and for several
    (which take another launch); a scale per row has a general kernel."""
    run(f"""
h = engine(small(vocab=512), synthetic=False)
def tensor(O, I):
    q, s = np.zeros((O, I // 2), np.uint8), np.ones(O * (I // 64 if {gs} else 1), np.float32)
    t, qt = pa.PkQtHost(pa.FMT_INT4, q.ctypes.data, s.ctypes.data, O, I, {gs}), vp()
    pa.check(L.pk_qt_upload(h, C.byref(t), C.byref(qt)))
    return qt
for I, rc in ((8192, 0), (8256, {-4 if gs else 0})):
    for O in (64, 1000, 20000):
        qt = tensor(O, I)
        for S in (1, 2, 3, 8, 17, 300):
            x, y = dev(S * I), dev(S * O)
            assert L.pk_matmul_qt(h, y, x, qt, S) == rc, (I, O, S)
        pa.check(L.pk_qt_free(h, qt))
""")


def test_experts_above_8192_columns():
    run("""
for hidden, inter, rc in ((8256, 128, -4), (128, 2 * 8256, -4), (8192, 128, 0), (128, 2 * 8192, 0)):
    h = engine(small(n_layers=1, hidden=hidden, moe_inter=inter, vocab=64, ctx_len=64))
    for T in (1, 5, 6, 40, 300):
        x, out = dev(T * hidden), dev(T * hidden)
        assert L.pk_moe_forward_batch(h, 0, x, T, out, None, None) == rc, (hidden, inter, T)
        assert L.pk_moe_forward_batch_noalloc(h, 0, x, min(T, 40), out, None, None) == rc, (hidden, inter, T)
    pa.check(L.pk_engine_destroy(h))
""")
