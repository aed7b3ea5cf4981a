"""Which launches the batched MoE's experts take, on the host side alone
(hip_host): one per (token, expert) pair, or grouped by expert where experts
have several and their rows fill the device."""
import pytest

from hip_host import run


@pytest.mark.parametrize("D,inter,E,single,grouped", [
    # (136 row blocks of gate_up and down, as many as 2880 / 5760 has but for one)
    (128, 8576, 8, 5, 6), (128, 8576, 32, 5, 6), (128, 8576, 64, 9, 10), (128, 8576, 128, 19, 20),
    # small experts: 12 row blocks per CU
    (128, 256, 8, 127, 128), (256, 512, 8, 63, 64), (1024, 2048, 32, 15, 16)])
def test_pairs_are_grouped_where_it_pays(D, inter, E, single, grouped):
    """On 256 CUs."""
    run(f"""
h = engine(small(n_layers=1, n_experts={E}, vocab=64, ctx_len=64, hidden={D}, moe_inter={inter}))
x, out = dev(256 * {D}), dev(256 * {D})
for T, rows in ((1, False), ({single}, False), ({grouped}, True), (256, True)):
    hh.hh_clear()
    pa.check(L.pk_moe_forward_batch(h, 0, x, T, out, None, None))
    n = launches()
    assert any(k.startswith("k_i4_rows") for k in n) == rows == ("k_group_pairs" in n), (T, n)
""")


@pytest.mark.parametrize("O,I,per_row,rows", [(1024, 1024, 32, 33), (512, 512, 64, 65), (5760, 576, 5, 6), (4096, 4096, 8, 9),
                                              (2048, 2048, 16, 17), (2880, 2880, 5, 6), (5760, 2880, 2, 3),
                                              (2880, 5760, 5, 6), (2880, 8192, 5, 6)])
@pytest.mark.parametrize("gs", [64, 0])
def test_matmul_rows_share_weights_where_it_pays(O, I, per_row, rows, gs):
    """On 256 CUs: two workgroups per CU of the per-row launch, or one where the
    rows fill their spans of 48 groups."""
    run(f"""
h = engine(small(n_layers=1, vocab=64, ctx_len=64), synthetic=False)
O, I, gs = {O}, {I}, {gs}
q, s = np.zeros((O, I // 2), np.uint8), np.ones(O * (I // 64 if gs else 1), np.float32)
t, qt = pa.PkQtHost(pa.FMT_INT4, q.ctypes.data, s.ctypes.data, O, I, gs), vp()
pa.check(L.pk_qt_upload(h, C.byref(t), C.byref(qt)))
for S, many in ((1, False), ({per_row}, False), ({rows}, True), (64 + {rows}, True)):
    x, y = dev(S * I), dev(S * O)
    hh.hh_clear()
    pa.check(L.pk_matmul_qt(h, y, x, qt, S))
    n = launches()
    assert len(n) == 1 and n[0].startswith("k_i4_rows<") == many, (S, n)
""")
