"""The quantizer's launches cover the device whatever the shape of the
matrix, on the host side alone (hip_host)."""
import pytest

from hip_host import run


@pytest.mark.parametrize("O,I,gs", [(1, 1 << 20, 64), (32, 100000, 128), (32, 100001, 64), (5760, 2880, 64),
                                    (100000, 64, 4)])
def test_workgroups_follow_the_columns(O, I, gs):
    """At least a wave for 4096 columns up to 16384 waves, whether these are a
    few long rows or many short ones."""
    run(f"""
h = engine(small(n_layers=1, vocab=64, ctx_len=64), synthetic=False)
O, I, gs = {O}, {I}, {gs}
w, p, s = dev(O * I), dev(O * ((I + 1) // 2), np.uint8), dev(O * (-(-I // gs)))
hh.hh_clear()
pa.check(L.pk_quantize_int4_gs(h, w, O, I, gs, p, s))
assert hh.hh_launches() == 1 and hh.hh_groups(0) >= min(O * I // 4096, 16384) // 4, hh.hh_groups(0)
""")
