"""Which launches the batched MoE's experts take, on the host side alone
(hip_host): one per (token, expert) pair while most experts have a single
pair, grouped by expert beyond."""
import pytest

from hip_host import run


@pytest.mark.parametrize("E,single,grouped", [(8, 5, 6), (32, 5, 6), (64, 9, 10), (128, 19, 20)])
def test_pairs_are_grouped_by_pairs_per_expert(E, single, grouped):
    run(f"""
h = engine(small(n_layers=1, n_experts={E}, vocab=64, ctx_len=64))
x, out = dev(64 * 128), dev(64 * 128)
for T, rows in ((1, False), ({single}, False), ({grouped}, True), (64, True)):
    hh.hh_clear()
    pa.check(L.pk_moe_forward_batch(h, 0, x, T, out, None, None))
    n = launches()
    assert any(k.startswith("k_i4_rows") for k in n) == rows == ("k_group_pairs" in n), (T, n)
""")
