"""decode_replay's captured step against the sampling settings, on the host
side alone (hip_host): after any change of settings the next replay runs the
launches that a step captured under the new ones holds."""
from hip_host import run


def test_captured_step_follows_the_settings():
    run("""
# temperature, top_p, top_k, penalty: one workgroup, over the device with and
# without a top-k, with and without a cut, with and without a penalty; greedy
S = [(t, p, k, r) for t, k in ((0.0, 0), (0.8, 40), (0.8, 0), (0.8, 5000), (0.8, 30000)) for p in (1.0, 0.9)
     for r in (1.0, 1.1)]
out = np.zeros(4, np.int32)
def replay(h):
    hh.hh_clear()
    pa.check(L.pk_decode_replay(h, 3, 0, 2, pa.ptr(out)))
    return launches()
want = []
for s in S:
    h = engine(small(n_layers=1))
    pa.check(L.pk_set_sampling(h, *s, 5))
    want.append(replay(h))
    pa.check(L.pk_engine_destroy(h))
kinds = len(set(map(tuple, want)))
assert kinds == 8, kinds        # argmax, one workgroup, top-k +- penalty, no top-k +- penalty +- cut
h = engine(small(n_layers=1))
for a, sa in enumerate(S):
    for b, sb in enumerate(S):
        for turn in (0, 1) if sa[3] == sb[3] else (0,):
            pa.check(L.pk_set_sampling(h, *sa, 5))
            assert replay(h) == want[a], (sa, sb)
            if turn:
                pa.check(L.pk_set_turn_sampling(h, *sb[:3]))
            else:
                pa.check(L.pk_set_sampling(h, *sb, 5))
            assert replay(h) == want[b], (sa, sb, turn)
# each set of launches is captured once, however often the settings change
assert hh.hh_instantiated() == len(S) + kinds, hh.hh_instantiated()
pa.check(L.pk_set_sampling(h, 0.8, 0.9, 0, 1.0, 5))
a = replay(h)
pa.check(L.pk_set_sampling_fast_sums(h, 1))
b = replay(h)
pa.check(L.pk_set_sampling_fast_sums(h, 0))
assert replay(h) == a and b != a and hh.hh_stale() == 0
""")
