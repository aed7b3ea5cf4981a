"""Device buffers over their life, on the host side alone (hip_host): what a
captured graph addresses outlives the calls that need larger buffers."""
import pytest

from hip_host import run

GROW = {
    "prompt": "pa.check(prompt(h, 600))",
    "batch": "pa.check(L.pk_moe_forward_batch(h, 1, x, 200, out, None, None))",
    "grouped": "pa.check(L.pk_moe_forward_grouped(h, 1, x, 200, None, None, out, None, None))",
    "decode_batch": """
pa.check(L.pk_batch_reserve(h, 90))
toks, res = np.zeros(90, np.int32), np.zeros(180, np.int32)
pa.check(L.pk_decode_batch(h, 90, pa.ptr(toks), 0, 2, pa.ptr(res)))""",
}


@pytest.mark.parametrize("grow", sorted(GROW))
@pytest.mark.parametrize("call", ["pk_moe_forward_batch(h, 0, x, 64, out, None, None)",
                                  "pk_moe_forward_grouped(h, 0, x, 64, None, None, out, None, None)"],
                         ids=["captured-batch", "captured-grouped"])
def test_captured_buffers_outlive_growth(call, grow):
    run(f"""
h = engine(small(n_experts=8))
x, out = dev(200 * 128), dev(200 * 128)
pa.check(L.{call})                       # (sizes the buffers)
pa.check(L.pk_capture_begin(h))
pa.check(L.{call})
g = vp()
pa.check(L.pk_capture_end(h, C.byref(g)))
{GROW[grow]}
pa.check(L.pk_graph_launch(h, g))
assert hh.hh_stale() == 0, hh.hh_stale()
# given back: the growth after the last graph's end frees what it kept
pa.check(L.pk_graph_destroy(g))
used = hh.hh_in_use()
big_x, big_out = dev(1000 * 128), dev(1000 * 128)
pa.check(L.pk_moe_forward_grouped(h, 0, big_x, 1000, None, None, big_out, None, None))
once = hh.hh_in_use()
pa.check(L.pk_engine_destroy(h))
assert hh.hh_in_use() == 4 * 128 * (200 + 200 + 1000 + 1000), hh.hh_in_use()
# an engine that never captured holds as much
h = engine(small(n_experts=8))
{GROW[grow]}
pa.check(L.pk_moe_forward_grouped(h, 0, big_x, 1000, None, None, big_out, None, None))
assert hh.hh_in_use() == once, (hh.hh_in_use(), once)
""")


@pytest.mark.parametrize("call,bufs", [("pk_moe_forward_batch(h, 1, x, T, out, None, None)", 10),
                                       ("pk_moe_forward_grouped(h, 1, x, T, None, None, out, None, None)", 14)],
                         ids=["batch", "grouped"])
def test_growth_keeps_only_what_a_graph_addresses(call, bufs):
    """A graph lives over a slow growth: only the buffers of its own time stay
    beside the present ones, and go at the first growth after its end, while a
    later graph keeps its own."""
    run(f"""
h = engine(small(n_experts=8))
x, out = dev(300 * 128), dev(300 * 128)
def call(T):
    pa.check(L.{call})
def capture(T):
    call(T)
    pa.check(L.pk_capture_begin(h))
    call(T)
    g = vp()
    pa.check(L.pk_capture_end(h, C.byref(g)))
    return g
g = capture(64)
n = hh.hh_buffers()
for T in range(65, 200):
    call(T)
assert hh.hh_buffers() == n + {bufs}, (n, hh.hh_buffers())
g2 = capture(200)
call(201)
assert hh.hh_buffers() == n + 2 * {bufs}
pa.check(L.pk_graph_launch(h, g))
pa.check(L.pk_graph_launch(h, g2))
assert hh.hh_stale() == 0, hh.hh_stale()
pa.check(L.pk_graph_destroy(g))
call(202)
assert hh.hh_buffers() == n + {bufs}
pa.check(L.pk_graph_launch(h, g2))
assert hh.hh_stale() == 0
pa.check(L.pk_graph_destroy(g2))
call(203)
assert hh.hh_buffers() == n
""")


def test_graph_may_outlive_its_engine():
    run("""
h = engine(small())
x, out = dev(64 * 128), dev(64 * 128)
pa.check(L.pk_moe_forward_batch(h, 0, x, 64, out, None, None))
pa.check(L.pk_capture_begin(h))
pa.check(L.pk_moe_forward_batch(h, 0, x, 64, out, None, None))
g = vp()
pa.check(L.pk_capture_end(h, C.byref(g)))
pa.check(L.pk_engine_destroy(h))
pa.check(L.pk_graph_destroy(g))
""")


@pytest.mark.parametrize("sized", [0, 100])
def test_prompt_in_the_memory_of_one_chunk(sized):
    """Wherever the memory for a prompt chunk by chunk is there (the router
    trace keeps one chunk of 64 per pass), the prompt runs, and buffers sized
    for a capture are as they were after a pass of 512 rows did not fit."""
    run(f"""
T = {sized}
def start():
    h = engine(small(vocab=512))
    if T:
        pa.check(L.pk_moe_forward_batch(h, 0, x, T, x, None, None))
    return h
x, trace = dev(1 + T * 128), dev(16)
h = start()
base = hh.hh_in_use()
pa.check(L.pk_set_router_trace(h, trace, 16))
hh.hh_peak(1)
pa.check(prompt(h, 600))
need = hh.hh_peak(0)
pa.check(L.pk_set_router_trace(h, None, 0))
pa.check(prompt(h, 600))
wide = hh.hh_peak(0)
pa.check(L.pk_engine_destroy(h))
assert need - base > 1 << 17 and wide - need > 1 << 20, (base, need, wide)
for budget in range(need, wide + (1 << 16), (wide - need) // 60):
    h = start()
    if T:
        pa.check(L.pk_capture_begin(h))
        pa.check(L.pk_moe_forward_batch(h, 0, x, T, x, None, None))
        g = vp()
        pa.check(L.pk_capture_end(h, C.byref(g)))
    hh.hh_budget(budget)
    pa.check(prompt(h, 600))
    if T:
        pa.check(L.pk_graph_launch(h, g))
        assert hh.hh_stale() == 0
        pa.check(L.pk_graph_destroy(g))
        pa.check(L.pk_capture_begin(h))
        pa.check(L.pk_moe_forward_batch(h, 0, x, T, x, None, None))
        pa.check(L.pk_capture_end(h, C.byref(g)))
        pa.check(L.pk_graph_destroy(g))
    pa.check(L.pk_engine_destroy(h))
    hh.hh_budget(-1)
""")


@pytest.mark.parametrize("case", [(1.0, 0.9, 0, 1.0), (1.0, 1.0, 50, 1.1), (1.0, 1.0, 0, 1.1)])
def test_step_graph_after_a_larger_vocabulary(case):
    """decode_replay keeps its captured step; a draw over a larger vocabulary
    than the model's replaces the scratch that the step addresses."""
    run(f"""
h = engine(small())
pa.check(L.pk_set_sampling(h, {case[0]}, {case[1]}, {case[2]}, {case[3]}, 5))
out, lg, tok = np.zeros(8, np.int32), dev(70000), C.c_int32()
pa.check(L.pk_decode_replay(h, 3, 0, 4, pa.ptr(out)))
pa.check(L.pk_decode_replay(h, 3, 0, 4, pa.ptr(out)))
assert hh.hh_instantiated() == 1
pa.check(L.pk_sample_logits(h, lg, 70000, C.byref(tok)))
assert hh.hh_execs() == 0                # (the step is gone with what it addressed)
pa.check(L.pk_decode_replay(h, 3, 0, 4, pa.ptr(out)))
assert hh.hh_stale() == 0, hh.hh_stale()
pa.check(L.pk_sample_logits(h, lg, 70000, C.byref(tok)))
assert hh.hh_execs() == 1 and hh.hh_instantiated() == 2
""")


def test_row_scaled_int4_holds_one_scale_per_row():
    run("""
h = engine(small(vocab=512), synthetic=False)
O, I = 1000, 2880
q, s = np.zeros((O, I // 2), np.uint8), np.ones(O, np.float32)
t, qt = pa.PkQtHost(pa.FMT_INT4, q.ctypes.data, s.ctypes.data, O, I, 0), vp()
pa.check(L.pk_qt_upload(h, C.byref(t), C.byref(qt)))
pa.check(L.pk_qt_free(h, qt))                         # (the upload's staging stays)
before = hh.hh_in_use()
pa.check(L.pk_qt_upload(h, C.byref(t), C.byref(qt)))
rows = (O + 63) // 64 * 64
assert hh.hh_in_use() - before == rows * (I // 2 + 4), hh.hh_in_use() - before
""")


@pytest.mark.parametrize("gs", [0, 64])
def test_int4_upload_needs_no_second_tensor(gs):
    """The staging of an upload is bounded: a large tensor fits beside it."""
    run(f"""
h = engine(small(vocab=512), synthetic=False)
O, I = 60000, 8192
q, s = np.zeros((O, I // 2), np.uint8), np.ones(O * (1 if {gs} == 0 else I // 64), np.float32)
t, qt = pa.PkQtHost(pa.FMT_INT4, q.ctypes.data, s.ctypes.data, O, I, {gs}), vp()
before = hh.hh_in_use()
hh.hh_peak(1)
pa.check(L.pk_qt_upload(h, C.byref(t), C.byref(qt)))
rows = (O + 63) // 64 * 64
tensor = rows * (I // 2 + 4 * (1 if {gs} == 0 else I // 64))
assert hh.hh_peak(0) - before <= tensor + (33 << 20), hh.hh_peak(0) - before - tensor
""")
