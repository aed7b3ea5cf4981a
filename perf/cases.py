"""The work that users of this framework have it do, as timed cases.

A case is a dict of plain values; its "kind" names the entry point it goes
through (all at the GPT-OSS widths: hidden 2880, expert rows 5760, 64 query
heads over 8 KV heads of 64, vocabulary 201,088):

  ffn       expert_gate_up + expert_down of n experts of one layer, one token
  moe       moe_forward of single tokens over the layers (batch-1 decode's MoE)
  rows      moe_forward_batch, T rows (a prompt chunk's MoE)
  grouped   moe_forward_grouped, T rows on the matrix cores (a long prompt's MoE)
  attn      gqa_attention of one token at a position, a sliding-window and a
            full-context layer
  matmul    matmul_qt of S rows: QKV / O-projection and lm_head shapes, fp32,
            INT8 rows, INT4 rows, INT4 groups of 64
  sample    sample_logits over the vocabulary, a run of consecutive draws
  quantize  quantize_int4_gs of one matrix (the converter's INT4 step)
  prompt    prefill_tokens, then the logits of the token after it
  decode    decode_replay steps over a context, then the next token's logits
  batch     decode_batch steps of several sequences, then the first one's logits

The whole-model calls run a few layers of the named shapes (every layer is the
same work). One model serves all inputs of a case, as in a program that keeps
it loaded: its weights follow from the case, the inputs from the seed.
"""
import ctypes
import functools
import math
import weakref

import numpy as np
import torch

import picchio_amd as pa

D, INTER, HALF, TOPK = 2880, 5760, 2880, 4
H, KVH, HD, VOCAB = 64, 8, 64, 201088
EXPERT_BYTES = 3 * D * HALF // 2 + 3 * D * HALF // 64 * 4 + (INTER + D) * 4
EXPERT_FLOPS = 2 * 3 * D * HALF
ATT_PARAMS = (H + 2 * KVH) * HD * D + D * H * HD


def listed():
    return [
        # one expert after another, one token: expert_apply's work, the smallest call
        dict(name="expert_ffn_1", kind="ffn", n=1, calls=16, experts=32, dot=False),
        # the MoE layers of a decoded token, picchio's fp32 arithmetic (the default)
        dict(name="moe_token_20b", kind="moe", tokens=4, layers=2, experts=32, dot=False),
        # the MoE of one prompt chunk (64 positions)
        dict(name="moe_rows_64", kind="rows", T=64, experts=32, dot=False),
        # the MoE of a 2048-token prompt as expert-grouped matrix products
        dict(name="moe_grouped_2048", kind="grouped", T=2048, experts=32),
        # a decoded token's attention after 4096 positions
        dict(name="attention_4096", kind="attn", pos=4096),
        # the INT8 lm_head of one token
        dict(name="lm_head_int8", kind="matmul", fmt="int8", S=1, O=VOCAB, I=D),
        # picchio's default sampling (temperature 1, top-p 0.95, top-k 50, penalty 1.1)
        dict(name="sample_default", kind="sample", draws=8, temperature=1.0, top_p=0.95, top_k=50, penalty=1.1),
        # nucleus sampling without a top-k cut, as chat clients commonly ask for it
        dict(name="sample_nucleus", kind="sample", draws=4, temperature=0.8, top_p=0.95, top_k=0, penalty=1.0),
        # one expert's gate_up through the converter's quantizer
        dict(name="quantize_gate_up", kind="quantize", O=INTER, I=D, gs=64),
        # a 512-token prompt
        dict(name="prompt_512", kind="prompt", n=512, layers=4, experts=32),
        # single-sequence decode after 512 positions, integer-dot experts
        dict(name="decode_20b", kind="decode", steps=16, pos=512, layers=4, experts=32, dot=True),
        # 32 sequences in lockstep, 128 experts, 4096 positions each
        dict(name="decode_batch_32", kind="batch", n=32, steps=4, pos=4096, layers=2, experts=128),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["ffn", "moe", "rows", "grouped", "attn", "matmul", "matmul", "sample", "quantize", "prompt",
                       "decode", "batch"])
    if kind == "ffn":
        return dict(kind=kind, n=_log(rng, 1, 32), calls=rng.randint(4, 16), experts=32, dot=rng.random() < 0.4)
    if kind == "moe":
        return dict(kind=kind, tokens=rng.randint(1, 8), layers=rng.randint(1, 3), experts=rng.choice([32, 32, 128]),
                    dot=rng.random() < 0.5)
    if kind == "rows":
        return dict(kind=kind, T=_log(rng, 2, 256), experts=rng.choice([32, 32, 128]), dot=rng.random() < 0.2)
    if kind == "grouped":
        return dict(kind=kind, T=_log(rng, 65, 2048), experts=32)
    if kind == "attn":
        return dict(kind=kind, pos=_log(rng, 1, 8000))
    if kind == "matmul":
        fmt = rng.choice(["f32", "int8", "int4", "int4_gs"])
        O, I = rng.choice([((H + 2 * KVH) * HD, D), (D, H * HD), (INTER, D), (_log(rng, 1000, 16000), D),
                           (rng.randint(500, 3000), rng.choice([1000, 1441, 2880])),
                           (VOCAB, D) if fmt != "f32" else (32 * 1024, D)])
        return dict(kind=kind, fmt=fmt, S=_log(rng, 1, 64 if O < 20000 else 4), O=O, I=I)
    if kind == "sample":
        top_k = rng.choice([0, 0, 40, 50, 50, 1000])
        return dict(kind=kind, draws=rng.randint(1, 8 if top_k else 3), temperature=round(rng.uniform(0.5, 1.0), 2),
                    top_p=rng.choice([0.9, 0.95, 1.0]), top_k=top_k, penalty=rng.choice([1.0, 1.1]))
    if kind == "quantize":
        return dict(kind=kind, O=_log(rng, 500, 2 * INTER), I=rng.choice([D, D, 4096, 1441, rng.randint(500, 5000)]),
                    gs=rng.choice([64, 64, 64, 32]))
    if kind == "prompt":
        return dict(kind=kind, n=_log(rng, 5, 512), layers=rng.randint(2, 4), experts=rng.choice([32, 32, 128]))
    if kind == "decode":
        return dict(kind=kind, steps=rng.randint(4, 24), pos=_log(rng, 3, 6000), layers=rng.randint(2, 4),
                    experts=rng.choice([32, 32, 128]), dot=rng.random() < 0.5)
    return dict(kind=kind, n=_log(rng, 2, 32), steps=rng.randint(2, 4), pos=_log(rng, 16, 4096), layers=2,
                experts=rng.choice([32, 128]))


# ───────────────────────────── models ─────────────────────────────

class _Model:
    """An engine and what was loaded into it; closed when no state holds it."""

    def __init__(self, **kw):
        self.cfg = pa.gptoss_cfg(**kw)
        self.eng = pa.Engine(self.cfg)
        self.qt = None

    def __del__(self):
        eng = getattr(self, "eng", None)
        if eng is not None:
            if self.qt is not None:
                eng.qt_free(self.qt)
            eng.close()


_models = weakref.WeakValueDictionary()
WSEED = 20           # the models' weight seed


def _shape(case):
    """Engine configuration of a case, and the parts of it that are built."""
    k = case["kind"]
    if k in ("ffn", "moe", "rows", "grouped"):
        return dict(n_layers=case.get("layers", 1), n_experts=case["experts"], ctx_len=16, vocab=64), 1
    if k == "attn":
        return dict(n_layers=2, n_experts=4, ctx_len=case["pos"] + 1, vocab=64), 2
    if k == "prompt":
        return dict(n_layers=case["layers"], n_experts=case["experts"], ctx_len=case["n"] + 1), 7
    if k in ("decode", "batch"):
        return dict(n_layers=case["layers"], n_experts=case["experts"], ctx_len=case["pos"] + case["steps"] + 1), 7
    return dict(n_layers=1, n_experts=4, ctx_len=16, vocab=VOCAB if k == "sample" else 64), 0


def _model(case):
    key = repr(sorted((k, v) for k, v in case.items() if k != "name"))
    m = _models.get(key)
    if m is not None:
        return m
    kw, what = _shape(case)
    m = _Model(**kw)
    if what:
        m.eng.build_synthetic(WSEED, what)
    if case["kind"] == "matmul":
        w, s = _qt_weights(case)
        fmt = {"f32": pa.FMT_F32, "int8": pa.FMT_INT8}.get(case["fmt"], pa.FMT_INT4)
        m.qt = m.eng.qt_upload(fmt, w.cpu().numpy(), None if s is None else s.cpu().numpy(), case["O"], case["I"],
                               64 if case["fmt"] == "int4_gs" else 0)
    if "dot" in case:
        m.eng.set_i4_dot(case["dot"])
    if case["kind"] == "attn":
        m.eng.kv_fill_synthetic(0, case["pos"], 5)
    if case["kind"] == "decode":
        m.eng.kv_fill_synthetic(0, case["pos"], 5)
    if case["kind"] == "batch":
        m.eng.batch_reserve(case["n"])
        for s in range(case["n"]):
            m.eng.kv_fill_synthetic(s, case["pos"], 5)
    m.eng.sync()
    _models[key] = m
    return m


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _qt_weights(case):
    """Weights of a matmul case in picchio's tensor layout, on the GPU."""
    O, I, g = case["O"], case["I"], _gen(WSEED)
    if case["fmt"] == "f32":
        return torch.randn((O, I), generator=g, device="cuda") * 0.02, None
    if case["fmt"] == "int8":
        q = torch.randint(-127, 128, (O, I), generator=g, device="cuda", dtype=torch.int8)
        return q, (torch.rand(O, generator=g, device="cuda") + 0.5) * 1e-3
    q = torch.randint(0, 256, (O, (I + 1) // 2), generator=g, device="cuda", dtype=torch.uint8)
    groups = (I + 63) // 64 if case["fmt"] == "int4_gs" else 1
    return q, (torch.rand((O, groups), generator=g, device="cuda") + 0.5) * 1e-2


def _inputs(case, seed):
    """The seed's inputs: hidden rows as RMSNorm leaves them, expert ids,
    token ids, logits with a model's spread (a few strong candidates over a
    broad tail)."""
    g, k = _gen(seed), case["kind"]
    if k == "ffn":
        ids = torch.stack([torch.randperm(case["experts"], generator=g, device="cuda")[:case["n"]]
                           for _ in range(case["calls"])]).to(torch.int32)
        return dict(x=torch.randn((case["calls"], D), generator=g, device="cuda"), ids=ids)
    if k == "moe":
        return dict(x=torch.randn((case["tokens"], D), generator=g, device="cuda"))
    if k in ("rows", "grouped"):
        return dict(x=torch.randn((case["T"], D), generator=g, device="cuda"))
    if k == "attn":
        return dict(x=torch.randn((2, D), generator=g, device="cuda"))
    if k == "matmul":
        return dict(x=torch.randn((case["S"], case["I"]), generator=g, device="cuda"))
    if k == "sample":
        lg = torch.randn((case["draws"], VOCAB), generator=g, device="cuda") * 2.0
        hot = torch.randint(0, VOCAB, (case["draws"], 24), generator=g, device="cuda")
        lg.scatter_add_(1, hot, torch.rand((case["draws"], 24), generator=g, device="cuda") * 10.0)
        return dict(logits=lg)
    if k == "quantize":
        return dict(w=torch.randn((case["O"], case["I"]), generator=g, device="cuda") * 0.02)
    n = {"prompt": case.get("n"), "decode": 1, "batch": case.get("n")}[k]
    ids = torch.randint(0, VOCAB, (n + 1,), generator=g, device="cuda").cpu().numpy().astype(np.int32)
    return dict(ids=ids)


def prepare(case, seed):
    k, m = case["kind"], _model(case)
    st = dict(case=case, m=m, **_inputs(case, seed))
    f32 = functools.partial(torch.empty, dtype=torch.float32, device="cuda")
    if k == "ffn":
        n, c = case["n"], case["calls"]
        st.update(act=f32((c, n, HALF)), out=f32((c, n, D)))
        if case["dot"]:
            st.update(rec=torch.empty((c, D // 32, 24), dtype=torch.int32, device="cuda"),
                      act_rec=torch.empty((c, n, INTER // 64, 24), dtype=torch.int32, device="cuda"))
    elif k == "moe":
        st.update(out=f32((case["tokens"], case["layers"], D)))
    elif k in ("rows", "grouped"):
        T = case["T"]
        st.update(out=f32((T, D)))
        if k == "rows":
            st.update(sel=torch.empty((T, TOPK), dtype=torch.int32, device="cuda"), w=f32((T, TOPK)))
    elif k == "attn":
        st.update(out=f32((2, D)))
    elif k == "matmul":
        st.update(y=f32((case["S"], case["O"])))
    elif k == "sample":
        st.update(probs=torch.empty_like(st["logits"]))
    elif k == "quantize":
        O, I = case["O"], case["I"]
        st.update(packed=torch.empty((O, (I + 1) // 2), dtype=torch.uint8, device="cuda"),
                  scales=f32((O, -(-I // case["gs"]))))
    else:
        st.update(logits=f32((VOCAB,)))
    torch.cuda.synchronize()
    return st


def run(st):
    case, eng = st["case"], st["m"].eng
    k = case["kind"]
    if k == "ffn":
        for c in range(case["calls"]):
            if case["dot"]:
                eng.act_records(st["x"][c], st["rec"][c])
                eng.expert_gate_up_dot(0, st["ids"][c], st["rec"][c], st["act"][c], st["act_rec"][c])
                eng.expert_down_dot(0, st["ids"][c], st["act_rec"][c], st["out"][c])
            else:
                eng.expert_gate_up(0, st["ids"][c], st["x"][c], st["act"][c])
                eng.expert_down(0, st["ids"][c], st["act"][c], st["out"][c])
        return dict(act=st["act"], out=st["out"])
    if k == "moe":
        for t in range(case["tokens"]):
            for l in range(case["layers"]):
                eng.moe_forward(l, st["x"][t], st["out"][t, l])
        return dict(out=st["out"])
    if k == "rows":
        eng.moe_forward_batch(0, st["x"], st["out"], st["sel"], st["w"])
        return dict(out=st["out"], sel=st["sel"], w=st["w"])
    if k == "grouped":
        eng.moe_forward_grouped(0, st["x"], st["out"])
        return dict(out=st["out"])
    if k == "attn":
        for l in range(2):
            eng.gqa_attention(l, st["x"][l], case["pos"], st["out"][l])
        return dict(out=st["out"])
    if k == "matmul":
        eng.matmul_qt(st["y"], st["x"], st["m"].qt, case["S"])
        return dict(y=st["y"])
    if k == "sample":
        # a new turn: the sampler's settings, then a draw from each step's
        # logits (the copy stands for the model's lm_head writing them)
        eng.set_sampling(case["temperature"], case["top_p"], case["top_k"], case["penalty"], 88172645463325252)
        with torch.cuda.stream(eng.stream):
            st["probs"].copy_(st["logits"])
        toks = [eng.sample_logits(st["probs"][d]) for d in range(case["draws"])]
        return dict(toks=np.array(toks, np.int32), probs=st["probs"])
    if k == "quantize":
        eng.quantize_int4_gs(st["w"], case["O"], case["I"], case["gs"], st["packed"], st["scales"])
        return dict(packed=st["packed"], scales=st["scales"])
    if k == "prompt":
        nxt = eng.prefill_tokens(st["ids"][:case["n"]])
        eng.forward_token(int(st["ids"][case["n"]]), case["n"], st["logits"])
        return dict(next=nxt, logits=st["logits"])
    if k == "decode":
        toks = eng.decode_replay(int(st["ids"][0]), case["pos"], case["steps"])
        eng.forward_token(int(toks[-1]), case["pos"] + case["steps"], st["logits"])
        return dict(toks=toks, logits=st["logits"])
    toks = eng.decode_batch(st["ids"][:case["n"]], case["pos"], case["steps"])
    eng.forward_token(int(toks[-1, 0]), case["pos"] + case["steps"], st["logits"])
    return dict(toks=toks, logits=st["logits"])


# ───────────────────────────── work ─────────────────────────────

def _att_bytes(pos, layers):
    """K and V rows that one token reads: sliding layers 128, full ones all."""
    full = layers // 2
    return 2 * KVH * HD * 4 * (min(pos + 1, 128) * (layers - full) + (pos + 1) * full)


def _distinct(T, E):
    """Expected number of experts that T tokens' routings touch."""
    return E * (1.0 - (1.0 - TOPK / E) ** T)


def work(case):
    k = case["kind"]
    router = D * case.get("experts", 0) * 4
    token = TOPK * EXPERT_FLOPS + 2 * D * case.get("experts", 0)
    head = VOCAB * D * 4
    if k == "ffn":
        pairs = case["n"] * case["calls"]
        return dict(bytes=pairs * EXPERT_BYTES + (case["calls"] * D + pairs * (HALF + D)) * 4,
                    flops=pairs * EXPERT_FLOPS)
    if k == "moe":
        n = case["tokens"] * case["layers"]
        return dict(bytes=n * (TOPK * EXPERT_BYTES + router + 2 * D * 4), flops=n * token)
    if k in ("rows", "grouped"):
        T = case["T"]
        return dict(bytes=_distinct(T, case["experts"]) * EXPERT_BYTES + router + 2 * T * D * 4, flops=T * token)
    if k == "attn":
        return dict(bytes=2 * ATT_PARAMS * 4 + _att_bytes(case["pos"], 2) + 4 * D * 4,
                    flops=2 * 2 * ATT_PARAMS + 2 * H // KVH * _att_bytes(case["pos"], 2) // 4)
    if k == "matmul":
        S, O, I = case["S"], case["O"], case["I"]
        per = {"f32": 4.0, "int8": 1.0, "int4": 0.5, "int4_gs": 0.5 + 4 / 64}[case["fmt"]]
        return dict(bytes=O * I * per + S * (I + O) * 4, flops=2 * S * O * I)
    if k == "sample":
        return dict(bytes=case["draws"] * VOCAB * 8, flops=case["draws"] * VOCAB * 4)
    if k == "quantize":
        O, I = case["O"], case["I"]
        return dict(bytes=O * I * 4 + O * I // 2 + O * (-(-I // case["gs"])) * 4, flops=3 * O * I)
    L = case["layers"]
    if k == "prompt":
        n = case["n"]
        layer = ATT_PARAMS * 4 + _distinct(n, case["experts"]) * EXPERT_BYTES + router
        att = 2 * 2 * H * HD * n * (min(n, 128) + n / 2) / 2
        return dict(bytes=L * layer + head + L * (ATT_PARAMS * 4 + TOPK * EXPERT_BYTES) + head,
                    flops=n * L * (2 * ATT_PARAMS + token) + L * att)
    if k == "decode":
        n = case["steps"] + 1
        return dict(bytes=n * (L * (ATT_PARAMS * 4 + TOPK * EXPERT_BYTES + router) + _att_bytes(case["pos"], L) + head),
                    flops=n * (L * (2 * ATT_PARAMS + token) + 2 * VOCAB * D))
    n, s = case["n"], case["steps"]
    step = L * (ATT_PARAMS * 4 + _distinct(n, case["experts"]) * EXPERT_BYTES + router)
    return dict(bytes=s * (step + n * _att_bytes(case["pos"], L) + head),
                flops=s * n * (L * (2 * ATT_PARAMS + token) + 2 * VOCAB * D))


def tolerance(case):
    """About four times what the path shows against 64-bit sums."""
    k = case["kind"]
    if k == "quantize":
        return "exact"
    if k == "sample":
        # a sum of 200k floats is off by up to ~2e-4 in one order or another,
        # which now and then moves the nucleus by an entry
        return {"rel": 1e-3, "max": 0.9, "differ": 0.01}
    if k in ("ffn", "attn", "matmul"):
        # (the integer dot is within ~5e-6 of the fp32 chains per layer)
        return {"rel": 3e-5 if case.get("dot") else 2e-6}
    if k in ("moe", "rows", "grouped"):
        # fp32 router sums in one order or another: ~1.3e-6 in the weights
        return {"rel": 3e-5 if case.get("dot") else 6e-6, "max": 1e-3, "differ": 0.005}
    # whole calls: a last-bit difference travels through layers and routing
    return {"rel": 1e-3, "max": 2e-2, "differ": 0.01}


# ───────────────────── the same in 64 bits, plain torch ─────────────────────

def _lsr(z, k):
    return (z >> k) & ((1 << (64 - k)) - 1)


def _i64(v):
    v &= (1 << 64) - 1
    return v - (1 << 64) if v >> 63 else v


def _mix(z):
    z = z + _i64(0x9E3779B97F4A7C15)
    z = (z ^ _lsr(z, 30)) * _i64(0xBF58476D1CE4E5B9)
    z = (z ^ _lsr(z, 27)) * _i64(0x94D049BB133111EB)
    return z ^ _lsr(z, 31)


def _mix_int(z):
    m = (1 << 64) - 1
    z = (z + 0x9E3779B97F4A7C15) & m
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return z ^ (z >> 31)


def _stream(kind, layer=0, index=0, seed=WSEED):
    return _mix_int(seed ^ _mix_int((kind << 56) ^ (layer << 36) ^ index))


def _normal(stream, n, std=0.02, first=0):
    """The synthetic models' values: n floats of a stream from value `first`
    (even) on, in fp32."""
    s, std = _i64(stream), float(np.float32(std))
    c = torch.arange(first // 2, (first + n + 1) // 2, dtype=torch.int64, device="cuda")
    a, b = _mix(_mix(2 * c) ^ s), _mix(_mix(2 * c + 1) ^ s)
    u1 = (_lsr(a, 11) + 1).double() * 2.0 ** -53
    t = 6.283185307179586 * (_lsr(b, 11).double() * 2.0 ** -53)
    r = torch.sqrt(-2.0 * torch.log(u1))
    return torch.stack([r * torch.cos(t) * std, r * torch.sin(t) * std], 1).reshape(-1)[:n].float()


def _quant(w, gs):
    """(scales fp32 [O][groups], the values fp64 that the INT4 form stands for)"""
    O, I = w.shape
    pad = -I % gs
    v = torch.nn.functional.pad(w, (0, pad)).reshape(O, -1, gs)
    amax = v.abs().amax(2)
    s = torch.where(amax > 1e-8, (amax.double() / 7.0).float(), torch.full_like(amax, 1e-8))
    q = torch.round((v.double() / s.double()[:, :, None]).float()).clamp(-8, 7)
    return s, (q.double() * s.double()[:, :, None]).reshape(O, -1)[:, :I]


class _Exact:
    """The synthetic model's functions in fp64."""

    def __init__(self, case):
        kw, _ = _shape(case)
        self.cfg = pa.gptoss_cfg(**kw)
        self.E = self.cfg.n_experts
        self.cache = {}

    def tensor(self, kind, shape, layer=0, index=0):
        n = int(np.prod(shape))
        return _normal(_stream(kind, layer, index), n).double().reshape(shape)

    def expert(self, l, e):
        if (l, e) not in self.cache:
            if len(self.cache) > 160:
                self.cache.clear()
            self.cache[l, e] = (_quant(_normal(_stream(2, l, e), INTER * D).reshape(INTER, D), 64)[1],
                                self.tensor(3, (INTER,), l, e),
                                _quant(_normal(_stream(4, l, e), D * HALF).reshape(D, HALF), 64)[1],
                                self.tensor(5, (D,), l, e))
        return self.cache[l, e]

    def ffn(self, l, e, x):
        gu, gub, dn, dnb = self.expert(l, e)
        y = x @ gu.T + gub
        gate, up = y[:, 0::2].clamp(max=7.0), y[:, 1::2].clamp(-7.0, 7.0)
        act = (up + 1.0) * gate * torch.sigmoid(np.float64(np.float32(1.702)) * gate)
        return act, act @ dn.T + dnb

    def moe(self, l, x):
        lg = x @ self.tensor(6, (self.E, D), l).T + self.tensor(7, (self.E,), l)
        top, sel = torch.topk(lg, TOPK, dim=1)
        w = torch.softmax(top, 1)
        out = torch.zeros_like(x)
        for e in sel.unique().tolist():
            t, j = torch.nonzero(sel == e, as_tuple=True)
            out.index_add_(0, t, w[t, j][:, None] * self.ffn(l, e, x[t])[1])
        return out, w

    def rope(self, v, pos):
        """v [rows][heads][64] at positions pos: fp32 angles as the model defines them, fp64 sines."""
        libm = ctypes.CDLL("libm.so.6")
        libm.powf.restype = libm.logf.restype = ctypes.c_float
        f = np.float32
        powf = lambda a, b: f(libm.powf(ctypes.c_float(a), ctypes.c_float(b)))
        logf = lambda a: f(libm.logf(ctypes.c_float(a)))
        c, theta = self.cfg, f(150000.0)
        edge = lambda beta: f(f(64) * logf(f(f(4096) / f(f(f(beta) * f(2)) * f(math.pi)))) / f(f(2) * logf(theta)))
        lo, hi = max(edge(32.0), f(0)), min(edge(1.0), f(63))
        inv = []
        for j in range(32):
            ext = f(f(1) / powf(theta, f(f(2) * f(j)) / f(64)))
            ef = f(1) - min(max(f(f(j) - lo) / f(hi - lo), f(0)), f(1))
            inv.append(f(float(f(ext / f(32))) * float(f(f(1) - ef)) + float(f(ext * ef))))
        ang = torch.from_numpy(np.asarray(pos, np.float32)[:, None] * np.array(inv, np.float32)).cuda().double()
        at = float(c.rope_attn_factor)
        cs, sn = (torch.cos(ang) * at)[:, None, :], (torch.sin(ang) * at)[:, None, :]
        a, b = v[..., :32], v[..., 32:]
        return torch.cat([a * cs - b * sn, a * sn + b * cs], -1)

    def kv(self, seq, l, n):
        s = (5 * 0x9E3779B97F4A7C15 + (seq * 1024 + l) * 2) & ((1 << 64) - 1)
        get = lambda t: _normal(t, n * KVH * HD, 1.0).double().reshape(n, KVH, HD)
        return get(s), get((s + 1) & ((1 << 64) - 1))

    def attention(self, l, x, pos, past):
        """Rows x at positions pos.. over `past` (K, V), which grow by them."""
        n = len(x)
        q = (x @ self.tensor(8, (H * HD, D), l).T + self.tensor(12, (H * HD,), l)).reshape(n, H, HD)
        k = (x @ self.tensor(9, (KVH * HD, D), l).T + self.tensor(13, (KVH * HD,), l)).reshape(n, KVH, HD)
        v = (x @ self.tensor(10, (KVH * HD, D), l).T + self.tensor(14, (KVH * HD,), l)).reshape(n, KVH, HD)
        at = np.arange(pos, pos + n)
        q, k = self.rope(q, at), self.rope(k, at)
        K, V = torch.cat([past[0], k]), torch.cat([past[1], v])
        sinks = self.tensor(16, (H,), l)
        row, col = torch.arange(pos, pos + n, device="cuda")[:, None], torch.arange(len(K), device="cuda")[None]
        seen = (col <= row) & ((col > row - 128) if self.cfg.layer_type[l] == 0 else (col >= 0))
        out = torch.empty_like(q)
        for h in range(H):
            sc = q[:, h] @ K[:, h // 8].T * 0.125
            sc = sc.masked_fill(~seen, -math.inf)
            p = torch.softmax(torch.cat([sc, sinks[h].expand(n, 1)], 1), 1)[:, :-1]
            out[:, h] = p @ V[:, h // 8].contiguous()
        return out.reshape(n, H * HD) @ self.tensor(11, (D, H * HD), l).T + self.tensor(15, (D,), l), (K, V)

    def norm(self, x):
        return x / torch.sqrt((x * x).mean(1, keepdim=True) + np.float64(np.float32(1e-5)))

    def embed(self, ids):
        return torch.stack([_normal(_stream(17), D, first=int(t) * D) for t in ids]).double()

    def forward(self, ids, pos, past):
        x = self.embed(ids)
        for l in range(self.cfg.n_layers):
            a, past[l] = self.attention(l, self.norm(x), pos, past[l])
            x = x + a
            x = x + self.moe(l, self.norm(x))[0]
        return x

    def logits(self, x):
        h, out, step = self.norm(x[-1:])[0], [], 1 << 14
        for r in range(0, VOCAB, step):
            n = min(step, VOCAB - r)
            out.append(_normal(_stream(18), n * D, first=r * D).double().reshape(n, D) @ h)
        return torch.cat(out)


def _exact_sample(case, lg):
    rng, hist, toks, probs, f = 88172645463325252, [], [], [], np.float32
    for d in range(case["draws"]):
        v = lg[d].double()
        if case["penalty"] > 1.0:
            pen = np.float64(f(case["penalty"]))
            for t in hist:
                v[t] = v[t] / pen if v[t] > 0 else v[t] * pen
        v = v * np.float64(f(1) / f(case["temperature"]))
        if case["top_k"]:
            v = torch.where(v < torch.topk(v, case["top_k"])[0][-1], torch.full_like(v, -1e30), v)
        p = torch.softmax(v, 0)
        if case["top_p"] < 1.0:
            s, i = torch.sort(p, descending=True, stable=True)
            cut = int((torch.cumsum(s, 0) < np.float64(f(case["top_p"]))).sum()) + 1
            p[i[cut:]] = 0.0
            p = p / p.sum()
        rng ^= (rng << 13) & ((1 << 64) - 1)
        rng ^= rng >> 7
        rng ^= (rng << 17) & ((1 << 64) - 1)
        r = float(f(f(rng >> 33) / f(1 << 31)))
        hist.append(min(int((torch.cumsum(p, 0) < r).sum()), VOCAB - 1))
        probs.append(p)
    return dict(toks=None, probs=torch.stack(probs))


def exact(case, seed):
    k, st = case["kind"], _inputs(case, seed)
    if k == "sample":
        return _exact_sample(case, st["logits"])
    if k == "quantize":
        return dict(packed=None, scales=_quant(st["w"], case["gs"])[0].double())
    if k == "matmul":
        q, s = _qt_weights(case)
        I, rows = case["I"], []
        for r in range(0, case["O"], 1 << 14):
            w = q[r:r + (1 << 14)]
            if case["fmt"].startswith("int4"):
                w = torch.stack([(w & 15), (w >> 4)], 2).reshape(len(w), -1)[:, :I].double() - 8.0
            w = w.double()
            if s is not None:
                sc = s[r:r + (1 << 14)].double().reshape(len(w), -1)
                w = w * (sc.repeat_interleave(64, 1)[:, :I] if case["fmt"] == "int4_gs" else sc)
            rows.append(st["x"].double() @ w.T)
        return dict(y=torch.cat(rows, 1))
    m = _Exact(case)
    if k == "ffn":
        got = [[m.ffn(0, e, st["x"][c:c + 1].double()) for e in st["ids"][c].tolist()] for c in range(case["calls"])]
        return dict(act=torch.stack([torch.cat([a for a, _ in r]) for r in got]),
                    out=torch.stack([torch.cat([o for _, o in r]) for r in got]))
    if k == "moe":
        return dict(out=torch.stack([m.moe(l, st["x"].double())[0] for l in range(case["layers"])], 1))
    if k in ("rows", "grouped"):
        out, w = m.moe(0, st["x"].double())
        return dict(out=out, sel=None, w=w) if k == "rows" else dict(out=out)
    if k == "attn":
        return dict(out=torch.cat([m.attention(l, st["x"][l:l + 1].double(), case["pos"], m.kv(0, l, case["pos"]))[0]
                                   for l in range(2)]))
    L, none = case["layers"], torch.empty((0, KVH, HD), dtype=torch.float64, device="cuda")
    if k == "prompt":
        past = [(none, none)] * L
        x = m.forward(st["ids"][:case["n"]], 0, past)
        x = m.forward(st["ids"][case["n"]:], case["n"], past)
        return dict(next=None, logits=m.logits(x))
    past, tok = [m.kv(0, l, case["pos"]) for l in range(L)], int(st["ids"][0])
    for s in range(case["steps"]):
        tok = int(m.logits(m.forward([tok], case["pos"] + s, past)).argmax())
    return dict(toks=None, logits=m.logits(m.forward([tok], case["pos"] + case["steps"], past)))
