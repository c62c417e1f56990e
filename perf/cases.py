"""Performance cases of the quantized decode / ragged-prefill path, through its public entry points.

The sizes are those of the hybrid benchmark model (halo_amd.c4_config): hidden 2048, 16 query heads and 2 kv heads of
256, 16 key / 32 value DeltaNet heads of 128, 512 experts of 512 with top-10 routing and a shared expert, vocabulary
151,936. Decode operators are recorded into a graph over several layers with weights, states or caches of their own,
as a decode step replays them: no layer finds its weights left on the chip by the pass before. Prefill operators and
the sampler are called directly.
"""
from __future__ import annotations

import ctypes
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "halo-flash_amd"))
import halo_amd as H  # noqa: E402

HIDDEN, HEADS, KV_HEADS, HEAD = 2048, 16, 2, 256
KEY_HEADS, VALUE_HEADS, STATE = 16, 32, 128
EXPERTS, USED, FF = 512, 10, 512
VOCAB = 151936
PAGE = 16
ROTARY, THETA, EPS = 64, 1e7, 1e-6
# the layers that one recorded decode pass runs: all DeltaNet and attention layers of the 48-layer model
PROJ_LAYERS, MOE_LAYERS, GDN_LAYERS, ATTN_LAYERS, MODEL_LAYERS = 12, 4, 36, 12, 4
# projections of one model layer, (rows, cols): DeltaNet qkv, q | gate and z, output, k or v, alpha | beta
GEMMS = [(8192, 2048), (4096, 2048), (2048, 4096), (512, 2048), (64, 2048)]
# filters of a request: greedy, plain temperature, top-k with top-p, top-p alone, min-p
FILTERS = {
    "greedy": dict(temperature=0.0),
    "temperature": dict(temperature=1.0),
    "top_k": dict(temperature=0.7, top_k=40, top_p=0.95),
    "top_p": dict(temperature=0.8, top_p=0.9),
    "min_p": dict(temperature=1.0, min_p=0.05),
}


def listed():
    return [
        # One token through an attention layer's projections in each of 12 layers: the launch-bound end of decode.
        {"name": "proj_1", "kind": "proj", "tokens": 1},
        # A prompt of ragged length through the DeltaNet input projection: prefill's plain matrix product.
        {"name": "gemm_1500", "kind": "gemm", "tokens": 1500, "rows": 8192, "cols": 2048},
        # Four sessions' tokens through routed experts and the shared expert, 4 layers of one decode step.
        {"name": "moe_decode_4", "kind": "moe_decode", "tokens": 4},
        # A long prompt's MoE layer: router product, grouping by expert, grouped matrix products, combine.
        {"name": "moe_prefill_5000", "kind": "moe_prefill", "tokens": 5000},
        # Four sessions' recurrent states advanced by one token in all 36 DeltaNet layers.
        {"name": "gdn_decode_4", "kind": "gdn_decode", "sessions": 4},
        # The benchmark's ragged batch of prompts through one DeltaNet layer.
        {"name": "gdn_prefill_ragged", "kind": "gdn_prefill", "lengths": "37 512 2048 8191"},
        # A single conversation's decode attention at 8.5 K positions, in all 12 attention layers.
        {"name": "attn_decode_1", "kind": "attn_decode", "sessions": 1, "prefix": 0, "context": 8576},
        # Four sessions that share a long system prompt.
        {"name": "attn_decode_4", "kind": "attn_decode", "sessions": 4, "prefix": 8192, "context": 8576},
        # Causal attention of one 8192-token prompt, one layer.
        {"name": "attn_prefill_8192", "kind": "attn_prefill", "starts": "0", "lengths": "8192"},
        # One request's draw from its logits, called directly: the smallest call.
        {"name": "sample_top_p", "kind": "sample", "rows": 1, "vocab": VOCAB, "filter": "top_p"},
        # Four sessions after a shared prompt, 16 decode steps each through a 4-layer stack and the head.
        {"name": "model_decode_4", "kind": "model_decode", "sessions": 4, "prefix": 8192, "steps": 16},
        # Ingestion of one long prompt through a 4-layer stack (three DeltaNet layers and one attention) and the head.
        {"name": "model_prefill_8000", "kind": "model_prefill", "lengths": "8000"},
    ]


def _spread(rng, low, high):
    """A whole number of [low, high], even over the logarithm."""
    return min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def _lengths(rng, total, most):
    """1 to `most` ragged prompt lengths that sum to `total` at the most."""
    n = rng.randint(1, most)
    return [_spread(rng, 16, total // n) for _ in range(n)]


def draw(rng):
    kind = rng.choice(["proj", "gemm", "moe_decode", "moe_prefill", "gdn_decode", "gdn_prefill", "attn_decode",
                       "attn_prefill", "sample", "model_decode", "model_prefill"])
    text = lambda v: " ".join(str(x) for x in v)  # noqa: E731
    if kind == "proj":
        return {"kind": kind, "tokens": rng.randint(2, 16)}
    if kind == "gemm":
        rows, cols = rng.choice(GEMMS)
        return {"kind": kind, "tokens": _spread(rng, 17, 8192), "rows": rows, "cols": cols}
    if kind == "moe_decode":
        return {"kind": kind, "tokens": rng.choice([1, 2, 3, *range(5, 17)])}
    if kind == "moe_prefill":
        return {"kind": kind, "tokens": _spread(rng, 33, 8192)}
    if kind == "gdn_decode":
        return {"kind": kind, "sessions": rng.choice([1, 2, 3, 5, 6, 7, 8])}
    if kind == "gdn_prefill":
        return {"kind": kind, "lengths": text(_lengths(rng, 10788, 4))}
    if kind == "attn_decode":
        sessions = rng.randint(1, 4)
        prefix = 64 * rng.randint(0, 128) if sessions > 1 else 0
        return {"kind": kind, "sessions": sessions, "prefix": prefix,
                "context": prefix + _spread(rng, 65, 2048 if sessions > 1 else 16384)}
    if kind == "attn_prefill":
        lengths = _lengths(rng, 6144, 4)
        return {"kind": kind, "starts": text(rng.choice([0, rng.randint(1, 2048)]) for _ in lengths),
                "lengths": text(lengths)}
    if kind == "sample":
        return {"kind": kind, "rows": rng.randint(1, 8), "vocab": _spread(rng, 8192, VOCAB),
                "filter": rng.choice(sorted(FILTERS))}
    if kind == "model_decode":
        return {"kind": kind, "sessions": rng.randint(1, 4), "prefix": 64 * rng.randint(1, 128),
                "steps": rng.randint(4, 16)}
    return {"kind": kind, "lengths": text(_lengths(rng, 7999, 4))}


# ---- inputs ----------------------------------------------------------------------------------------------------------

class _Source:
    """Seeded tensors on the GPU, in the order in which they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)

    def normal(self, *shape, sigma=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * sigma

    def q8(self, rows, cols):
        """A repacked Q8_0 matrix: values uniform in -127 .. 127, scales |N(0, 0.02)| / 127."""
        qs = torch.randint(-127, 128, (rows, cols), generator=self.g, device="cuda", dtype=torch.int8)
        return qs, (self.normal(rows, cols // 32).abs() * (0.02 / 127)).half()


def _dense(w):
    """The values of a Q8_0 matrix in 64 bits."""
    qs, d = w
    return (qs.double().unflatten(-1, (-1, 32)) * d.double().unsqueeze(-1)).flatten(-2)


def _codes(x):
    """Activation rows as the int8 quantizer defines them (scale amax / 127, round half to even), in 64 bits."""
    b = x.unflatten(-1, (-1, 32))
    top = b.abs().amax(-1, keepdim=True)
    s = top / torch.full_like(top, 127)  # a true division: by a plain number torch multiplies with the reciprocal
    q = torch.where(s > 0, (b / torch.where(s > 0, s, torch.ones_like(s))).round(), torch.zeros_like(b))
    return (q.double() * s.double()).flatten(-2)


def _numbers(text):
    return [int(v) for v in str(text).split()]


def _proj_inputs(case, seed):
    s, M = _Source(seed), case["tokens"]
    return [dict(x=s.normal(M, HIDDEN), a=s.normal(M, HEADS * HEAD), qg=s.q8(4096, 2048), kv=s.q8(512, 2048),
                 o=s.q8(2048, 4096)) for _ in range(PROJ_LAYERS)]


def _gemm_inputs(case, seed):
    s = _Source(seed)
    return dict(x=s.normal(case["tokens"], case["cols"]), w=s.q8(case["rows"], case["cols"]))


def _moe_inputs(case, seed, layers):
    s, T = _Source(seed), case["tokens"]
    return [dict(x=s.normal(T, HIDDEN), router=s.normal(EXPERTS, HIDDEN, sigma=0.02),
                 shared=s.normal(HIDDEN, sigma=0.02), gate=s.q8(EXPERTS * FF, HIDDEN), up=s.q8(EXPERTS * FF, HIDDEN),
                 down=s.q8(EXPERTS * HIDDEN, FF), sgate=s.q8(FF, HIDDEN), sup=s.q8(FF, HIDDEN),
                 sdown=s.q8(HIDDEN, FF)) for _ in range(layers)]


def _gdn_inputs(seed, shape, states):
    """q and k of unit length, v, log-decay and beta of `shape` tokens, and the states they meet."""
    s = _Source(seed)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)  # noqa: E731
    return dict(q=unit(s.normal(*shape, KEY_HEADS, STATE)), k=unit(s.normal(*shape, KEY_HEADS, STATE)),
                v=s.normal(*shape, VALUE_HEADS, STATE),
                g=-torch.nn.functional.softplus(s.normal(*shape, VALUE_HEADS)),
                beta=torch.sigmoid(s.normal(*shape, VALUE_HEADS)),
                state=s.normal(*states, VALUE_HEADS, STATE, STATE, sigma=0.1))


def _pages(source, sessions, prefix, context):
    """A page table over scattered physical pages, the prefix's shared by all sessions, and the number of pages."""
    n, shared = -(-context // PAGE), prefix // PAGE
    total = shared + sessions * (n - shared)
    order = torch.randperm(total, generator=source.g, device="cuda").to(torch.int32)
    own = order[shared:].view(sessions, n - shared)
    return torch.cat([order[:shared].expand(sessions, shared), own], 1).contiguous(), total


def _attn_decode_inputs(case, seed):
    s, S, L = _Source(seed), case["sessions"], ATTN_LAYERS
    table, total = _pages(s, S, case["prefix"], case["context"])
    # ragged: every session is within its last page, the first one at the full context
    nkv = torch.tensor([case["context"] - min(11 * i, case["context"] - case["prefix"] - 1) for i in range(S)],
                       dtype=torch.int32, device="cuda")
    return dict(table=table, nkv=nkv, k_pool=s.normal(L, total, KV_HEADS, PAGE, HEAD),
                v_pool=s.normal(L, total, KV_HEADS, PAGE, HEAD), qg=s.normal(L, S, HEADS, 2 * HEAD),
                k=s.normal(L, S, KV_HEADS, HEAD), v=s.normal(L, S, KV_HEADS, HEAD),
                q_norm=1 + s.normal(L, HEAD, sigma=0.02), k_norm=1 + s.normal(L, HEAD, sigma=0.02))


def _attn_prefill_inputs(case, seed):
    s, starts, lengths = _Source(seed), _numbers(case["starts"]), _numbers(case["lengths"])
    T, context = sum(lengths), max(a + n for a, n in zip(starts, lengths))
    table, total = _pages(s, len(starts), 0, context)
    return dict(table=table, context=context, q=s.normal(T, HEADS, HEAD), gate=s.normal(T, HEADS, HEAD),
                k_pool=s.normal(total, KV_HEADS, PAGE, HEAD), v_pool=s.normal(total, KV_HEADS, PAGE, HEAD))


# ---- states ----------------------------------------------------------------------------------------------------------

_DEVICE = None


def _device():
    global _DEVICE
    if _DEVICE is None:
        _DEVICE = H.Device()
    return _DEVICE


class _State:
    """What a program holds between calls: tensors, descriptors, and a recorded graph or a model."""

    def __init__(self, call=None, out=None, keep=(), record=False):
        self.dev, self.call, self.out, self.keep, self.graph, self.model = _device(), call, out, keep, None, None
        if record:
            torch.cuda.synchronize()
            self.dev.begin_capture()
            call()
            self.graph = self.dev.end_capture()
        torch.cuda.synchronize()

    def __del__(self):
        try:
            if self.graph is not None:
                self.dev.free_graph(self.graph)
            if self.model is not None:
                self.model.close()
        except Exception:
            pass


def _matrix(w):
    qs, d = w
    return H.Q8Matrix(qs.data_ptr(), d.data_ptr(), qs.shape[0], qs.shape[1], qs.shape[1], 0)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _prepare_proj(case, seed):
    dev, M, layers, out, todo = _device(), case["tokens"], _proj_inputs(case, seed), [], []
    for t in layers:
        ys = [_empty(M, 4096), _empty(M, 512), _empty(M, 2048)]
        mats = (H.Q8Matrix * 3)(_matrix(t["qg"]), _matrix(t["kv"]), _matrix(t["o"]))
        outs = (ctypes.c_void_p * 3)(*[y.data_ptr() for y in ys])
        q = [_empty(M, 2048, dtype=torch.int8), _empty(M, 64), _empty(M, 4096, dtype=torch.int8), _empty(M, 128)]
        if M == 1:
            inp = [H.ProjInput(x=t["x"].data_ptr(), mode=H.PROJ_F), H.ProjInput(x=t["a"].data_ptr(), mode=H.PROJ_F)]
        else:
            inp = [H.ProjInput(xq=q[0].data_ptr(), xs=q[1].data_ptr(), mode=H.PROJ_Q),
                   H.ProjInput(xq=q[2].data_ptr(), xs=q[3].data_ptr(), mode=H.PROJ_Q)]
        todo.append((t, mats, outs, q, inp))
        out.append(ys)

    def call():
        for t, mats, outs, q, inp in todo:
            if M == 1:
                dev.op("proj_q8", mats, outs, 2, ctypes.byref(inp[0]), 1)
                dev.op("proj_q8", ctypes.cast(ctypes.byref(mats, 2 * ctypes.sizeof(H.Q8Matrix)),
                                              ctypes.POINTER(H.Q8Matrix)),
                       ctypes.cast(ctypes.byref(outs, 2 * ctypes.sizeof(ctypes.c_void_p)),
                                   ctypes.POINTER(ctypes.c_void_p)), 1, ctypes.byref(inp[1]), 1)
            else:
                dev.op("quantize_q8_pair", t["x"].data_ptr(), q[0].data_ptr(), q[1].data_ptr(), 2048,
                       t["a"].data_ptr(), q[2].data_ptr(), q[3].data_ptr(), 4096, M)
                dev.op("proj_q8_pair", mats, outs, 2, ctypes.byref(inp[0]), ctypes.byref(inp[1]), M)

    stacked = [[ys[i] for ys in out] for i in range(3)]
    return _State(call, {"qg": stacked[0], "kv": stacked[1], "o": stacked[2]}, (layers, todo), record=True)


def _prepare_gemm(case, seed):
    dev, t = _device(), _gemm_inputs(case, seed)
    M, rows, cols = case["tokens"], case["rows"], case["cols"]
    xq, xs, y, m = _empty(M, cols, dtype=torch.int8), _empty(M, cols // 32), _empty(M, rows), _matrix(t["w"])

    def call():
        dev.op("quantize_q8", t["x"].data_ptr(), xq.data_ptr(), xs.data_ptr(), M, cols)
        dev.op("matvec_q8a8", ctypes.byref(m), xq.data_ptr(), xs.data_ptr(), y.data_ptr(), M, rows)

    return _State(call, y, (t, xq, xs))


def _moe_weights(t):
    return H.MoeWeights(router=t["router"].data_ptr(), shared_gate=t["shared"].data_ptr(), gate=_matrix(t["gate"]),
                        up=_matrix(t["up"]), down=_matrix(t["down"]), shared_gate_proj=_matrix(t["sgate"]),
                        shared_up=_matrix(t["sup"]), shared_down=_matrix(t["sdown"]), n_experts=EXPERTS, n_used=USED,
                        hidden=HIDDEN, ff=FF, shared_ff=FF)


def _prepare_moe_decode(case, seed):
    dev, T, layers = _device(), case["tokens"], _moe_inputs(case, seed, MOE_LAYERS)
    ws = [_moe_weights(t) for t in layers]
    out = [_empty(T, HIDDEN) for _ in layers]
    work = _empty(H.lib().halo_op_moe_workspace_bytes(ctypes.byref(ws[0]), T), dtype=torch.uint8)

    def call():
        for t, w, y in zip(layers, ws, out):
            dev.op("moe_decode", ctypes.byref(w), t["x"].data_ptr(), y.data_ptr(), T, work.data_ptr(), work.numel())

    return _State(call, out, (layers, work), record=True)


def _prepare_moe_prefill(case, seed):
    dev, T, t = _device(), case["tokens"], _moe_inputs(case, seed, 1)[0]
    w, out = _moe_weights(t), _empty(case["tokens"], HIDDEN)
    work = _empty(H.lib().halo_op_moe_prefill_workspace_bytes(ctypes.byref(w), T), dtype=torch.uint8)

    def call():
        dev.op("moe_prefill", ctypes.byref(w), t["x"].data_ptr(), out.data_ptr(), T, work.data_ptr(), work.numel())

    return _State(call, out, (t, work))


def _prepare_gdn_decode(case, seed):
    dev, S = _device(), case["sessions"]
    t = _gdn_inputs(seed, (GDN_LAYERS, S), (GDN_LAYERS, S))
    o = _empty(GDN_LAYERS, S, VALUE_HEADS, STATE)

    def call():
        for i in range(GDN_LAYERS):
            p = [t[n][i].data_ptr() for n in ("state", "q", "k", "v", "g", "beta")]
            dev.op("gdn_decode", *p, o[i].data_ptr(), S, VALUE_HEADS, KEY_HEADS, STATE)

    return _State(call, {"o": o, "state": t["state"]}, t, record=True)


def _prepare_gdn_prefill(case, seed):
    dev, lengths = _device(), _numbers(case["lengths"])
    t = _gdn_inputs(seed, (sum(lengths),), (len(lengths),))
    for n in ("q", "k", "v"):
        t[n] = t[n].bfloat16()
    lens = np.array(lengths, np.uint32)
    n = H.lib().halo_gdn_chunk_table(lens.ctypes.data, len(lengths), None, None)
    chunks, seqs = np.zeros((n, 3), np.uint32), np.zeros((len(lengths), 2), np.uint32)
    H.lib().halo_gdn_chunk_table(lens.ctypes.data, len(lengths), chunks.ctypes.data, seqs.ctypes.data)
    chunks, seqs = (torch.from_numpy(a.view(np.int32)).cuda() for a in (chunks, seqs))
    o = _empty(sum(lengths), VALUE_HEADS, STATE)
    work = _empty(H.lib().halo_op_gdn_prefill_workspace_bytes(n, VALUE_HEADS), dtype=torch.uint8)

    def call():
        p = [t[name].data_ptr() for name in ("q", "k", "v", "g", "beta")]
        dev.op("gdn_prefill", *p, chunks.data_ptr(), seqs.data_ptr(), n, len(lengths), t["state"].data_ptr(),
               o.data_ptr(), VALUE_HEADS, KEY_HEADS, STATE, work.data_ptr(), work.numel())

    return _State(call, {"o": o, "state": t["state"]}, t)


def _prepare_attn_decode(case, seed):
    dev, S, t = _device(), case["sessions"], _attn_decode_inputs(case, seed)
    L, A = ATTN_LAYERS, HEADS * HEAD
    kv = [H.PagedKV(t["k_pool"][i].data_ptr(), t["v_pool"][i].data_ptr(), t["table"].data_ptr(), t["nkv"].data_ptr(),
                    S, KV_HEADS, HEAD, t["table"].shape[1], case["prefix"], case["context"]) for i in range(L)]
    o, oq, os_ = _empty(L, S, A), _empty(L, S, A, dtype=torch.int8), _empty(L, S, A // 32)
    work = _empty(H.lib().halo_op_attn_decode_workspace_bytes(ctypes.byref(kv[0]), HEADS), dtype=torch.uint8)

    def call():
        for i in range(L):
            p = [t[n][i].data_ptr() for n in ("qg", "k", "v", "q_norm", "k_norm")]
            dev.op("attn_decode_step_q8", ctypes.byref(kv[i]), *p, ROTARY, THETA, EPS, o[i].data_ptr(),
                   oq[i].data_ptr(), os_[i].data_ptr(), HEADS, work.data_ptr(), work.numel())

    return _State(call, {"o": o, "oq": oq, "os": os_, "k_pool": t["k_pool"], "v_pool": t["v_pool"]}, (t, kv),
                  record=True)


def _prepare_attn_prefill(case, seed):
    dev, t = _device(), _attn_prefill_inputs(case, seed)
    starts, lengths = _numbers(case["starts"]), _numbers(case["lengths"])
    T, A = sum(lengths), HEADS * HEAD
    segs = (H.PrefillSegment * len(starts))(*[H.PrefillSegment(i, a, n, sum(lengths[:i]))
                                              for i, (a, n) in enumerate(zip(starts, lengths))])
    kv = H.PagedKV(t["k_pool"].data_ptr(), t["v_pool"].data_ptr(), t["table"].data_ptr(), None, len(starts), KV_HEADS,
                   HEAD, t["table"].shape[1], 0, t["context"])
    o, oq, os_ = _empty(T, A), _empty(T, A, dtype=torch.int8), _empty(T, A // 32)
    work = _empty(H.lib().halo_op_attn_prefill_workspace_bytes(segs, len(starts)), dtype=torch.uint8)

    def call():
        dev.op("attn_prefill", ctypes.byref(kv), segs, len(starts), t["q"].data_ptr(), t["gate"].data_ptr(),
               o.data_ptr(), oq.data_ptr(), os_.data_ptr(), HEADS, work.data_ptr(), work.numel())

    return _State(call, {"o": o, "oq": oq, "os": os_}, (t, work))


def _prepare_sample(case, seed):
    dev, rows, V = _device(), case["rows"], case["vocab"]
    s = _Source(seed)
    logits = s.normal(rows, V, sigma=3.0)
    prm = (H.SampleParams * rows)()
    for r in range(rows):
        prm[r] = H.SampleParams(top_p=1.0, repeat_penalty=1.0, vocab=V, rng=(int(seed) + 1) * 1000003 + r)
        for k, v in FILTERS[case["filter"]].items():
            setattr(prm[r], k, v)
    params = torch.frombuffer(bytearray(bytes(prm)), dtype=torch.uint8).cuda()
    out = _empty(rows, 16, dtype=torch.uint8)
    work = _empty(H.lib().halo_op_sample_workspace_bytes(rows, V), dtype=torch.uint8)

    def call():
        dev.op("sample", logits.data_ptr(), rows, V, V, params.data_ptr(), None, 0, out.data_ptr(), work.data_ptr(),
               work.numel())

    return _State(call, out, (logits, params, work))


def _model(seed, sessions, prefix, context):
    cfg = H.c4_config(max_sessions=sessions, prefix_tokens=prefix, max_context=context)
    cfg.layers = MODEL_LAYERS
    return H.Model(_device(), cfg, seed=int(seed))


def _prepare_model_decode(case, seed):
    S, P, steps = case["sessions"], case["prefix"], case["steps"]
    m = _model(seed, S, P, P + steps + 16)
    rng = np.random.default_rng(int(seed))
    prefix = rng.integers(0, VOCAB, P)
    prompts = [np.concatenate([prefix, rng.integers(0, VOCAB, steps)]).astype(np.uint32) for _ in range(S)]
    m.set_session(0, prompts[0])
    m.prefill([(0, 0, P)])
    for s in range(1, S):
        m.fork(0, s)

    def call():
        for s in range(S):  # back to the end of the shared prompt: the turn is decoded anew
            m.set_session(s, prompts[s], nkv=P)
        m.run(S, steps, prefix=P if S > 1 else 0)  # the turn's own tokens, one decode step each
        return [m.logits(s) for s in range(S)]

    state = _State(call)
    state.model = m
    return state


def _prepare_model_prefill(case, seed):
    lengths = _numbers(case["lengths"])
    m = _model(seed, len(lengths), 0, max(lengths) + 16)
    rng = np.random.default_rng(int(seed))
    prompts = [rng.integers(0, VOCAB, n).astype(np.uint32) for n in lengths]
    for s, p in enumerate(prompts):  # a server has its prefill buffers from an earlier request
        m.set_session(s, p)
    m.prefill([(s, 0, n) for s, n in enumerate(lengths)])

    def call():
        m.reset()
        for s, p in enumerate(prompts):
            m.set_session(s, p)
        m.prefill([(s, 0, n) for s, n in enumerate(lengths)])
        return [m.logits(s) for s in range(len(lengths))]

    state = _State(call)
    state.model = m
    return state


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    if state.graph is not None:
        state.dev.launch_graph(state.graph)
        return state.out
    out = state.call()
    return state.out if out is None else out


# ---- work ------------------------------------------------------------------------------------------------------------

def _q8_bytes(rows, cols):
    return rows * (cols // 32) * 34


def _distinct(tokens):
    """Experts that `tokens` tokens are routed to between them, expected."""
    return EXPERTS * (1 - (1 - USED / EXPERTS) ** tokens)


def _moe_work(T):
    one = 2 * _q8_bytes(FF, HIDDEN) + _q8_bytes(HIDDEN, FF)
    return ((EXPERTS + 1) * HIDDEN * 4 + (1 + _distinct(T)) * one + 2 * T * HIDDEN * 4,
            2 * T * HIDDEN * (EXPERTS + 1) + 2 * T * (USED + 1) * 3 * HIDDEN * FF)


def _gdn_work(tokens, sequences, item):
    state = VALUE_HEADS * STATE * STATE
    return (sequences * state * 8 + tokens * (item * STATE * (2 * KEY_HEADS + VALUE_HEADS) + 4 * STATE * VALUE_HEADS
                                              + 8 * VALUE_HEADS), 6 * tokens * state)


def _attn_work(rows, queries, pairs):
    """Cache rows read, tokens attending, and (token, position) pairs scored per query head."""
    return (rows * KV_HEADS * HEAD * 8 + queries * HEADS * HEAD * 12, 4 * HEADS * HEAD * pairs)


def _layer_weights():
    """Q8_0 weights of three DeltaNet layers' and one attention layer's projections (values)."""
    return 3 * HIDDEN * (8192 + 4096 + 64 + 4096) + HIDDEN * (8192 + 1024 + 4096)


def work(case):
    kind = case["kind"]
    if kind == "proj":
        M, w = case["tokens"], [(4096, 2048), (512, 2048), (2048, 4096)]
        b = sum(_q8_bytes(*s) for s in w) + M * 4 * (2048 + 4096 + 4096 + 512 + 2048)
        b, f = PROJ_LAYERS * b, PROJ_LAYERS * 2 * M * sum(r * c for r, c in w)
    elif kind == "gemm":
        M, r, c = case["tokens"], case["rows"], case["cols"]
        b, f = _q8_bytes(r, c) + 4 * M * (r + c), 2 * M * r * c
    elif kind in ("moe_decode", "moe_prefill"):
        n = MOE_LAYERS if kind == "moe_decode" else 1
        b, f = (n * v for v in _moe_work(case["tokens"]))
    elif kind == "gdn_decode":
        b, f = (GDN_LAYERS * v for v in _gdn_work(case["sessions"], case["sessions"], 4))
    elif kind == "gdn_prefill":
        n = _numbers(case["lengths"])
        b, f = _gdn_work(sum(n), len(n), 2)
    elif kind == "attn_decode":
        S, P, n = case["sessions"], case["prefix"], case["context"]
        b, f = (ATTN_LAYERS * v for v in _attn_work(P + S * (n - P), S, S * n))
    elif kind == "attn_prefill":
        n = list(zip(_numbers(case["starts"]), _numbers(case["lengths"])))
        b, f = _attn_work(sum(a + l for a, l in n), sum(l for _, l in n), sum(a * l + l * (l + 1) // 2 for a, l in n))
    elif kind == "sample":
        b, f = case["rows"] * case["vocab"] * 4, 0
    elif kind == "model_decode":
        S, P, n = case["sessions"], case["prefix"], case["steps"]
        moe, gdn = _moe_work(S), _gdn_work(S, S, 4)
        attn = _attn_work(P + S * n // 2, S, S * (P + n // 2))
        w = _layer_weights() + VOCAB * HIDDEN
        b = n * (w * 34 / 32 + 4 * moe[0] + 3 * gdn[0] + attn[0] + 4 * S * VOCAB)
        f = n * (2 * S * w + 4 * moe[1] + 3 * gdn[1] + attn[1])
    else:
        n = _numbers(case["lengths"])
        T = sum(n)
        moe, gdn = _moe_work(T), _gdn_work(T, len(n), 4)
        attn = _attn_work(sum(n), T, sum(l * (l + 1) // 2 for l in n))
        b = _q8_bytes(1, _layer_weights() + VOCAB * HIDDEN) + 4 * moe[0] + 3 * gdn[0] + attn[0]
        f = 2 * T * _layer_weights() + 2 * len(n) * VOCAB * HIDDEN + 4 * moe[1] + 3 * gdn[1] + attn[1]
    return {"bytes": b, "flops": f}


# ---- what another correct implementation may differ by ---------------------------------------------------------------

def tolerance(case):
    # about four times the distance from 64 bits (for whole models: between prefill in one batch, in two, and decode).
    # An activation near a rounding boundary takes the next int8 code: hence the quantized outputs' share, and MoE
    # layers whose hidden rows are quantized. Attention decode meets the rotation angle of an fp32 power.
    return {
        "proj": {"rel": 4e-7, "max": 2.5e-6},
        "gemm": {"rel": 8e-7, "max": 8e-6},
        "moe_decode": {"rel": 4e-4, "max": 0.08},
        "moe_prefill": {"rel": 4e-4, "max": 0.08},
        "gdn_decode": {"rel": 6e-7, "max": 4e-6},
        "gdn_prefill": {"rel": 3e-6, "max": 1e-4},
        "attn_decode": {"rel": 2e-4, "max": 4e-3, "differ": 5e-4},
        "attn_prefill": {"rel": 2e-6, "max": 1e-4, "differ": 5e-4},
        "sample": "exact",
        "model_decode": {"rel": 0.03, "max": 0.3},
        "model_prefill": {"rel": 0.03, "max": 0.3},
    }[case["kind"]]


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------

def _exact_proj(case, seed):
    out = {"qg": [], "kv": [], "o": []}
    for t in _proj_inputs(case, seed):
        x, a = _codes(t["x"]), _codes(t["a"])
        out["qg"].append(x @ _dense(t["qg"]).T)
        out["kv"].append(x @ _dense(t["kv"]).T)
        out["o"].append(a @ _dense(t["o"]).T)
    return out


def _exact_gemm(case, seed):
    t = _gemm_inputs(case, seed)
    return _codes(t["x"]) @ _dense(t["w"]).T


def _exact_moe(t):
    x = t["x"]
    prob = torch.softmax(x.double() @ t["router"].double().T, -1)
    top, ids = prob.topk(USED, -1)
    weight = top / top.sum(-1, keepdim=True).clamp(min=2.0 ** -14)
    xq = _codes(x)

    def expert(rows, gate, up, down):
        h = torch.nn.functional.silu(rows @ _dense(gate).T) * (rows @ _dense(up).T)
        return _codes(h) @ _dense(down).T

    part = lambda w, e, n: (w[0][e * n:(e + 1) * n], w[1][e * n:(e + 1) * n])  # noqa: E731
    out = torch.sigmoid(x.double() @ t["shared"].double()).unsqueeze(-1) * expert(xq, t["sgate"], t["sup"], t["sdown"])
    for e in ids.unique().tolist():
        tok, slot = (ids == e).nonzero(as_tuple=True)
        y = expert(xq[tok], part(t["gate"], e, FF), part(t["up"], e, FF), part(t["down"], e, HIDDEN))
        out[tok] += weight[tok, slot].unsqueeze(-1) * y
    return out


def _exact_moe_decode(case, seed):
    return [_exact_moe(t) for t in _moe_inputs(case, seed, MOE_LAYERS)]


def _exact_moe_prefill(case, seed):
    return _exact_moe(_moe_inputs(case, seed, 1)[0])


def _gdn_step(state, q, k, v, g, beta):
    """One token of every leading index: states [..., Hv, d, d] and the outputs, in 64 bits."""
    rep = VALUE_HEADS // KEY_HEADS
    q, k = (torch.cat([t.double()] * rep, -2) for t in (q, k))  # value head h reads key head h % KEY_HEADS
    state = state * g.double().exp()[..., None, None]
    delta = (v.double() - (k.unsqueeze(-2) @ state).squeeze(-2)) * beta.double().unsqueeze(-1)
    state = state + k.unsqueeze(-1) * delta.unsqueeze(-2)
    return state, (q.unsqueeze(-2) @ state).squeeze(-2) / math.sqrt(STATE)


def _exact_gdn_decode(case, seed):
    t = _gdn_inputs(seed, (GDN_LAYERS, case["sessions"]), (GDN_LAYERS, case["sessions"]))
    state, o = _gdn_step(t["state"].double(), t["q"], t["k"], t["v"], t["g"], t["beta"])
    return {"o": o, "state": state}


def _exact_gdn_prefill(case, seed):
    lengths = _numbers(case["lengths"])
    t = _gdn_inputs(seed, (sum(lengths),), (len(lengths),))
    for n in ("q", "k", "v"):
        t[n] = t[n].bfloat16()
    first = torch.tensor([sum(lengths[:i]) for i in range(len(lengths))], device="cuda")
    o = _empty(sum(lengths), VALUE_HEADS, STATE, dtype=torch.float64)
    # longest first, so that the sequences that are still running are a leading slice
    order = sorted(range(len(lengths)), key=lambda i: -lengths[i])
    states, at = t["state"].double()[order], first[order]
    for j in range(max(lengths)):
        n = sum(1 for x in lengths if x > j)
        rows = at[:n] + j
        states[:n], o[rows] = _gdn_step(states[:n], *(t[name][rows] for name in ("q", "k", "v", "g", "beta")))
    back = torch.empty_like(states)
    back[order] = states
    return {"o": o, "state": back}


def _scales(o):
    return o.float().unflatten(-1, (-1, 32)).abs().amax(-1) / 127


def _norm_rope(x, weight, position):
    """RMSNorm of heads, then NEOX rotation of the first ROTARY dims; the angle is fp32 as the model defines it."""
    x = x.double()
    x = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * weight.double()
    freq = (THETA ** (-torch.arange(0, ROTARY, 2, device="cuda", dtype=torch.float64) / ROTARY)).float()
    angle = (position.float()[..., None] * freq).double().unsqueeze(-2)
    a, b = x[..., :ROTARY // 2], x[..., ROTARY // 2:ROTARY]
    return torch.cat([a * angle.cos() - b * angle.sin(), a * angle.sin() + b * angle.cos(), x[..., ROTARY:]], -1)


def _exact_attn_decode(case, seed):
    t, S = _attn_decode_inputs(case, seed), case["sessions"]
    L = ATTN_LAYERS
    o = _empty(L, S, HEADS * HEAD, dtype=torch.float64)
    k_pool, v_pool = t["k_pool"].double(), t["v_pool"].double()
    for i in range(L):
        pos = t["nkv"] - 1
        q = _norm_rope(t["qg"][i][..., :HEAD], t["q_norm"][i], pos)
        k = _norm_rope(t["k"][i], t["k_norm"][i], pos)
        for s in range(S):
            n = int(t["nkv"][s])
            page, slot = int(t["table"][s, (n - 1) // PAGE]), (n - 1) % PAGE
            k_pool[i, page, :, slot], v_pool[i, page, :, slot] = k[s], t["v"][i, s].double()
        for s in range(S):
            n = int(t["nkv"][s])
            pages = t["table"][s, : -(-n // PAGE)].long()
            keys, vals = (p[i][pages].transpose(0, 1).reshape(KV_HEADS, -1, HEAD)[:, :n] for p in (k_pool, v_pool))
            p = torch.softmax(q[s].view(KV_HEADS, -1, HEAD) @ keys.transpose(1, 2).contiguous() / math.sqrt(HEAD), -1)
            y = (p @ vals).reshape(HEADS, HEAD) * torch.sigmoid(t["qg"][i, s, :, HEAD:].double())
            o[i, s] = y.reshape(-1)
    return {"o": o, "oq": None, "os": _scales(o), "k_pool": k_pool, "v_pool": v_pool}


def _exact_attn_prefill(case, seed):
    t, starts, lengths = _attn_prefill_inputs(case, seed), _numbers(case["starts"]), _numbers(case["lengths"])
    o, first = _empty(sum(lengths), HEADS, HEAD, dtype=torch.float64), 0
    for s, (a, n) in enumerate(zip(starts, lengths)):
        pages = t["table"][s].long()
        keys, vals = (p[pages].transpose(0, 1).reshape(KV_HEADS, -1, HEAD)[:, :a + n].double()
                      for p in (t["k_pool"], t["v_pool"]))
        for b in range(0, n, 256):
            m = min(256, n - b)
            rows = slice(first + b, first + b + m)
            pos = torch.arange(a + b, a + b + m, device="cuda")
            q = t["q"][rows].double().view(m, KV_HEADS, -1, HEAD)
            for h in range(KV_HEADS):
                score = q[:, h].reshape(-1, HEAD) @ keys[h].T.contiguous() / math.sqrt(HEAD)
                hide = torch.arange(a + n, device="cuda")[None] > pos.repeat_interleave(HEADS // KV_HEADS)[:, None]
                p = torch.softmax(score.masked_fill_(hide, -math.inf), -1)
                o[rows, h * (HEADS // KV_HEADS):(h + 1) * (HEADS // KV_HEADS)] = (p @ vals[h]).view(m, -1, HEAD)
        first += n
    o = (o * torch.sigmoid(t["gate"].double())).reshape(sum(lengths), -1)
    return {"o": o, "oq": None, "os": _scales(o)}


def exact(case, seed):
    """The same in 64 bits; none for a whole model (its weights are the library's own) and for drawn tokens."""
    if case["kind"] in ("sample", "model_decode", "model_prefill"):
        return None
    return globals()["_exact_" + case["kind"]](case, seed)
