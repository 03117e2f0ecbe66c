"""The work that a program built on this package has it do, as cases that can be timed and compared.

Each case goes through the public entry points: the affine GEMV, the routed-expert decode, one verify layer, a whole
verify round, the draft chain, a prompt chunk through a MoE layer, and the acceptance of a round. `listed` holds one
case per kind of call, from the smallest to the largest; `draw` gives others of the same ranges. Weights, routing bias
(Zipf 1.1) and logits are the package's seeded synthetic ones (slotstream_spark_amd.memory.synth).
"""
import math

import numpy as np
import torch

from slotstream_spark_amd.engine.accept import Acceptor, UniformStream
from slotstream_spark_amd.engine.mtp import DraftGraph, MTPHead
from slotstream_spark_amd.engine.prefill import MoEPrefillLayer
from slotstream_spark_amd.engine.sampler import SampleParams
from slotstream_spark_amd.engine.step import MoEWeights, MTPStepGraph
from slotstream_spark_amd.engine.verify import MoEVerifyLayer
from slotstream_spark_amd.kernels.gemv_affine import gemv
from slotstream_spark_amd.kernels.moe_gemv_affine import moe_decode, record_layout
from slotstream_spark_amd.memory.slot_pool import SlotPool
from slotstream_spark_amd.memory.synth import (LayerWeights, affine4, head_weights, normal_bf16, verify_logits,
                                               zipf_bias)

DEV = "cuda"
EXPERTS, TOP_K = 512, 10
# The two layer shapes of the package: (hidden, moe intermediate, shared intermediate).
BASE = dict(hidden=2048, inter=512, shared=512)
REFERENCE = dict(hidden=2560, inter=640, shared=640)
VOCAB = 248320


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # The shared expert's gate projection for one token: the smallest launch of a decode step.
        dict(name="gemv_shared_r1", path="gemv", n=640, k=2560, rows=1, x="bf16"),
        # The lm_head over the four rows of a depth-3 verify round.
        dict(name="lm_head_r4", path="gemv", n=VOCAB, k=2560, rows=4, x="bf16"),
        # One token through ten experts: a decode step without drafts, fp32 activations as the reference passes them.
        dict(name="decode_r1", path="decode", rows=1, x="f32", **REFERENCE),
        # One layer of a depth-2 verify round at the reference model's shape, shared expert in affine 4-bit.
        dict(name="verify_t3_q4", path="verify", tokens=3, shared_q4=True, **REFERENCE),
        # A depth-1 verify round: 16 chained layers, the lm_head with the greedy round, the head's MoE, in one graph.
        dict(name="round_t2", path="round", layers=16, depth=1, vocab=VOCAB, **BASE),
        # Two chained draft tokens of the MTP head, as every speculative round drafts them.
        dict(name="draft_2", path="draft", depth=2, vocab=VOCAB, **BASE),
        # A few new tokens of a chat turn: most experts see one or two rows.
        dict(name="prefill_19", path="prefill", tokens=19, **BASE),
        # A short prompt of odd length at the reference model's hidden and expert sizes.
        dict(name="prefill_333", path="prefill", tokens=333, hidden=2560, inter=640, shared=512),
        # The default prompt chunk.
        dict(name="prefill_2048", path="prefill", tokens=2048, **BASE),
        # A long prompt in one chunk: every expert sees many rows.
        dict(name="prefill_8192", path="prefill", tokens=8192, **BASE),
        # The reference's verify width with its sampler at the default parameters.
        dict(name="accept_sampled_d2", path="accept", mode="sampled", depth=2, vocab=VOCAB, temperature=0.8,
             top_p=0.95, top_k=40),
        # Draft proposal and p/q acceptance of a depth-3 round.
        dict(name="accept_pq_d3", path="accept", mode="pq", depth=3, vocab=151936, temperature=0.7),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["gemv", "gemv", "decode", "verify", "prefill", "prefill", "prefill", "accept", "round", "draft"])
    if path == "gemv":
        return dict(path=path, n=_log_int(rng, 64, VOCAB), k=rng.choice([1024, 2048, 2560, 4096]),
                    rows=rng.choice([1, 2, 3, 4, rng.randint(5, 16)]), x=rng.choice(["bf16", "bf16", "f32"]))
    if path == "decode":
        return dict(path=path, rows=rng.choice([1, 2, 3, 4, rng.randint(5, 8)]), x=rng.choice(["bf16", "f32"]),
                    **rng.choice([BASE, REFERENCE]))
    if path == "verify":
        return dict(path=path, tokens=rng.randint(1, 4), shared_q4=rng.random() < 0.5, **rng.choice([BASE, REFERENCE]))
    if path == "round":
        return dict(path=path, layers=rng.randint(2, 16), depth=rng.randint(1, 3), vocab=_log_int(rng, 32000, VOCAB),
                    **BASE)
    if path == "draft":
        return dict(path=path, depth=rng.randint(1, 3), vocab=_log_int(rng, 32000, VOCAB), **BASE)
    if path == "prefill":
        return dict(path=path, tokens=_log_int(rng, 5, 6000), shared=512,
                    **rng.choice([dict(hidden=2048, inter=512), dict(hidden=2560, inter=640)]))
    case = dict(path=path, mode=rng.choice(["sampled", "sampled", "pq", "greedy"]), depth=rng.randint(1, 3),
                vocab=_log_int(rng, 32000, VOCAB), temperature=round(rng.uniform(0.5, 1.2), 2))
    if case["mode"] == "sampled":
        case.update(top_p=round(rng.uniform(0.8, 0.99), 2), top_k=rng.choice([20, 40, 100, rng.randint(1, 400)]))
    return case


# ---------------------------------------------------------------- inputs
class State:
    """What a program keeps between calls: inputs, weights, plans and buffers, as attributes."""

    def __init__(self, **kw):
        self.__dict__.update(kw)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _pool(case, seed, layers=1):
    pool = SlotPool(layers, EXPERTS, case["hidden"], case["inter"], device=DEV)
    pool.fill_random(seed)
    pool.place_permuted(seed + 1)
    return pool


def _rows(shape, seed, kind):
    x = normal_bf16(shape, 1.0, seed, DEV)
    return x if kind == "bf16" else x.float() + torch.randn(shape, generator=_gen(seed + 1), device=DEV) * 1e-3


def _decode_inputs(case, seed):
    r = case["rows"]
    score = torch.rand((r, EXPERTS), generator=_gen(seed), device=DEV)
    ids = score.topk(TOP_K, dim=1).indices.to(torch.int32)
    w = torch.softmax(torch.randn((r, TOP_K), generator=_gen(seed + 1), device=DEV), dim=-1)
    return _rows((r, case["hidden"]), seed + 2, case["x"]), ids.contiguous(), w.contiguous()


def _layer_inputs(case, seed, layers=1, q4=False):
    pool = _pool(case, seed, layers)
    lws = [LayerWeights(case["hidden"], EXPERTS, case["shared"], seed + 7 + l, DEV, shared_q4=q4) for l in range(layers)]
    biases = [zipf_bias(EXPERTS, 1.1, seed + 100 + l, DEV) for l in range(layers)]
    return pool, lws, biases


def prepare(case, seed):
    path, seed = case["path"], int(seed) * 1000 + 17
    if path == "gemv":
        return State(path=path, w=affine4(case["n"], case["k"], seed, device=DEV),
                     x=_rows((case["rows"], case["k"]), seed + 1, case["x"]))
    if path == "decode":
        r, h, i = case["rows"], case["hidden"], case["inter"]
        x, ids, w = _decode_inputs(case, seed + 2)
        return State(path=path, pool=_pool(case, seed), x=x, ids=ids, w=w,
                     h=torch.empty((r, TOP_K, i), device=DEV), o=torch.empty((r, TOP_K, h), device=DEV),
                     out=torch.empty((r, h), device=DEV))
    if path in ("verify", "prefill"):
        t = case["tokens"]
        pool, (lw,), (bias,) = _layer_inputs(case, seed, q4=case.get("shared_q4", False))
        args = (pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g)
        if path == "verify":
            layer = MoEVerifyLayer(*args, top_k=TOP_K, router_bias=bias)
            return State(path=path, layer=layer, x=normal_bf16((t, case["hidden"]), 1.0, seed + 3, DEV), lw=lw, bias=bias,
                         routed=torch.empty((t, case["hidden"]), device=DEV))
        layer = MoEPrefillLayer(*args, top_k=TOP_K, router_bias=bias, max_tokens=t)
        return State(path=path, layer=layer, x=normal_bf16((t, case["hidden"]), 1.0, seed + 3, DEV), lw=lw, bias=bias)
    if path == "round":
        nl, rows = case["layers"], case["depth"] + 1
        pool, lws, biases = _layer_inputs(case, seed, nl + 1)
        mw = [MoEWeights(w.router_w, w.sh_gate, w.sh_up, w.sh_down, w.sh_g, b) for w, b in zip(lws, biases)]
        lm = affine4(case["vocab"], case["hidden"], seed + 3, device=DEV)
        graph = MTPStepGraph(pool, mw[:nl], lm, case["depth"], head=mw[nl], top_k=TOP_K, keep_logits=True, device=DEV)
        graph.capture()
        return State(path=path, graph=graph, x=normal_bf16((rows, case["hidden"]), 1.0, seed + 4, DEV),
                     drafts=torch.randint(0, case["vocab"], (case["depth"],), generator=_gen(seed + 5), device=DEV,
                                          dtype=torch.int32))
    if path == "draft":
        hc = 4
        pool, (lw,), (bias,) = _layer_inputs(case, seed)
        moe = MoEVerifyLayer(pool, 0, lw.router_w, lw.sh_gate, lw.sh_up, lw.sh_down, lw.sh_g, top_k=TOP_K,
                             router_bias=bias)
        head = MTPHead(head_weights(case["hidden"], hc, 320, case["vocab"], seed % 100003, DEV), moe,
                       affine4(case["vocab"], case["hidden"], seed + 3, device=DEV), hc)
        graph = DraftGraph(head, case["depth"])
        graph.token.fill_(seed % case["vocab"])
        graph.multi.copy_(normal_bf16((1, hc * case["hidden"]), 1.0, seed + 4, DEV))
        graph.capture()
        return State(path=path, head=head, graph=graph, depth=case["depth"])
    d, v = case["depth"], case["vocab"]
    target, draft = verify_logits(d, v, seed, device=DEV)
    u = UniformStream(seed).peek(2 * d + 1)
    return State(path=path, case=case, acc=Acceptor(d, v, device=DEV), target=target, draft=draft,
                 drafts=target[:d].argmax(dim=1).to(torch.int32),
                 u_draft=torch.from_numpy(u[:d].copy()).to(DEV), u=torch.from_numpy(u[d:].copy()).to(DEV),
                 params=SampleParams(temperature=case["temperature"], top_p=case.get("top_p", 1.0),
                                     top_k=case.get("top_k", 0)))


def run(state):
    s = state
    if s.path == "gemv":
        return gemv(s.x, s.w)
    if s.path == "decode":
        out = moe_decode(s.x, s.ids, s.w, 0, s.pool.map, s.pool.slot_ptr, s.h, s.o, s.out, experts_per_layer=EXPERTS)
        return [out, s.o, s.h]
    if s.path == "verify":
        y, ids, w = s.layer(s.x, routed=s.routed)
        return [y, ids, w, s.routed]
    if s.path == "prefill":
        return list(s.layer(s.x))
    if s.path == "round":
        g = s.graph
        out = g.step(s.x, s.drafts)
        return [out, g.logits, g.streams[-1], g.ids, g.weights, g.head_y]
    if s.path == "draft":
        out = s.graph.replay()
        rows = s.head.draft_rows(s.depth)
        return [out, rows.out, rows.h, rows.ids]
    if s.case["mode"] == "greedy":
        return s.acc.greedy_async(s.target, s.drafts)
    if s.case["mode"] == "sampled":
        return s.acc.sampled_async(s.target, s.drafts, s.params, (), s.u)
    drafts = s.acc.draw_drafts_async(s.draft, s.u_draft, s.case["temperature"])
    return [drafts, s.acc.pq_async(s.target, s.draft, drafts, s.u, s.case["temperature"])]


# ---------------------------------------------------------------- what a pass cannot do without
def _unique_experts(tokens, hidden):
    """Expected number of distinct experts of `tokens` rows under the Zipf-biased router."""
    rng = np.random.default_rng(1)
    logits = rng.standard_normal((tokens, EXPERTS), dtype=np.float32) * (0.02 * math.sqrt(hidden))
    logits -= 1.1 * np.log(np.arange(1, EXPERTS + 1, dtype=np.float32))
    return len(np.unique(np.argpartition(-logits, TOP_K, axis=1)[:, :TOP_K]))


def _layer_work(case, t):
    h, i, s = case["hidden"], case["inter"], case["shared"]
    per = 0.5625 if case.get("shared_q4") else 2.0
    weights = _unique_experts(t, h) * record_layout(h, i)[1] + EXPERTS * h * 2 + 3 * h * s * per + h * 2
    return (weights + t * (h * 8 + TOP_K * 8), 2.0 * t * (TOP_K * 3 * h * i + 3 * h * s + h * EXPERTS))


def _affine_work(n, k, rows, xb=2, out=True):
    return n * (k / 2 + 4 * k / 64) + rows * k * xb + (rows * n * 4 if out else 0), 2.0 * n * k * rows


def work(case):
    path = case["path"]
    if path == "gemv":
        b, f = _affine_work(case["n"], case["k"], case["rows"], 2 if case["x"] == "bf16" else 4)
    elif path == "decode":
        r, h, i = case["rows"], case["hidden"], case["inter"]
        u = EXPERTS * (1 - (1 - TOP_K / EXPERTS) ** r)
        b = u * record_layout(h, i)[1] + r * (h * 8 + TOP_K * (4 * i + 4 * h + 8))
        f = 2.0 * r * TOP_K * 3 * h * i
    elif path in ("verify", "prefill"):
        b, f = _layer_work(case, case["tokens"])
    elif path == "round":
        t, n = case["depth"] + 1, case["layers"] + 1
        lb, lf = _layer_work(case, t)
        ab, af = _affine_work(case["vocab"], case["hidden"], t)
        b, f = n * lb + ab, n * lf + af
    elif path == "draft":
        h, n, d = case["hidden"], 4 * case["hidden"], case["depth"]
        lb, lf = _layer_work(case, 1)
        ab, af = _affine_work(case["vocab"], h, 1, out=False)
        dense = 2 * h * h + 4 * 320 * n + 4 * n
        b, f = d * (lb + ab + 2 * dense), d * (lf + af + 2.0 * (h * h + 4 * h * h + 4 * 320 * n + 4 * n))
    else:
        d, v = case["depth"], case["vocab"]
        rows = (2 * d + 1) if case["mode"] == "pq" else d + 1
        b, f = rows * v * 4.0, rows * v * 2.0
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    path = case["path"]
    if path == "gemv":
        # fp32 sums; an fp32 x enters the products as two bf16 parts
        return {"rel": 1e-5 if case["x"] == "bf16" else 4e-5}
    if path == "decode":
        # fp32 sums; h enters the down products as two bf16 parts
        return {"rel": 7e-5}
    if path == "verify":
        # bf16 y and shared-expert roundings; the ids are exact up to ties of bf16 logits
        return {"rel": 1e-2}
    if path == "prefill":
        # bf16 weights, h and y; a tie of bf16 router logits may pick another expert for a row
        return {"rel": 2e-2, "max": 0.9, "differ": 2e-3}
    if path in ("round", "draft"):
        # bf16 streams through chained layers
        return {"rel": 2e-2, "differ": 0.01}
    return "exact"


# ---------------------------------------------------------------- the same in 64 bits
def _dequant(q, s, b):
    """Affine 4-bit rows -> fp64: q int32 [n, k / 8] (nibble i at bits 4 i), s and b bf16 [n, k / 64]."""
    shift = torch.arange(0, 32, 4, device=q.device, dtype=torch.int32)
    nib = ((q.unsqueeze(-1) >> shift) & 15).reshape(q.shape[0], -1, 64).double()
    return (nib * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(q.shape[0], -1)


def _expert(pool, e):
    """(gate, up, down) of expert e in fp64."""
    h, i, off = pool.hidden, pool.inter, pool.offsets
    rec = pool.record(int(pool.map[e]))
    out = []
    for p, (n, k) in enumerate(((i, h), (i, h), (h, i))):
        o = off[3 * p: 3 * p + 3]
        q = rec[o[0]: o[0] + n * k // 2].view(torch.int32).reshape(n, k // 8)
        s, b = (rec[a: a + n * k // 32].view(torch.bfloat16).reshape(n, k // 64) for a in o[1:])
        out.append(_dequant(q, s, b))
    return out


def _routed(pool, x, ids, w):
    """h [T, K, I], o [T, K, H] (weighted expert outputs) and their sums over K, in fp64."""
    t, k = ids.shape
    h = torch.zeros((t, k, pool.inter), dtype=torch.float64, device=DEV)
    o = torch.zeros((t, k, pool.hidden), dtype=torch.float64, device=DEV)
    for e in torch.unique(ids).tolist():
        at = (ids == e).nonzero()
        gate, up, down = _expert(pool, e)
        xe = x[at[:, 0]]
        he = torch.nn.functional.silu(xe @ gate.T) * (xe @ up.T)
        h[at[:, 0], at[:, 1]] = he
        o[at[:, 0], at[:, 1]] = (he @ down.T) * w[at[:, 0], at[:, 1], None]
    return h, o, o.sum(dim=1)


def exact(case, seed):
    """The path in fp64 on the same inputs. Router logits are rounded to bf16 before the softmax, as the path defines
    them (they decide the routing); nothing else is rounded. A chain of layers (round, draft) has no such value: a
    rounding of one layer's bf16 output changes the routing of the layers behind it."""
    path = case["path"]
    if path not in ("gemv", "decode", "verify", "prefill"):
        return None
    s = prepare(case, seed)
    x = s.x.double()
    if path == "gemv":
        step = 16384
        return torch.cat([x @ _dequant(s.w.q[n: n + step], s.w.s[n: n + step], s.w.b[n: n + step]).T
                          for n in range(0, case["n"], step)], dim=1)
    if path == "decode":
        h, o, out = _routed(s.pool, x, s.ids.long(), s.w.double())
        return [out, o, h]
    pool, lw = s.layer.pool, s.lw
    logits = (x @ lw.router_w.double().T).to(torch.bfloat16).double() + s.bias.double()
    top, ids = torch.sort(torch.softmax(logits, dim=1), dim=1, descending=True, stable=True)
    top, ids = top[:, :TOP_K], ids[:, :TOP_K]
    w = top / top.sum(dim=1, keepdim=True)
    _, _, routed = _routed(pool, x, ids, w)
    sh = [_dequant(p.q, p.s, p.b) if case.get("shared_q4") else p.double() for p in (lw.sh_gate, lw.sh_up, lw.sh_down)]
    shared = (torch.nn.functional.silu(x @ sh[0].T) * (x @ sh[1].T)) @ sh[2].T
    y = routed + torch.sigmoid(x @ lw.sh_g.double().T) * shared
    return [y, None, w, routed]
