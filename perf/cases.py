"""The framework's work as measurable cases.

Each case is one pass through a public entry point on device or host data that
a user's program already holds: inference of the bundled networks
(`Model.eval_infer_device`, the per-network C-ABI driver), training steps
(`Model.train_step_device` with the updated weights fetched at the end) and a
kernel entry point (`nsh_op_attention_bwd`).  Networks and sizes are the
bundled plans' (neuralscript_amd/nets) at the benchmark's sizes, at small ones
and at ragged ones.

  kind       net           size                what it stands for
  infer      c1, c2        rows                dense MLP serving on device buffers
  infer_abi  c1, c2        rows                the same through ns_eval_infer on host arrays
  infer      c3, c3d       token ids           embedding, attention over the whole call, LayerNorm
  infer      c4            tokens              top-1 mixture of experts (64 experts, Zipf routing)
  train      c5            tokens              transformer training step (Muon on every matrix)
  train      moeb          tokens              mixture-of-experts training step
  attn_bwd   -             tokens, D, heads    the attention core's gradients
"""
from __future__ import annotations

import math

import numpy as np
import torch

from neuralscript_amd import runtime as rt

DEV = "cuda"


def listed():
    return [
        # one small dense call: launches and latency
        {"name": "mlp_small", "kind": "infer", "net": "c1", "n": 256},
        # a serving batch through the C ABI: host arrays in and out
        {"name": "mlp_host", "kind": "infer_abi", "net": "c2", "n": 512},
        # a handful of rows against 100 MB of weights
        {"name": "mlp_few_rows", "kind": "infer", "net": "c2", "n": 33},
        # the benchmark's dense batch
        {"name": "mlp_large", "kind": "infer", "net": "c2", "n": 8192},
        # a ragged sequence, heads of 128
        {"name": "attn_ragged", "kind": "infer", "net": "c3d", "n": 3001},
        # the benchmark's sequence: 16384 ids, 16 heads of 64
        {"name": "attn_large", "kind": "infer", "net": "c3", "n": 16384},
        # few tokens over 64 experts
        {"name": "moe_small", "kind": "infer", "net": "c4", "n": 1000},
        # the benchmark's MoE batch
        {"name": "moe_large", "kind": "infer", "net": "c4", "n": 65536},
        # training: a ragged short batch, and the benchmark's
        {"name": "train_ragged", "kind": "train", "net": "c5", "n": 1500, "steps": 4},
        {"name": "train_large", "kind": "train", "net": "c5", "n": 16384, "steps": 2},
        # training with experts
        {"name": "train_moe", "kind": "train", "net": "moeb", "n": 4096, "steps": 8},
        # the attention gradients alone, ragged
        {"name": "attn_bwd", "kind": "attn_bwd", "n": 5000, "D": 1024, "H": 16},
    ]


def _spread(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "abi", "attn", "attn", "moe", "moe", "train", "train", "train_moe", "attn_bwd"])
    if kind == "mlp":
        return {"kind": "infer", "net": rng.choice(["c1", "c2"]), "n": _spread(rng, 1, 8192)}
    if kind == "abi":
        return {"kind": "infer_abi", "net": rng.choice(["c1", "c2"]), "n": _spread(rng, 1, 4096)}
    if kind == "attn":
        return {"kind": "infer", "net": rng.choice(["c3", "c3d"]), "n": _spread(rng, 64, 16384)}
    if kind == "moe":
        return {"kind": "infer", "net": "c4", "n": _spread(rng, 64, 65536)}
    if kind == "train":
        return {"kind": "train", "net": "c5", "n": _spread(rng, 1024, 16384), "steps": 2}
    if kind == "train_moe":
        return {"kind": "train", "net": "moeb", "n": _spread(rng, 256, 16384), "steps": 8}
    D, H = rng.choice([(256, 8), (512, 8), (1024, 8), (1024, 16)])
    return {"kind": "attn_bwd", "n": _spread(rng, 128, 16384), "D": D, "H": H}


# ---- networks: weight shapes in blob order ------------------------------------

LR = 3e-4

SHAPES = {
    "c1": [(64, 256), (256, 256), (256, 10)],
    "c2": [(1024, 4096), (4096, 4096), (4096, 1024)],
    "c3": [(32000, 1024)] + [(1024, 1024)] * 4,
    "c3d": [(32000, 1024)] + [(1024, 1024)] * 4,
    "c4": [(1024, 64), (64, 1024 * 1024), (64, 1024 * 1024)],
    "c5": [(8192, 512)] + [(512, 512)] * 4 + [(512, 2048), (2048, 512), (512, 8192)],
    "moeb": [(512, 64), (64, 8), (8, 64 * 256), (8, 256 * 64), (64, 16)],
}
HEADS = {"c3": 16, "c3d": 8, "c5": 8}
IN_COLS = {"c1": 64, "c2": 1024, "c3": 1, "c3d": 1, "c4": 1024, "c5": 1, "moeb": 1}
OUT_COLS = {"c1": 10, "c2": 1024, "c3": 1024, "c3d": 1024, "c4": 1024, "c5": 8192, "moeb": 16}


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _normal(g, shape, std):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std


def _ids(g, n, vocab):
    """Token ids as floats, their frequency falling as 1 / rank."""
    u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
    return torch.clamp(torch.floor(torch.exp(u * math.log(vocab + 1.0))) - 1.0, 0, vocab - 1).float()


def _weights(net, g):
    """The weight matrices: Xavier-uniform for the MLPs; unit embeddings and
    variance 1 / fan-in for the transformers (scores of order 1, gradients of
    full rank where the network allows it: a Gram-Schmidt step on a matrix of
    rounding residue has no determined result); N(0, 0.02) experts under a
    router with Zipf(1.1) log-priors in the row that c4's constant last input
    column feeds; N(0, 0.2) for the small MoE network."""
    out = []
    for i, (r, c) in enumerate(SHAPES[net]):
        if net in ("c1", "c2"):
            a = math.sqrt(6.0 / (r + c))
            w = torch.rand((r, c), generator=g, device=DEV, dtype=torch.float32) * (2 * a) - a
        elif net == "c4" and i == 0:
            w = _normal(g, (r, c), math.sqrt(1.0 / r))
            p = torch.arange(1, c + 1, device=DEV, dtype=torch.float64) ** -1.1
            w[r - 1] = torch.log(p / p.sum()).float()
        elif net in HEADS:
            w = _normal(g, (r, c), 1.0 if i == 0 else math.sqrt(1.0 / r))
        else:
            w = _normal(g, (r, c), 0.2 if net == "moeb" else 0.02)
        out.append(w)
    return out


def _inputs(net, n, g):
    if net == "c1":
        return torch.rand((n, 64), generator=g, device=DEV, dtype=torch.float32) * 2 - 1
    if net == "c2":
        return _normal(g, (n, 1024), 1.0)
    if net == "c4":
        x = _normal(g, (n, 1024), 1.0)
        x[:, -1] = 1.0
        return x
    return _ids(g, n, SHAPES[net][0][0])


def _problem(case, seed):
    """Weights, inputs and (training) class ids of a network case."""
    g = _gen(seed)
    net, n = case["net"], case["n"]
    w = _weights(net, g)
    x = _inputs(net, n, g)
    y = _ids(g, n, OUT_COLS[net]).long() if case["kind"] == "train" else None
    return w, x, y


class _Buf:
    """A torch tensor as the device buffer the Model methods take."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()
        self.n = t.numel()


class _State:
    pass


class _Driver(_State):
    """A model of the per-network C-ABI driver, freed with the state."""

    def __init__(self, net, blob):
        self.lib = rt.net_lib(net)
        self.m = self.lib.init(blob)

    def __del__(self):
        if self.m:
            self.lib.free(self.m)
            self.m = None


def _qkv(case, seed):
    """Q, K, V and dO of an attention layer: projections of unit-variance rows."""
    g = _gen(seed)
    S, D, H = case["n"], case["D"], case["H"]
    return [_normal(g, (S, D), 1.0) for _ in range(4)]


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "attn_bwd":
        S, D, H = n, case["D"], case["H"]
        st = _State()
        st.S, st.D, st.H = S, D, H
        st.q, st.k, st.v, st.do = _qkv(case, seed)
        st.o = torch.empty_like(st.q)
        st.lse = torch.empty((H, S), device=DEV, dtype=torch.float32)
        torch.cuda.synchronize()  # the entry points run on streams of their own
        rt.op("attention_fwd", *(t.data_ptr() for t in (st.q, st.k, st.v, st.o, st.lse)), S, D, H)
        st.grads = [torch.empty_like(st.q) for _ in range(3)]
        nb = rt.lib().nsh_op_attention_bwd_workspace(S, D, H, 1)
        st.ws = torch.empty(max(1, nb), device=DEV, dtype=torch.uint8)
        torch.cuda.synchronize()
        return st
    w, x, y = _problem(case, seed)
    blob = torch.cat([t.reshape(-1) for t in w]).cpu().numpy()
    if kind == "infer_abi":
        st = _Driver(case["net"], blob)
        st.x = x.cpu().numpy()
        return st
    st = _State()
    st.model = rt.Model(rt.Plan.load(case["net"]), blob)
    st.x = _Buf(x.reshape(-1))
    if kind == "infer":
        st.out = _Buf(torch.empty((n, OUT_COLS[case["net"]]), device=DEV, dtype=torch.float32))
    else:
        st.steps = case["steps"]
        st.layout = st.model.plan.layout()
        st.y = _Buf(torch.nn.functional.one_hot(y, OUT_COLS[case["net"]]).float())
    torch.cuda.synchronize()  # the model runs on a stream of its own
    return st


def run(st):
    if isinstance(st, _Driver):
        return st.lib.eval_infer(st.m, st.x)
    if hasattr(st, "grads"):
        ptrs = [t.data_ptr() for t in (st.q, st.k, st.v, st.o, st.do, st.lse, *st.grads)]
        rt.op("attention_bwd", *ptrs, st.S, st.D, st.H, 1, st.ws.data_ptr())
        return st.grads
    if hasattr(st, "steps"):
        losses = [float(st.model.train_step_device(st.x, st.y, LR)) for _ in range(st.steps)]
        w = st.model.get_weights()
        return losses, [w[off:off + count] for _, off, count in st.layout]
    st.model.eval_infer_device(st.x, st.out)
    return st.out.t


# ---- work ---------------------------------------------------------------------

def _dense_flops(net, n):
    """Multiply-adds (x2) of the forward's dense products."""
    if net in ("c1", "c2"):
        return 2.0 * n * sum(r * c for r, c in SHAPES[net])
    if net in ("c3", "c3d"):
        return 2.0 * n * 4 * 1024 * 1024
    if net == "c4":
        return 2.0 * n * (1024 * 64 + 2 * 1024 * 1024)
    if net == "c5":
        return 2.0 * n * sum(r * c for r, c in SHAPES[net][1:])
    return 2.0 * n * (64 * 8 + 2 * 64 * 256 + 64 * 16)


def _weight_bytes(net, n):
    """Weights a pass must read: embedding rows only where ids hit them, at
    most one expert a token."""
    sh = SHAPES[net]
    b = 0
    for i, (r, c) in enumerate(sh):
        rows = r
        if net in ("c3", "c3d", "c5", "moeb") and i == 0:
            rows = min(r, n)
        if net == "c4" and i > 0:
            rows = min(r, n)
        b += rows * c * 4
    return b


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "attn_bwd":
        D, H = case["D"], case["H"]
        # S = QK^T again, dP = dO V^T, dV, dK, dQ; q, k, v, o, do in, three gradients out
        return {"bytes": 4.0 * (8 * n * D + H * n), "flops": 10.0 * n * n * D}
    net = case["net"]
    flops = _dense_flops(net, n)
    if kind in ("infer", "infer_abi"):
        if net in HEADS:
            flops += 4.0 * n * n * 1024
        return {"bytes": _weight_bytes(net, n) + 4.0 * n * (IN_COLS[net] + OUT_COLS[net]), "flops": flops}
    # a step: forward, both gradients of every product, Gram-Schmidt of each matrix
    # (2 R C^2); every weight read and written, ids and labels read
    flops *= 3
    if net == "c5":
        flops += 14.0 * n * n * 512
    total = 0
    for r, c in SHAPES[net]:
        total += r * c
        flops += 2.0 * max(r, c) * min(r, c) ** 2
    bytes_ = 8.0 * total + 4.0 * n * (1 + OUT_COLS[net])
    return {"bytes": bytes_ * case["steps"], "flops": flops * case["steps"]}


# ---- exactness ----------------------------------------------------------------

def tolerance(case):
    """About four times the largest distance measured over the range: of the
    forward passes and the gradients from 64 bits; of a training run from the
    same run on weights moved by at most half an ulp, i.e. what rounding of
    another order does to the Gram-Schmidt columns that are nearly dependent
    (3.6e-3 of a c5 projection, whose update in those steps is 2.6e-2; 7e-4
    of moeb's)."""
    kind = case["kind"]
    if kind == "train":
        return {"rel": 1.5e-2, "max": 0.3} if case["net"] == "c5" else {"rel": 3e-3, "max": 0.04}
    if kind == "attn_bwd":
        return {"rel": 1e-5, "max": 1e-4}
    if case["net"] in HEADS:
        return {"rel": 5e-5, "max": 3e-4}
    return {"rel": 8e-6, "max": 5e-5}


F64 = torch.float64
C_SQRT2 = float(np.float32(1.41421356))      # the constants the networks' formulas are written with
C_RSQRT2 = float(np.float32(0.7071067811865476))
EPS = float(np.float32(1e-5))


def _softmax_rows(s):
    s -= s.amax(1, keepdim=True)
    s.exp_()
    s /= s.sum(1, keepdim=True)
    return s


def _blocks(S):
    step = max(1, min(S, (1 << 28) // max(S, 1)))  # score blocks of at most 2 GiB
    return [(i, min(S, i + step)) for i in range(0, S, step)]


def _attn(q, k, v, H):
    S, D = q.shape
    dk = D // H
    scale = float(np.float32(1.0) / np.sqrt(np.float32(dk)))
    out = torch.empty_like(q)
    for h in range(H):
        c = slice(h * dk, (h + 1) * dk)
        kt, vh = k[:, c].t().contiguous(), v[:, c].contiguous()
        for a, b in _blocks(S):
            out[a:b, c] = _softmax_rows(q[a:b, c].contiguous() @ kt * scale) @ vh
    return out


def _attn_grads(q, k, v, do, H):
    S, D = q.shape
    dk = D // H
    scale = float(np.float32(1.0) / np.sqrt(np.float32(dk)))
    dq, dkk, dv = (torch.zeros_like(q) for _ in range(3))
    for h in range(H):
        c = slice(h * dk, (h + 1) * dk)
        kh, vt = k[:, c].contiguous(), v[:, c].t().contiguous()
        kt = kh.t().contiguous()
        for a, b in _blocks(S):
            qb, gb = q[a:b, c].contiguous(), do[a:b, c].contiguous()
            p = _softmax_rows(qb @ kt * scale)
            dv[:, c] += p.t().contiguous() @ gb
            ds = gb @ vt
            ds -= (p * ds).sum(1, keepdim=True)
            ds *= p
            dq[a:b, c] = ds @ kh * scale
            dkk[:, c] += ds.t().contiguous() @ qb * scale
    return dq, dkk, dv


def _layernorm(x):
    xc = x - x.mean(1, keepdim=True)
    return xc / torch.sqrt((xc * xc).mean(1, keepdim=True) + EPS)


def _gelu(x):
    return 0.5 * x * (1.0 + torch.erf(x / C_SQRT2))


def _route(x, wg):
    lg = x @ wg
    best = lg.argmax(1)
    return torch.softmax(lg, 1), best


def _moe(x, wg, w1, w2):
    D = x.shape[1]
    p, best = _route(x, wg)
    out = torch.zeros_like(x)
    for e in range(wg.shape[1]):
        t = (best == e).nonzero().flatten()
        if len(t):
            u = x[t] @ w1[e].view(D, -1).to(F64)
            g = 0.5 * u * (1.0 + torch.erf(u * C_RSQRT2))
            out[t] = p[t, e][:, None] * (g @ w2[e].view(-1, D).to(F64))
    return out


def _first_loss(net, w, x, y):
    w = [t.to(F64) for t in w]
    h = w[0][x.long()]
    if net == "moeb":
        logits = _moe(h, *w[1:4]) @ w[4]
    else:
        at = _attn(h @ w[1], h @ w[2], h @ w[3], HEADS[net]) @ w[4]
        logits = torch.relu(_layernorm(at) @ w[5]) @ w[6] @ w[7]
    return float(torch.nn.functional.cross_entropy(logits, y))


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn_bwd":
        q, k, v, do = (t.to(F64) for t in _qkv(case, seed))
        return list(_attn_grads(q, k, v, do, case["H"]))
    w, x, y = _problem(case, seed)
    net = case["net"]
    if kind == "train":
        # the first loss only: from the first update on, the columns that are
        # nearly dependent make Gram-Schmidt amplify rounding (see tolerance),
        # so the weights and later losses have no value to 32 bits
        return [_first_loss(net, w, x, y)] + [None] * (case["steps"] - 1), [None] * len(SHAPES[net])
    if net == "c4":
        return _moe(x.to(F64), w[0].to(F64), w[1], w[2])
    w = [t.to(F64) for t in w]
    if net in HEADS:
        h = w[0][x.long()]
        return _layernorm(_attn(h @ w[1], h @ w[2], h @ w[3], HEADS[net]) @ w[4])
    h = x.to(F64)
    act = torch.relu if net == "c1" else _gelu
    h = act(act(h @ w[0]) @ w[1]) @ w[2]
    return h.reshape(-1) if kind == "infer_abi" else h
