"""The calls whose time counts: what a Gemma-4-sized MoE model (d 2816, 128
experts of 704, shared expert 2112, vocabulary 262144) has this package do
while it reads a prompt and while it generates tokens, one call each through
the operator classes of edgeexpert_amd.ops.

Decode, one token per call:
  gemv       one quantised projection, or the logits over the vocabulary
  qkv        the fused q/k/v projection
  attention  GQA attention over an fp16 KV cache
  moe_token  router, top-k and the routed experts of one token
  layers     whole decoder layers, the KV cache updated
Prefill, a block of prompt tokens per call:
  gemm          one quantised projection
  shared_block  the shared expert
  moe_block     router, grouping, routed experts and combine

Inputs follow the distributions of edgeexpert_amd.synth, drawn on the GPU.
"""
from __future__ import annotations

import math

import torch

from edgeexpert_amd import ops
from edgeexpert_amd._lib import DTYPE_BF16, DTYPE_F16, ROUTER_WORKSPACE_BYTES

D, F, E, TOP_K, SHARED_F, VOCAB = 2816, 704, 128, 8, 2112, 262144
GROUP = 64
EPS = 1e-6
# (outputs, inputs) of the model's projections: sliding q, k/v and o, full q
# and o, shared expert gate/up and down, routed gate/up and down
PROJECTIONS = ((4096, 2816), (2048, 2816), (2816, 4096), (8192, 2816), (2816, 8192), (2112, 2816), (2816, 2112),
               (704, 2816), (2816, 704))
# (head_dim, query heads, kv heads): sliding layers, full-attention layers,
# and a grouped head_dim 128 model
HEADS = ((256, 16, 8), (512, 16, 2), (128, 8, 2))
# tokens of one prompt share a direction, so experts are unevenly popular:
# this much of it beside N(0, 1) gives a popularity close to Zipf(1.1)
COMMON = 0.8


def listed():
    return [
        # one projection of one token: the smallest call, launch and latency
        {"name": "gemv_2816x2816_q4", "kind": "gemv", "m": 2816, "k": 2816, "bits": 4},
        # q, k and v of a token, with the 3-bit attention weights option
        {"name": "qkv_8192x2816_q3", "kind": "qkv", "mq": 4096, "mkv": 2048, "k": 2816, "bits": 3},
        # the logits of one token: the largest weight stream
        {"name": "logits_262144x2816_q4", "kind": "gemv", "m": VOCAB, "k": 2816, "bits": 4},
        # a sliding layer's attention at 4096 keys
        {"name": "attention_h256_4096", "kind": "attention", "hd": 256, "nq": 16, "nkv": 8, "seq": 4096, "window": 0},
        # a full-attention layer's attention over a long conversation
        {"name": "attention_h512_32768", "kind": "attention", "hd": 512, "nq": 16, "nkv": 2, "seq": 32768,
         "window": 0},
        # the routed experts of one token, at the default width
        {"name": "moe_token_q4", "kind": "moe_token", "d": D, "f": F, "experts": E, "top_k": TOP_K, "bits": 4},
        # a sliding and a full-attention layer of one token at 4096 keys, the
        # shared expert at its default 8 bits
        {"name": "layers_sliding_full_4096", "kind": "layers", "pattern": "sf", "position": 4095, "window": 0,
         "shared_bits": 8},
        # a projection of a 512-token prompt block
        {"name": "gemm_512x8192x2816_bf16_q4", "kind": "gemm", "t": 512, "n": 8192, "k": 2816, "bits": 4,
         "dtype": "bf16"},
        # a short prompt (or several conversations' tokens) through the output projection
        {"name": "gemm_45x2816x4096_f16_q4", "kind": "gemm", "t": 45, "n": 2816, "k": 4096, "bits": 4, "dtype": "f16"},
        # the shared expert of a 512-token prompt block at its default 8 bits
        {"name": "shared_block_512_q8", "kind": "shared_block", "t": 512, "d": D, "f": SHARED_F, "bits": 8},
        # the routed experts of a 512-token prompt block
        {"name": "moe_block_512_q4", "kind": "moe_block", "t": 512, "d": D, "f": F, "experts": E, "top_k": TOP_K,
         "bits": 4},
        # the routed experts of a short prompt, with the 3-bit experts option
        {"name": "moe_block_33_q3", "kind": "moe_block", "t": 33, "d": D, "f": F, "experts": E, "top_k": TOP_K,
         "bits": 3},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], even over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step) * step))


def _projection(rng, k_max):
    """One of the model's projections, or (one time in three) any size."""
    if rng.random() < 2 / 3:
        return rng.choice([p for p in PROJECTIONS if p[1] <= k_max])
    return _log(rng, 64, 8192), _log(rng, 512, k_max, GROUP)


def draw(rng):
    kind = rng.choice(("gemv", "qkv", "logits", "attention", "moe_token", "layers", "gemm", "shared_block",
                       "moe_block"))
    if kind == "gemv":
        bits = rng.choice((4, 4, 3, 8))
        m, k = _projection(rng, 4096 if bits == 8 else 8192)
        return {"kind": "gemv", "m": m, "k": k, "bits": bits}
    if kind == "qkv":
        return {"kind": "qkv", "mq": _log(rng, 512, 8192, 64), "mkv": _log(rng, 128, 2048, 64),
                "k": rng.choice((D, _log(rng, 512, 4096, GROUP))), "bits": rng.choice((4, 4, 3))}
    if kind == "logits":
        return {"kind": "gemv", "m": _log(rng, 32000, VOCAB), "k": rng.choice((2816, 2816, 2048, 2560)),
                "bits": rng.choice((4, 4, 3))}
    if kind == "attention":
        hd, nq, nkv = rng.choice(HEADS)
        return {"kind": "attention", "hd": hd, "nq": nq, "nkv": nkv, "seq": _log(rng, 32, 32768),
                "window": rng.choice((0, 0, 1024)) if hd != 512 else 0}
    if kind == "moe_token":
        return {"kind": "moe_token", "d": rng.choice((D, D, _log(rng, 512, 4096, GROUP))),
                "f": rng.choice((F, F, _log(rng, 256, 1024, GROUP))), "experts": rng.choice((E, E, 64, 40)),
                "top_k": rng.choice((TOP_K, TOP_K, 6)), "bits": rng.choice((4, 4, 3, 2))}
    if kind == "layers":
        return {"kind": "layers", "pattern": rng.choice(("s", "f", "sf")), "position": _log(rng, 32, 8192),
                "window": rng.choice((0, 1024)), "shared_bits": rng.choice((8, 8, 4))}
    if kind == "gemm":
        n, k = _projection(rng, 8192)
        return {"kind": "gemm", "t": _log(rng, 2, 1024), "n": n, "k": k, "bits": rng.choice((4, 4, 4, 3)),
                "dtype": rng.choice(("bf16", "f16"))}
    if kind == "shared_block":
        return {"kind": "shared_block", "t": _log(rng, 2, 512), "d": D, "f": rng.choice((SHARED_F, 1024, 2048)),
                "bits": rng.choice((8, 8, 4))}
    return {"kind": "moe_block", "t": _log(rng, 2, 512), "d": D, "f": rng.choice((F, F, 512)),
            "experts": rng.choice((E, E, 64)), "top_k": TOP_K, "bits": rng.choice((4, 4, 3, 2))}


# ------------------------------------------------------------ inputs ----

def _randn(gen, *shape):
    return torch.randn(shape, device="cuda", generator=gen)


def _bytes(gen, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=gen)


def _norm(gen, n):
    return (0.5 + torch.rand(n, device="cuda", generator=gen)).half()


def _affine(gen, bits, *shape):
    """fp16 scales and biases of `shape` groups of `bits`-bit codes."""
    s = (_randn(gen, *shape).abs() * (0.02 * 16 / 2 ** bits)).half()
    b = (-(2 ** (bits - 1)) * s.float() + 0.002 * _randn(gen, *shape)).half()
    return s, b


def _matrix(gen, rows, k, bits):
    return (_bytes(gen, rows, k * bits // 8), *_affine(gen, bits, rows, k // GROUP))


def _matrix_bytes(rows, k, bits):
    return rows * (k * bits // 8 + 4 * (k // GROUP))


def _pool(gen, experts, d, f, bits):
    """All experts' blobs [gate w s b, up w s b, down w s b] at a 16 KiB
    stride, and the offsets of the parts."""
    off, at = {}, 0
    for name, rows, k in (("gate", f, d), ("up", f, d), ("down", d, f)):
        for part, size in (("w", rows * k * bits // 8), ("s", rows * k // GROUP * 2), ("b", rows * k // GROUP * 2)):
            off["%s_%s" % (name, part)] = at
            at += size
    stride = (at + 16383) // 16384 * 16384
    pool = _bytes(gen, experts, stride)
    for name in ("gate", "up", "down"):
        s, b = _affine(gen, bits, experts, f * d // GROUP)
        for part, v in (("s", s), ("b", b)):
            at = off["%s_%s" % (name, part)]
            pool[:, at:at + 2 * v.shape[1]] = v.view(torch.uint8)
    return pool, off, stride


# ------------------------------------------------- the same in 64 bits ----

def _codes(w, bits):
    """Codes of packed rows [rows][bytes], as int32 [rows][codes]."""
    if bits == 8:
        return w.int()
    if bits == 3:
        v = w.view(w.shape[0], -1, 3).int()
        v, per = v[..., 0] | v[..., 1] << 8 | v[..., 2] << 16, 8
    else:
        v, per = w.int(), 8 // bits
    shifts = torch.arange(per, device=w.device, dtype=torch.int32) * bits
    return ((v[..., None] >> shifts) & (2 ** bits - 1)).view(w.shape[0], -1)


def _dense(matrix, bits):
    w, s, b = matrix
    q = _codes(w, bits).double().view(w.shape[0], -1, GROUP)
    return (q * s.double()[..., None] + b.double()[..., None]).view(w.shape[0], -1)


def _times(matrix, bits, x):
    """x · Wᵀ over blocks of rows (the vocabulary's do not fit at once)."""
    step = 16384
    return torch.cat([x @ _dense([p[r:r + step] for p in matrix], bits).T for r in range(0, matrix[0].shape[0], step)],
                     dim=-1)


def _gated(gate, up, x, bits):
    return torch.nn.functional.gelu(_times(gate, bits, x), approximate="tanh") * _times(up, bits, x)


def _rms(x, w=None):
    y = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt()
    return y if w is None else y * w.double()


def _blob(pool, off, expert, name, rows, k, bits):
    def part(p, n):
        return pool[expert, off["%s_%s" % (name, p)]:][:n].contiguous()
    g = rows * k // GROUP
    return (part("w", rows * k * bits // 8).view(rows, -1), part("s", 2 * g).view(torch.float16).view(rows, -1),
            part("b", 2 * g).view(torch.float16).view(rows, -1))


def _route(router, x, top_k):
    """(indices, weights) [tokens][top_k] of the int8 router."""
    w, eff, gain = router
    logits = _times(w, 8, x * eff.double())
    top, idx = logits.sort(dim=-1, descending=True, stable=True)
    idx = idx[:, :top_k]
    return idx, torch.softmax(top[:, :top_k], dim=-1) * gain.double()[idx]


def _experts(pool, off, x, idx, weights, d, f, bits):
    y = torch.zeros_like(x)
    for e in idx.unique().tolist():
        t, r = (idx == e).nonzero(as_tuple=True)
        a = _gated(_blob(pool, off, e, "gate", f, d, bits), _blob(pool, off, e, "up", f, d, bits), x[t], bits)
        y[t] += weights[t, r, None] * _times(_blob(pool, off, e, "down", d, f, bits), bits, a)
    return y


def _attend(q, k, v, scale):
    """q [heads][hd], k and v [keys][kv heads][hd]."""
    group = q.shape[0] // k.shape[1]
    q = q.view(k.shape[1], group, -1)
    s = torch.stack([q[h] @ k[:, h].T for h in range(k.shape[1])]) * scale
    p = torch.softmax(s, dim=-1)
    return torch.stack([p[h] @ v[:, h].contiguous() for h in range(k.shape[1])]).view(-1)


def _rope(x, pairs, position, theta):
    hd = x.shape[-1]
    i = torch.arange(pairs, device=x.device, dtype=torch.float64)
    a = position * theta ** (-2 * i / hd)
    lo, hi = x[..., :pairs], x[..., hd // 2:hd // 2 + pairs]
    y = x.clone()
    y[..., :pairs] = lo * a.cos() - hi * a.sin()
    y[..., hd // 2:hd // 2 + pairs] = lo * a.sin() + hi * a.cos()
    return y


# --------------------------------------------------------------- calls ----

_shared_context = None


def _context():
    """The process's one context (loaded kernels)."""
    global _shared_context
    if _shared_context is None:
        _shared_context = ops.Context()
    return _shared_context


def _p(t):
    return None if t is None else t.data_ptr()


def _proj(matrix, rows, k):
    return ops.Q4Projection(*(_p(t) for t in matrix), rows, k) if matrix else ops.Q4Projection(None, None, None, 0, 0)


def _empty(*shape, dtype=torch.float16):
    return torch.zeros(shape, dtype=dtype, device="cuda")


class _Call:
    """One case: `inputs` draws what a program has in hand, `bind` makes its
    handles and result buffers, `run` is the call."""

    def __init__(self, case, seed):
        self.c = case
        self.inputs(torch.Generator("cuda").manual_seed(seed), **{k: v for k, v in case.items()
                                                                  if k not in ("name", "kind")})

    def ready(self):
        self.bind(**{k: v for k, v in self.c.items() if k not in ("name", "kind")})
        return self


class _Gemv(_Call):
    def inputs(self, gen, m, k, bits):
        self.w, self.x = _matrix(gen, m, k, bits), _randn(gen, k).half()

    def bind(self, m, k, bits):
        self.y = _empty(m)
        args = [_p(t) for t in (*self.w, self.x, self.y)] + [m, k]
        if bits == 8:
            op = ops.DequantInt8GEMV(_context())
            self.call = lambda: op.encode(None, *args)
        else:
            op = ops.DequantInt4GEMV(_context())
            self.call = lambda: op.encode(None, *args, bits=bits)

    def run(self):
        self.call()
        return self.y

    def exact(self):
        return _times(self.w, self.c["bits"], self.x.double())

    @staticmethod
    def work(m, k, bits):
        return _matrix_bytes(m, k, bits) + 2 * (m + k), 2 * m * k


class _Qkv(_Call):
    def inputs(self, gen, mq, mkv, k, bits):
        self.w = [_matrix(gen, m, k, bits) for m in (mq, mkv, mkv)]
        self.x = _randn(gen, k).half()

    def bind(self, mq, mkv, k, bits):
        self.y = [_empty(m) for m in (mq, mkv, mkv)]
        q, kk, v = (_proj(w, m, k) for w, m in zip(self.w, (mq, mkv, mkv)))
        op, x, y = ops.DequantInt4GEMV(_context()), _p(self.x), [_p(t) for t in self.y]
        self.call = lambda: op.encode_qkv(None, q, kk, v, x, *y, mq, mkv, k, bits=bits)

    def run(self):
        self.call()
        return self.y

    def exact(self):
        return [_times(w, self.c["bits"], self.x.double()) for w in self.w]

    @staticmethod
    def work(mq, mkv, k, bits):
        m = mq + 2 * mkv
        return _matrix_bytes(m, k, bits) + 2 * (m + k), 2 * m * k


class _Attention(_Call):
    def inputs(self, gen, hd, nq, nkv, seq, window):
        self.q = _randn(gen, nq, hd).half()
        self.k, self.v = _randn(gen, seq, nkv, hd).half(), _randn(gen, seq, nkv, hd).half()

    def bind(self, hd, nq, nkv, seq, window):
        self.y = _empty(nq * hd)
        size = ops.Attention.workspace_bytes(hd, nq, seq, window)
        self.ws = _empty(size, dtype=torch.uint8)
        op, q, k, v, y, ws = (ops.Attention(_context()), *(_p(t) for t in (self.q, self.k, self.v, self.y, self.ws)))
        self.call = lambda: op.encode(None, q, k, v, y, hd, nq, nkv, seq, ws, size, window=window)

    def run(self):
        self.call()
        return self.y

    def exact(self):
        first = max(0, self.c["seq"] - self.c["window"]) if self.c["window"] else 0
        return _attend(self.q.double(), self.k[first:].double(), self.v[first:].double(), self.c["hd"] ** -0.5)

    @staticmethod
    def work(hd, nq, nkv, seq, window):
        keys = min(seq, window) if window else seq
        return 4 * keys * nkv * hd + 4 * nq * hd, 4 * keys * nq * hd


def _router(gen, experts, d):
    return _matrix(gen, experts, d, 8), _norm(gen, d), _norm(gen, experts)


def _router_desc(router, experts):
    w, eff, gain = router
    return ops.Router(*(_p(t) for t in w), experts, _p(eff), _p(gain))


class _MoeToken(_Call):
    def inputs(self, gen, d, f, experts, top_k, bits):
        self.pool, self.off, self.stride = _pool(gen, experts, d, f, bits)
        self.router = _router(gen, experts, d)
        self.x = _randn(gen, d).half()

    def bind(self, d, f, experts, top_k, bits):
        self.y, self.acts, self.weights = _empty(d), _empty(top_k, f), _empty(top_k)
        self.idx, self.ws = _empty(top_k, dtype=torch.int32), _empty(ROUTER_WORKSPACE_BYTES, dtype=torch.uint8)
        router = _router_desc(self.router, experts)
        pool = ops.ExpertPool(_p(self.pool), self.stride, experts, self.off, weight_bits=bits)
        x, y, idx, w, acts, ws = (_p(t) for t in (self.x, self.y, self.idx, self.weights, self.acts, self.ws))
        self.call = lambda: ops.moe_decode_token(_context(), None, router, pool, x, None, y, d, f, top_k, idx, w, acts,
                                                 ws)

    def run(self):
        self.call()
        return {"y": self.y, "experts": self.idx, "weights": self.weights}

    def exact(self):
        c, x = self.c, self.x.double()[None]
        idx, w = _route(self.router, x, c["top_k"])
        return {"y": _experts(self.pool, self.off, x, idx, w, c["d"], c["f"], c["bits"])[0], "experts": None,
                "weights": w[0]}

    @staticmethod
    def work(d, f, experts, top_k, bits):
        one = 2 * _matrix_bytes(f, d, bits) + _matrix_bytes(d, f, bits)
        return (_matrix_bytes(experts, d, 8) + 2 * (d + experts) + top_k * one + 4 * d + 6 * top_k,
                2 * experts * d + 6 * top_k * d * f)


class _Layers(_Call):
    """Layers "s" (sliding: head_dim 256, 8 kv heads) and "f" (full attention:
    head_dim 512, 2 kv heads, V from the k projection, partial rotary)."""
    SHAPES = {"s": (256, 16, 8, 128, 10000.0), "f": (512, 16, 2, 64, 1e6)}

    def inputs(self, gen, pattern, position, window, shared_bits):
        self.layers = []
        for kind in pattern:
            hd, nq, nkv, _, _ = self.SHAPES[kind]
            w = {n: _norm(gen, D) for n in ("input_norm", "post_attention_norm", "pre_ffn_norm", "pre_ffn2_norm",
                                            "post_ffn1_norm", "post_ffn2_norm", "post_ffn_norm")}
            w.update(q_norm=_norm(gen, hd), k_norm=_norm(gen, hd), q=_matrix(gen, nq * hd, D, 4),
                     k=_matrix(gen, nkv * hd, D, 4), v=_matrix(gen, nkv * hd, D, 4) if kind == "s" else None,
                     o=_matrix(gen, D, nq * hd, 4), router=_router(gen, E, D), pool=_pool(gen, E, D, F, 4),
                     gate=_matrix(gen, SHARED_F, D, shared_bits), up=_matrix(gen, SHARED_F, D, shared_bits),
                     down=_matrix(gen, D, SHARED_F, shared_bits),
                     kc=_randn(gen, position + 1, nkv, hd).half(), vc=_randn(gen, position + 1, nkv, hd).half())
            self.layers.append(w)
        self.hidden = _randn(gen, D).half()

    def bind(self, pattern, position, window, shared_bits):
        specs, shapes = [], []
        for kind, w in zip(pattern, self.layers):
            hd, nq, nkv, pairs, theta = self.SHAPES[kind]
            pool, off, stride = w["pool"]
            norms = {n: _p(w[n]) for n in w if n.endswith("norm")}
            specs.append(ops.DecodeLayerWeightsSpec(
                q_proj=_proj(w["q"], nq * hd, D), k_proj=_proj(w["k"], nkv * hd, D), v_proj=_proj(w["v"], nkv * hd, D),
                o_proj=_proj(w["o"], D, nq * hd), router=_router_desc(w["router"], E),
                experts=ops.ExpertPool(_p(pool), stride, E, off), shared_gate=_proj(w["gate"], SHARED_F, D),
                shared_up=_proj(w["up"], SHARED_F, D), shared_down=_proj(w["down"], D, SHARED_F),
                layer_scalar=0.75, shared_bits=shared_bits, **norms))
            shapes.append(ops.DecodeLayerShapeSpec(
                d=D, num_q_heads=nq, num_kv_heads=nkv, head_dim=hd, expert_f=F, shared_f=SHARED_F, top_k=TOP_K,
                rotated_pairs=pairs, window=window if kind == "s" else 0, rope_theta=theta))
        op = ops.DecodeLayers(_context(), specs, shapes)
        size = op.workspace_bytes(position + 1)
        self.ws, self.y = _empty(size, dtype=torch.uint8), _empty(len(pattern), D)
        x, y, ws = _p(self.hidden), _p(self.y), _p(self.ws)
        kc, vc = [_p(w["kc"]) for w in self.layers], [_p(w["vc"]) for w in self.layers]
        self.call = lambda: op.encode(None, x, y, kc, vc, position, ws, size)
        self.out = {"hidden": self.y, "k": [w["kc"][position] for w in self.layers],
                    "v": [w["vc"][position] for w in self.layers]}

    def run(self):
        self.call()
        return self.out

    def exact(self):
        c, x, out = self.c, self.hidden.double(), {"hidden": [], "k": [], "v": []}
        for kind, w in zip(c["pattern"], self.layers):
            hd, nq, nkv, pairs, theta = self.SHAPES[kind]
            xn = _rms(x, w["input_norm"])
            q, k = _times(w["q"], 4, xn).view(nq, hd), _times(w["k"], 4, xn).view(nkv, hd)
            v = _times(w["v"], 4, xn).view(nkv, hd) if w["v"] else k
            q, k = (_rope(_rms(t, w[n]), pairs, c["position"], theta) for t, n in ((q, "q_norm"), (k, "k_norm")))
            v = _rms(v)
            first = max(0, c["position"] + 1 - c["window"]) if c["window"] and kind == "s" else 0
            keys, vals = (torch.cat([w[n][first:c["position"]].double(), t[None]]) for n, t in (("kc", k), ("vc", v)))
            o = _times(w["o"], 4, _attend(q, keys, vals, 1.0))
            h = x + _rms(o, w["post_attention_norm"])
            idx, weights = _route(w["router"], _rms(h)[None], TOP_K)
            h1 = _times(w["down"], c["shared_bits"],
                        _gated(w["gate"], w["up"], _rms(h, w["pre_ffn_norm"]), c["shared_bits"]))
            pool, off, _ = w["pool"]
            h2 = _experts(pool, off, _rms(h, w["pre_ffn2_norm"])[None], idx, weights, D, F, 4)[0]
            x = (h + _rms(_rms(h1, w["post_ffn1_norm"]) + _rms(h2, w["post_ffn2_norm"]), w["post_ffn_norm"])) * 0.75
            for n, t in (("hidden", x), ("k", k), ("v", v)):
                out[n].append(t)
        out["hidden"] = torch.stack(out["hidden"])
        return out

    @classmethod
    def work(cls, pattern, position, window, shared_bits):
        size = flops = 4 * D
        for kind in pattern:
            hd, nq, nkv, _, _ = cls.SHAPES[kind]
            a = _Attention.work(hd, nq, nkv, position + 1, window if kind == "s" else 0)
            m = _MoeToken.work(D, F, E, TOP_K, 4)
            rows = (nq + (2 if kind == "s" else 1) * nkv) * hd
            size += a[0] + m[0] + _matrix_bytes(rows, D, 4) + _matrix_bytes(D, nq * hd, 4) + 14 * D \
                + 2 * _matrix_bytes(SHARED_F, D, shared_bits) + _matrix_bytes(D, SHARED_F, shared_bits)
            flops += a[1] + m[1] + 2 * D * (rows + nq * hd) + 6 * D * SHARED_F
        return size, flops


class _Gemm(_Call):
    def inputs(self, gen, t, n, k, bits, dtype):
        self.kind = torch.bfloat16 if dtype == "bf16" else torch.float16
        self.w, self.x = _matrix(gen, n, k, bits), _randn(gen, t, k).to(self.kind)

    def bind(self, t, n, k, bits, dtype):
        self.y = _empty(t, n, dtype=self.kind)
        op = ops.PrefillInt4QMM(_context())
        args = [_p(v) for v in (*self.w, self.x, self.y)] + [t, n, k, DTYPE_BF16 if dtype == "bf16" else DTYPE_F16]
        self.call = lambda: op.encode(None, *args, bits=bits)

    def run(self):
        self.call()
        return self.y

    def exact(self):
        return _times(self.w, self.c["bits"], self.x.double())

    @staticmethod
    def work(t, n, k, bits, dtype):
        return _matrix_bytes(n, k, bits) + 2 * t * (n + k), 2 * t * n * k


class _SharedBlock(_Call):
    def inputs(self, gen, t, d, f, bits):
        self.gate, self.up, self.down = (_matrix(gen, r, k, bits) for r, k in ((f, d), (f, d), (d, f)))
        self.x = _randn(gen, t, d).half()

    def bind(self, t, d, f, bits):
        self.y = _empty(t, d)
        size = ops.prefill_shared_expert_workspace_bytes(bits, t, f)
        self.ws = _empty(size, dtype=torch.uint8)
        op = ops.PrefillSharedExpert(_context(), weight_bits=bits)
        gate, up, down = _proj(self.gate, f, d), _proj(self.up, f, d), _proj(self.down, d, f)
        x, y, ws = _p(self.x), _p(self.y), _p(self.ws)
        self.call = lambda: op.encode_block(None, x, y, gate, up, down, ws, size, t, d, f, d, d)

    def run(self):
        self.call()
        return self.y

    def exact(self):
        bits = self.c["bits"]
        return _times(self.down, bits, _gated(self.gate, self.up, self.x.double(), bits))

    @staticmethod
    def work(t, d, f, bits):
        return 2 * _matrix_bytes(f, d, bits) + _matrix_bytes(d, f, bits) + 4 * t * d, 6 * t * d * f


def _active_experts(t, experts, top_k):
    """Expected experts that t tokens of one prompt use: expert with popularity
    u ~ N(0, COMMON) is taken by a token when u + N(0, 1) is over the cut that
    leaves top_k of them."""
    def taken(u, cut):
        return 0.5 * math.erfc((cut - u) / math.sqrt(2))
    us = [COMMON * math.sqrt(2) * _erfinv(2 * (e + 0.5) / experts - 1) for e in range(experts)]
    lo, hi = -10.0, 10.0
    for _ in range(60):
        cut = (lo + hi) / 2
        lo, hi = (cut, hi) if sum(taken(u, cut) for u in us) > top_k else (lo, cut)
    return sum(1 - (1 - taken(u, lo)) ** t for u in us)


def _erfinv(y):
    lo, hi = -6.0, 6.0
    for _ in range(60):
        mid = (lo + hi) / 2
        lo, hi = (mid, hi) if math.erf(mid) < y else (lo, mid)
    return (lo + hi) / 2


class _MoeBlock(_Call):
    def inputs(self, gen, t, d, f, experts, top_k, bits):
        self.pool, self.off, self.stride = _pool(gen, experts, d, f, bits)
        self.router = _router(gen, experts, d)
        self.x = (COMMON * _randn(gen, d) + _randn(gen, t, d)).half()

    def bind(self, t, d, f, experts, top_k, bits):
        self.y, self.weights = _empty(t, d), _empty(t, top_k)
        self.idx = _empty(t, top_k, dtype=torch.int32)
        size = ops.moe_prefill_workspace_bytes(t, top_k, experts, d, f)
        self.ws = _empty(size, dtype=torch.uint8)
        router = _router_desc(self.router, experts)
        pool = ops.ExpertPool(_p(self.pool), self.stride, experts, self.off, weight_bits=bits)
        x, y, idx, w, ws = (_p(v) for v in (self.x, self.y, self.idx, self.weights, self.ws))
        self.call = lambda: ops.moe_prefill(_context(), None, router, pool, x, d, t, d, f, top_k, y, idx, w, ws, size)

    def run(self):
        self.call()
        return {"y": self.y, "experts": self.idx, "weights": self.weights}

    def exact(self):
        c, x = self.c, self.x.double()
        idx, w = _route(self.router, x, c["top_k"])
        return {"y": _experts(self.pool, self.off, x, idx, w, c["d"], c["f"], c["bits"]), "experts": None,
                "weights": w}

    @staticmethod
    def work(t, d, f, experts, top_k, bits):
        one = 2 * _matrix_bytes(f, d, bits) + _matrix_bytes(d, f, bits)
        return (int(_active_experts(t, experts, top_k) * one) + _matrix_bytes(experts, d, 8) + 2 * (d + experts)
                + 4 * t * d + 6 * t * top_k, 2 * t * experts * d + 6 * t * top_k * d * f)


_KINDS = {"gemv": _Gemv, "qkv": _Qkv, "attention": _Attention, "moe_token": _MoeToken, "layers": _Layers,
          "gemm": _Gemm, "shared_block": _SharedBlock, "moe_block": _MoeBlock}


def prepare(case, seed):
    return _KINDS[case["kind"]](case, seed).ready()


def run(state):
    return state.run()


def exact(case, seed):
    return _KINDS[case["kind"]](case, seed).exact()


def work(case):
    size, flops = _KINDS[case["kind"]].work(**{k: v for k, v in case.items() if k not in ("name", "kind")})
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """About four times what the results were off their 64-bit values: the
    final rounding where there is one (fp16 2.1e-4, bf16 1.7e-3), the fp16
    weights of the matrix-core kernels (2.9e-4), the fp16 activations of the
    experts (5.4e-4), every fp16 vector of whole layers (1.3e-3). Expert
    indices may swap at ties of the fp32 logits."""
    rel = {"layers": 5e-3, "moe_token": 2e-3, "moe_block": 2e-3, "shared_block": 1.2e-3, "gemm": 1.2e-3}.get(
        case["kind"], 1e-3)
    if case.get("dtype") == "bf16":
        rel = 7e-3
    return {"rel": rel, "max": 10 * rel, "differ": 0.002}
