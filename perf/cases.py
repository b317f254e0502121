"""The calls that a serving program makes of this framework, with their inputs.

Five kinds of work, each through the public entry points:

  gemv     one quantised matrix times m rows (``q4_gemv_device``,
           ``q4k_matvec_device``): the smallest call there is;
  layers   a walk over MoE layers one call at a time (``moe_layer_device``), as
           a decoder does that runs its own attention between them;
  stack    the whole decoder stack of MoE layers in one call
           (``stack_forward_device``), or with the k-token acceptance after it
           (``verify_step_device``);
  prefill  the routed experts of a chunk of prompt tokens
           (``grouped_gemm_device``), layer after layer;
  head     final norm, LM head with the four best candidates, and the
           acceptance of the drafts (``rmsnorm_rows_device``,
           ``lm_head_logits_device``, ``accept_device``).

Model geometry: hidden 2048, 256 experts of width 512, top 8, one shared
expert, up to 40 layers, vocabulary 151936.  Each layer has its own weights at
its own address.  The weights, the context and the prepared stacks are made
once in a process and kept, as a server keeps them; a state holds the inputs
and outputs of one request.  A walk covers so many layers that the weights of
a pass do not stay in the 256 MB last-level cache.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from turboqwenfare_amd.backend import DeviceBuffer, HipBackend, Q4Weights

H, F, E, TOP_K, V = 2048, 512, 256, 8, 151936
SHAPES = ((F, H), (F, H), (H, F))  # gate, up, down
POOL = 8  # distinct matrices of each shape; expert e of layer l takes one of them
DEV = "cuda"


# ---- the cases -----------------------------------------------------------------------
def listed():
    return [
        # one expert matrix against one token: a caller that streams experts itself
        dict(name="gemv_q4_0_m1", kind="gemv", fmt="q4_0", rows=512, cols=2048, m=1),
        # plain decode, one token, attention between the layers done elsewhere
        dict(name="layers_q4_0_m1", kind="layers", fmt="q4_0", m=1, layers=16),
        # the same walk over four verify rows with the checkpoint's own expert format
        dict(name="layers_q4_k_m4", kind="layers", fmt="q4_k", m=4, layers=16),
        # plain decode and self-drafting: one token through the whole stack
        dict(name="stack_q4_0_m1", kind="stack", fmt="q4_0", m=1, layers=40, accept="none", vocab=0, temperature=0.0),
        dict(name="stack_q4_k_m1", kind="stack", fmt="q4_k", m=1, layers=40, accept="none", vocab=0, temperature=0.0),
        # the MTP verify step with three drafts, stochastic acceptance
        dict(name="verify_q4_0_m4", kind="stack", fmt="q4_0", m=4, layers=40, accept="stochastic", vocab=V, temperature=0.7),
        dict(name="verify_q4_k_m4", kind="stack", fmt="q4_k", m=4, layers=40, accept="stochastic", vocab=V, temperature=0.7),
        # the longest draft the interface takes: seven drafts, greedy
        dict(name="verify_q4_0_m8", kind="stack", fmt="q4_0", m=8, layers=40, accept="greedy", vocab=V, temperature=0.0),
        # a short prompt's tail, with an odd token count
        dict(name="prefill_t37", kind="prefill", t=37, layers=4, skew=1.1),
        # an ordinary prompt chunk with the skewed expert popularity of real routers
        dict(name="prefill_t512", kind="prefill", t=512, layers=2, skew=1.1),
        # the largest chunk the interface takes, experts evenly used
        dict(name="prefill_t4096", kind="prefill", t=4096, layers=1, skew=0.0),
        # logits of the four verify rows and the acceptance of three drafts
        dict(name="head_m4", kind="head", m=4, vocab=V, temperature=0.7),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["gemv", "layers", "stack", "stack", "prefill", "prefill", "head"])
    fmt = rng.choice(["q4_0", "q4_k"])
    if kind == "gemv":
        step = 32 if fmt == "q4_0" else 256
        return dict(kind=kind, fmt=fmt, rows=_log_int(rng, 64, 16384),
                    cols=step * max(1, _log_int(rng, 256, 8192) // step), m=rng.randint(1, 8))
    if kind == "layers":
        return dict(kind=kind, fmt=fmt, m=rng.randint(1, 8), layers=rng.randint(8, 20))
    if kind == "stack":
        m, accept = rng.randint(1, 8), rng.choice(["none", "greedy", "stochastic", "stochastic"])
        if accept == "none":
            return dict(kind=kind, fmt=fmt, m=m, layers=rng.randint(8, 40), accept=accept, vocab=0, temperature=0.0)
        return dict(kind=kind, fmt=fmt, m=max(m, 2), layers=rng.randint(8, 40), accept=accept,
                    vocab=rng.randint(32000, V), temperature=0.0 if accept == "greedy" else round(rng.uniform(0.5, 1.2), 2))
    if kind == "prefill":
        t = _log_int(rng, 9, 4096)
        return dict(kind=kind, t=t, layers=4 if t < 128 else 2 if t < 1024 else 1, skew=rng.choice([0.0, 0.7, 1.1]))
    return dict(kind=kind, m=rng.randint(1, 8), vocab=rng.randint(32000, V), temperature=round(rng.uniform(0.5, 1.2), 2))


# ---- seeded weights as GGML bytes, and their values ------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(shape, seed, std=1.0):
    return torch.randn(shape, generator=_gen(seed), device=DEV) * std


def _f16_bytes(x):
    return x.to(torch.float16).reshape(-1, 1).view(torch.uint8).reshape(-1, 2)


def _bytes(n, width, seed):
    return torch.randint(0, 256, (n, width), dtype=torch.uint8, device=DEV, generator=_gen(seed))


def _uniform(n, low, high, seed):
    return low + (high - low) * torch.rand(n, generator=_gen(seed), device=DEV)


def _q4_0_bytes(rows, cols, seed):
    """Nibbles symmetric around the zero point, scales U(0.005, 0.02)."""
    n = rows * (cols // 32)
    q = _bytes(n, 16, 2 * seed)
    q = torch.where((q & 15) == 0, q | 8, q)
    q = torch.where((q >> 4) == 0, q | 128, q)
    return torch.cat([_f16_bytes(_uniform(n, 0.005, 0.02, 2 * seed + 1)), q], 1).contiguous()


def _q4_0_values(b, rows, cols):
    d = b[:, :2].contiguous().view(torch.float16).double()
    q = b[:, 2:]
    return (d * (torch.cat([q & 15, q >> 4], 1).double() - 8.0)).reshape(rows, cols)


def _q4_k_bytes(rows, cols, seed, top=64):
    """Per sub-block the min equal to the scale (below `top`) and dmin = 7.5 d: values centred on zero."""
    n = rows * (cols // 256)
    d = _uniform(n, 1e-4, 4e-4, 3 * seed).to(torch.float16)
    sc = torch.randint(1, top, (n, 8), dtype=torch.uint8, device=DEV, generator=_gen(3 * seed + 1))
    lo, hi = sc[:, :4], sc[:, 4:]
    first = lo | ((hi >> 4) << 6)
    return torch.cat([_f16_bytes(d), _f16_bytes(d.float() * 7.5), first, first, (hi & 15) | ((hi & 15) << 4),
                      _bytes(n, 128, 3 * seed + 2)], 1).contiguous()


def _q4_k_values(b, rows, cols):
    d = b[:, 0:2].contiguous().view(torch.float16).double()[:, :, None]
    dmin = b[:, 2:4].contiguous().view(torch.float16).double()[:, :, None]
    s = b[:, 4:16]
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()[:, :, None]
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()[:, :, None]
    q = b[:, 16:].reshape(-1, 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
    return (d * sc * q - dmin * mn).reshape(rows, cols)


def _q6_k_bytes(rows, cols, seed):
    """Values with a standard deviation near 3 / sqrt(cols), so that logits are N(0, 9)."""
    n = rows * (cols // 256)
    sc = torch.randint(-16, 17, (n, 16), dtype=torch.int8, device=DEV, generator=_gen(3 * seed)).view(torch.uint8)
    std = 3.0 / math.sqrt(cols) / (9.5 * 18.5)
    return torch.cat([_bytes(n, 192, 3 * seed + 1), sc, _f16_bytes(_uniform(n, 0.5 * std, 1.5 * std, 3 * seed + 2))], 1).contiguous()


def _q6_k_values(b, rows, cols, dtype):
    out = torch.empty(rows, cols, dtype=dtype, device=DEV)
    per = cols // 256
    for r in range(0, rows, 8192):
        c = b[r * per:(r + 8192) * per]
        ql = c[:, :128].reshape(-1, 2, 2, 32)
        qh = c[:, 128:192].reshape(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        high = torch.cat([qh & 3, (qh >> 2) & 3, (qh >> 4) & 3, qh >> 6], 2)
        q = (low | (high << 4)).reshape(-1, 16, 16).to(dtype) - 32.0
        sc = c[:, 192:208].contiguous().view(torch.int8).to(dtype)[:, :, None]
        d = c[:, 208:210].contiguous().view(torch.float16).to(dtype)[:, :, None]
        out[r:r + 8192] = (d * sc * q).reshape(-1, cols)
    return out


_MAKE = {"q4_0": _q4_0_bytes, "q4_k": _q4_k_bytes}
_VALUES = {"q4_0": _q4_0_values, "q4_k": _q4_k_values}


def _pool_index(layer, expert, shape):
    return (layer * 5 + expert * 3 + shape) % POOL


def _pool_bytes(fmt):
    """The matrices of the three shapes.  The down matrices of q4_k have small scales, so that a layer adds a part
    of its residual stream and not a multiple of it: its 8-bit activations round, and a stack of layers that each
    replace the stream would show little but the rounding."""
    more = [{}, {}, dict(top=9) if fmt == "q4_k" else {}]
    return [[_MAKE[fmt](r, c, 1000 + 10 * i + j, **more[i]) for j in range(POOL)] for i, (r, c) in enumerate(SHAPES)]


def _layer_f32(layer):
    """(router [E, H], shared input gate [H], norm weight [H]) of a layer."""
    base = 100_000 + 10 * layer
    return (_normal((E, H), base, H ** -0.5), _normal((H,), base + 1, H ** -0.5),
            1.0 + 0.05 * _normal((H,), base + 2))


# ---- the resident model -----------------------------------------------------------------
_BACKEND, _MODELS, _HEADS = [], {}, {}


def _backend():
    if not _BACKEND:
        _BACKEND.append(HipBackend())
    return _BACKEND[0]


def _buf(t):
    return DeviceBuffer(t.data_ptr(), t.numel() * t.element_size())


def _upload(be, fmt, b, rows, cols):
    """A weight handle from GGML bytes that are already on the device."""
    if fmt == "q4_k":
        return be.upload_q4_k_device(_buf(b), rows, cols)
    if fmt == "q6_k":
        return be.upload_q6_k_device(_buf(b), rows, cols)
    h = ctypes.c_void_p()
    be._check(be.lib.tqf_hip_weights_upload_device(be.ctx, b.data_ptr(), b.numel(), rows, cols, ctypes.byref(h)))
    return Q4Weights(h.value, rows, cols)


class _Model:
    """The resident layers of one expert format, and the stacks prepared over them."""

    def __init__(self, fmt):
        self.fmt, self.pool, self.layers, self.norms, self.stacks = fmt, _pool_bytes(fmt), [], [], {}
        torch.cuda.synchronize()

    def ensure(self, n):
        be = _backend()
        for layer in range(len(self.layers), n):
            mats = [[_upload(be, self.fmt, self.pool[i][_pool_index(layer, e, i)], *SHAPES[i]) for e in range(E + 1)]
                    for i in range(3)]
            router, gate, norm = (t.cpu().numpy() for t in _layer_f32(layer))
            self.layers.append(be.prepare_moe_layer(be.upload_f32(router), be.upload_f32(gate), tuple(m[E] for m in mats),
                                                    mats[0][:E], mats[1][:E], mats[2][:E]))
            self.norms.append(be.upload_f32(norm))

    def stack(self, n):
        self.ensure(n)
        if n not in self.stacks:
            self.stacks[n] = _backend().prepare_stack(self.layers[:n], self.norms[:n])
        return self.stacks[n]


def _model(fmt):
    if fmt not in _MODELS:
        _MODELS[fmt] = _Model(fmt)
    return _MODELS[fmt]


def _head_norm():
    return 1.0 + 0.05 * _normal((H,), 77)


def _head(vocab):
    """(weights, norm, values in bf16 for a draft model's guess of the logits); the last vocabulary's are kept."""
    if vocab not in _HEADS:
        be = _backend()
        for w, norm, _ in _HEADS.values():
            be.free_weights(w)
            be.free_tensor(norm)
        _HEADS.clear()
        b = _q6_k_bytes(vocab, H, 5)
        torch.cuda.synchronize()
        _HEADS[vocab] = (_upload(be, "q6_k", b, vocab, H), be.upload_f32(_head_norm().cpu().numpy()),
                         _q6_k_values(b, vocab, H, torch.bfloat16))
    return _HEADS[vocab]


class _Gemv:
    """One matrix's handle, given back with the state."""

    def __init__(self, be, fmt, b, rows, cols):
        self.be, self.w = be, _upload(be, fmt, b, rows, cols)

    def __del__(self):
        self.be.free_weights(self.w)


# ---- inputs --------------------------------------------------------------------------------
def _routes(t, skew, seed):
    """Top-8 routes of t tokens from a Zipf(skew) expert popularity: ids [t, 8] and weights [t, 8]."""
    rng = np.random.default_rng(seed)
    rank = rng.permutation(E)
    scores = -skew * np.log(rank + 1.0)[None, :] + rng.gumbel(size=(t, E))
    ids = np.argsort(-scores, axis=1, kind="stable")[:, :TOP_K]
    p = np.exp(np.take_along_axis(scores, ids, 1) - scores.max(1, keepdims=True))
    return ids.astype(np.int16), (p / p.sum(1, keepdims=True)).astype(np.float32)


def _sample(logits, temperature, seed):
    """One token per row from softmax(logits / temperature), by Gumbel noise."""
    g = -torch.log(-torch.log(torch.rand(logits.shape, generator=_gen(seed), device=DEV).clamp_(1e-9, 1 - 1e-7)))
    return (logits / max(temperature, 1e-6) + (g if temperature > 0 else 0)).argmax(1).to(torch.int32)


def _drafts(guess, temperature, seed):
    """A draft model's logits near the target's, and the tokens drafted from them."""
    draft = (guess + _normal(guess.shape, seed)).contiguous()
    return draft, _sample(draft, temperature, seed + 1)


def _inputs(case, seed):
    """The tensors of one request, from the seed alone."""
    s = 1_000_003 * int(seed) + 17
    kind = case["kind"]
    if kind == "gemv":
        return dict(w=_MAKE[case["fmt"]](case["rows"], case["cols"], s), x=_normal((case["m"], case["cols"]), s + 1))
    if kind == "layers":
        return dict(x=_normal((case["layers"], case["m"], H), s))
    if kind == "prefill":
        routes = [_routes(case["t"], case["skew"], (s, i)) for i in range(case["layers"])]
        return dict(x=_normal((case["layers"], case["t"], H), s).to(torch.bfloat16),
                    ids=torch.from_numpy(np.stack([r[0] for r in routes])).to(DEV),
                    w=torch.from_numpy(np.stack([r[1] for r in routes])).to(DEV))
    m = case["m"]
    k = m - 1
    got = dict(h=_normal((m, H), s), u=torch.rand(max(k, 1), generator=_gen(s + 1), device=DEV),
               ur=torch.rand(m, generator=_gen(s + 2), device=DEV))
    if kind == "head":
        guess = (got["h"] * torch.rsqrt(got["h"].square().mean(1, keepdim=True) + 1e-6) * _head_norm()).to(torch.bfloat16)
        guess = (guess @ _head(case["vocab"])[2].T).float()
    elif case["accept"] != "none":
        guess = got["target"] = _normal((m, case["vocab"]), s + 3, 3.0)
    else:
        return got
    got["draft"], got["tokens"] = _drafts(guess[:k], case["temperature"], s + 4) if k else (guess[:0], torch.zeros(1, dtype=torch.int32, device=DEV))
    return got


def prepare(case, seed):
    be, kind, t = _backend(), case["kind"], _inputs(case, seed)
    new = lambda *shape, dtype=torch.float32: torch.zeros(shape, dtype=dtype, device=DEV)  # noqa: E731
    s = dict(be=be, case=dict(case), t=t)
    t["status"] = new(1, dtype=torch.int32)
    if kind == "gemv":
        torch.cuda.synchronize()
        s["w"] = _Gemv(be, case["fmt"], t.pop("w"), case["rows"], case["cols"])
        t["y"] = new(case["m"], case["rows"])
    elif kind == "layers":
        _model(case["fmt"]).ensure(case["layers"])
        s["layers"] = _model(case["fmt"]).layers[:case["layers"]]
        t.update(y=new(case["layers"], case["m"], H), ids=new(case["layers"], case["m"], TOP_K, dtype=torch.int16),
                 w=new(case["layers"], case["m"], TOP_K))
    elif kind == "prefill":
        _model("q4_0").ensure(case["layers"])
        s["layers"] = _model("q4_0").layers[:case["layers"]]
        t["y"] = new(case["layers"], case["t"], H)
    else:
        m = case["m"]
        t.update(out=new(m, H), accepted=new(1, dtype=torch.int32), emitted=new(m, dtype=torch.int32))
        if kind == "stack":
            s["stack"] = _model(case["fmt"]).stack(case["layers"])
        else:
            s["w"], s["norm"], _ = _head(case["vocab"])
            t.update(logits=new(m, case["vocab"]), tokens4=new(m, 4, dtype=torch.int32), logits4=new(m, 4))
    s["b"] = {k: _buf(v) for k, v in t.items()}
    if kind in ("layers", "prefill"):  # each layer's part of the buffers
        s["at"] = [{k: _buf(t[k][i]) for k in ("x", "y", "ids", "w")} for i in range(case["layers"])]
    torch.cuda.synchronize()
    return s


# ---- one pass ---------------------------------------------------------------------------------
def run(s):
    be, c, t, b = s["be"], s["case"], s["t"], s["b"]
    kind = c["kind"]
    if kind == "gemv":
        call = be.q4_gemv_device if c["fmt"] == "q4_0" else be.q4k_matvec_device
        call(s["w"].w, b["x"], c["m"], b["y"])
        return t["y"]
    if kind == "layers":
        for layer, at in zip(s["layers"], s["at"]):
            be.moe_layer_device(layer, at["x"], c["m"], at["y"], at["ids"], at["w"], b["status"])
        return dict(y=t["y"], ids=t["ids"], w=t["w"], status=t["status"])
    if kind == "prefill":
        for layer, at in zip(s["layers"], s["at"]):
            be.grouped_gemm_device(layer, at["x"], c["t"], at["ids"], at["w"], at["y"], b["status"])
        return dict(y=t["y"], status=t["status"])
    m = c["m"]
    if kind == "stack":
        if c["accept"] == "none":
            be.stack_forward_device(s["stack"], b["out"], m, d_status=b["status"], d_h_in=b["h"])
            return dict(h=t["out"], status=t["status"])
        be.verify_step_device(s["stack"], b["h"], b["out"], m, b["target"], b["draft"], b["tokens"], c["vocab"],
                              c["temperature"], c["accept"] == "greedy", b["u"], b["ur"], b["accepted"], b["emitted"],
                              b["status"])
        return dict(h=t["out"], accepted=t["accepted"], emitted=t["emitted"], status=t["status"])
    be.rmsnorm_rows_device(b["h"], m, H, s["norm"], b["out"])
    be.lm_head_logits_device(s["w"], b["out"], m, b["logits"], b["tokens4"], b["logits4"])
    be.accept_device(b["logits"], b["draft"] if m > 1 else b["logits"], b["tokens"], m - 1, c["vocab"], c["temperature"],
                     False, b["u"], b["ur"], b["accepted"], b["emitted"])
    return dict(logits=t["logits"], tokens4=t["tokens4"], logits4=t["logits4"], accepted=t["accepted"], emitted=t["emitted"])


# ---- what a pass cannot do without ------------------------------------------------------------
_MATRIX_BYTES = {"q4_0": F * H // 32 * 18, "q4_k": F * H // 256 * 144}


def _union(m):
    """Expected distinct experts of m tokens with even routes."""
    return E * (1.0 - (1.0 - TOP_K / E) ** m)


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        n = case["rows"] * case["cols"]
        return dict(bytes=n * (18 / 32 if case["fmt"] == "q4_0" else 144 / 256) + 4 * case["m"] * (case["rows"] + case["cols"]),
                    flops=2.0 * n * case["m"])
    if kind in ("layers", "stack"):
        m, n = case["m"], case["layers"]
        got = dict(bytes=n * ((_union(m) + 1) * 3 * _MATRIX_BYTES[case["fmt"]] + 4 * (E + 1) * H + 8 * m * H),
                   flops=n * m * 2.0 * H * ((TOP_K + 1) * 3 * F + E + 1))
        if case.get("accept", "none") != "none":
            rows = m + (m - 1 if case["accept"] == "stochastic" else 0)
            got["bytes"] += 4 * rows * case["vocab"]
            got["flops"] += 4.0 * rows * case["vocab"]
        return got
    if kind == "prefill":
        t, n = case["t"], case["layers"]
        used = sum(len(np.unique(_routes(t, case["skew"], i)[0])) for i in range(n))
        return dict(bytes=used * 3 * _MATRIX_BYTES["q4_0"] + n * t * (2 * H + 4 * H + 6 * TOP_K),
                    flops=6.0 * n * t * TOP_K * H * F)
    m, v = case["m"], case["vocab"]
    return dict(bytes=v * H / 256 * 210 + 8 * m * H + 4 * v * m + 4 * v * (m - 1), flops=2.0 * m * v * H + 4.0 * (2 * m - 1) * v)


def tolerance(case):
    kind = case["kind"]
    if kind == "gemv":  # f32 sums of exact products (3e-7 seen); the q4_k matvec's bits are defined
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "layers":
        # q4_0: f32 sums (6e-7 seen).  q4_k: activations rounded to 8 bits, where a last-bit change of the
        # hidden row moves a value to its other neighbour
        return {"rel": 1e-5, "max": 1e-4} if case["fmt"] == "q4_0" else {"rel": 5e-4, "max": 5e-3}
    if kind == "stack":
        # q4_0: f32 sums through 40 layers (4e-6 seen).  q4_k: a changed last bit moves 8-bit activations in
        # each layer that follows (1.1e-2 seen between f32 and 64-bit sums)
        return {"rel": 5e-5, "max": 2e-3} if case["fmt"] == "q4_0" else {"rel": 3e-2, "max": 0.5}
    if kind == "prefill":  # bf16 tokens, exact weights, the hidden row kept to 16 bits, f32 sums (3.4e-6 seen)
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 1e-3, "max": 1e-2}  # head: 8-bit activations, as for q4_k


# ---- the same in 64 bits ------------------------------------------------------------------------
def _q8(x):
    """Activations as the 8-bit block format keeps them: 256 values share one scale, -127 at the largest."""
    b = x.reshape(-1, 256)
    top = b.gather(1, b.abs().argmax(1, keepdim=True))
    inv = (-127.0 / torch.where(top == 0, torch.ones_like(top), top).float()).double()
    scale = (1.0 / inv.float()).double()
    return (torch.clamp(torch.round(b * inv), -128, 127) * scale * (top != 0)).reshape(x.shape)


class _Exact:
    """One format's layers in float64."""

    def __init__(self, fmt):
        self.q = _q8 if fmt == "q4_k" else (lambda x: x)
        self.values = [torch.stack([_VALUES[fmt](b, *SHAPES[i]) for b in row]) for i, row in enumerate(_pool_bytes(fmt))]

    def expert(self, layer, e, x):
        gate, up, down = (self.values[i][_pool_index(layer, e, i)] for i in range(3))
        x = self.q(x)
        return self.q(torch.nn.functional.silu(x @ gate.T) * (x @ up.T)) @ down.T

    def layer(self, layer, x):
        router, gate, _ = (t.double() for t in _layer_f32(layer))
        p = torch.softmax(x @ router.T, 1)
        w, ids = torch.topk(p, TOP_K, 1)
        w = w / w.sum(1, keepdim=True)
        y = torch.sigmoid(x @ gate)[:, None] * self.expert(layer, E, x)
        for r, row in enumerate(ids.tolist()):
            for k, e in enumerate(row):
                y[r] += w[r, k] * self.expert(layer, e, x[r:r + 1])[0]
        return y, w


def _norm64(x, weight):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * weight.double()


def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "gemv":
        x = t["x"].double()
        return (_q8(x) if case["fmt"] == "q4_k" else x) @ _VALUES[case["fmt"]](t["w"], case["rows"], case["cols"]).T
    if kind == "layers":
        ex = _Exact(case["fmt"])
        got = [ex.layer(i, t["x"][i].double()) for i in range(case["layers"])]
        return dict(y=torch.stack([g[0] for g in got]), ids=None, w=torch.stack([g[1] for g in got]), status=None)
    if kind == "stack":
        ex, h = _Exact(case["fmt"]), t["h"].double()
        for i in range(case["layers"]):
            h = h + ex.layer(i, _norm64(h, _layer_f32(i)[2]))[0]
        return dict(h=h, accepted=None, emitted=None, status=None) if case["accept"] != "none" else dict(h=h, status=None)
    if kind == "prefill":
        ex, y = _Exact("q4_0"), torch.zeros(case["layers"], case["t"], H, dtype=torch.float64, device=DEV)
        for i in range(case["layers"]):
            for e in range(E):
                at, k = torch.nonzero(t["ids"][i] == e, as_tuple=True)
                if len(at):
                    y[i].index_add_(0, at, ex.expert(i, e, t["x"][i][at].double()) * t["w"][i][at, k].double()[:, None])
        return dict(y=y, status=None)
    x = _q8(_norm64(t["h"].double(), _head_norm()))
    w = _q6_k_values(_q6_k_bytes(case["vocab"], H, 5), case["vocab"], H, torch.float64)
    logits = x @ w.T
    return dict(logits=logits, tokens4=None, logits4=torch.topk(logits, 4, 1).values, accepted=None, emitted=None)
