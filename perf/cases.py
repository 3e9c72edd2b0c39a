"""What the framework is timed on: the calls that a program decoding or
prefilling with packed weights makes, through the public entry points of
``vxg_amd.engine``.

A case is one call (one "pass"); ``op`` names it:

* ``matmul``   ``HipEngine.matmul_dev``: one projection, batch 1..8 (decode)
  or larger (prefill), for each weight kind, bf16 or f32 activations and
  outputs;
* ``glu``      ``HipEngine.ffn_glu_dev``: the gated FFN projection over
  [gate; up];
* ``attn``     ``KvQ8Cache.step``: the whole attention step over a Q8_0 KV
  cache, one token (decode) or a causal batch (prefill);
* ``model``    ``DecodeRunner.step``: a whole decoder, one token or a prompt,
  the last token's logits.

Weights, activations and caches are drawn on the GPU from the seed, in the
distributions of ``vxg_amd.synth`` (indices and int8 values uniform, f16
scales uniform in [0.002, 0.02], codebooks normal and sorted, 0.74 %
residual outliers, activations N(0, 1)).
"""
from __future__ import annotations

import math

import numpy as np
import torch

from vxg_amd import engine as E
from vxg_amd.formats import Cb4G64Matrix, CodebookMatrix, Q4_0Matrix, q8_from_planes

DEV = "cuda"
OUTLIERS = 0.0074
VOCAB = 151936

_engine = None


def engine() -> E.HipEngine:
    """One engine for the process, as a program keeps it."""
    global _engine
    if _engine is None:
        _engine = E.HipEngine(0)
    return _engine


# --------------------------------------------------------------------------
# cases
# --------------------------------------------------------------------------

def _matmul(name, kind, m, k, n, x="bf16", y="bf16"):
    return {"name": name, "op": "matmul", "kind": kind, "m": m, "k": k, "n": n, "x": x, "y": y}


def _glu(name, kind, m, k, ffn, act="silu"):
    return {"name": name, "op": "glu", "kind": kind, "m": m, "k": k, "ffn": ffn, "act": act}


def _attn(name, batch, pos, n_head, n_kv, hd, gated=True, norm=True, rope=64, neox=True):
    return {"name": name, "op": "attn", "batch": batch, "pos": pos, "n_head": n_head, "n_kv": n_kv, "hd": hd,
            "gated": gated, "norm": norm, "rope": rope, "neox": neox}


def _model(name, kind, layers, batch, pos, hidden=2048, ffn=6144, n_head=16, n_kv=16, hd=128, vocab=VOCAB,
           gated=False, act="silu"):
    return {"name": name, "op": "model", "kind": kind, "layers": layers, "batch": batch, "pos": pos,
            "hidden": hidden, "ffn": ffn, "n_head": n_head, "n_kv": n_kv, "hd": hd, "vocab": vocab, "gated": gated,
            "act": act}


def listed():
    return [
        # the gated FFN of one decode token, called on its own: launch and
        # latency count
        _glu("glu cb4 m1", "cb4", 1, 2048, 6144),
        # the LM head for eight sequences decoded together
        _matmul("head q8 m8", "q8", 8, 2048, VOCAB, y="f32"),
        # the gated FFN of four sequences decoded together
        _glu("glu cb4 m4", "cb4", 4, 2048, 6144),
        # a short prompt or a speculated run of tokens to verify, on GGUF's
        # 4-bit blocks
        _matmul("short q4_0 m32", "q4_0", 32, 2048, 6144),
        # a prompt of an ordinary chat turn, ragged
        _matmul("prompt g64 m100", "g64", 100, 6144, 2048),
        # the attention output projection of a prompt: f32 activations in, the
        # f32 residual delta out
        _matmul("out-proj q8 m500 f32", "q8", 500, 2048, 2048, x="f32", y="f32"),
        # a long prompt on the reference's own codebook layout
        _matmul("prompt cb4 m2048", "cb4", 2048, 2048, 6144),
        # the gated FFN of a long prompt
        _glu("glu g64 m1024", "g64", 1024, 2048, 6144),
        # one token's attention far into a conversation, grouped queries
        _attn("attn decode 32k", 1, 32000, 16, 4, 128),
        # a long prompt's causal attention
        _attn("attn prefill 2048", 2048, 0, 16, 16, 128),
        # one decode token through the whole decoder of the benchmark's
        # linear stack
        _model("token g64 24 layers", "g64", 24, 1, 600),
        # a prompt through the whole decoder on the reference's layout
        _model("prompt cb4 24 layers", "cb4", 24, 500, 0),
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    """Log-uniform in [lo, hi]; a multiple of `step` mostly, any size at times."""
    v = _logu(rng, lo, hi)
    return v if rng.random() < 0.15 else min(max(step, v // step * step), hi // step * step)


def draw(rng):
    op = rng.choice(("decode", "decode", "gemm", "gemm", "gemm", "glu", "glu", "attn1", "attnm", "token", "prompt"))
    kind = rng.choice(("cb4", "g64", "q8", "q4_0"))
    x = rng.choice(("bf16", "bf16", "bf16", "f32"))
    y = rng.choice(("bf16", "f32"))
    if op == "decode":
        m = rng.choice((1, 2, 3, 4, 5, 6, 8))
        if rng.random() < 0.25:
            return _unnamed(_matmul("", kind, m, _size(rng, 1024, 2048, 64), _size(rng, 32000, VOCAB, 16), "bf16", "f32"))
        return _unnamed(_matmul("", kind, m, _size(rng, 1024, 8192, 64), _size(rng, 1024, 16384, 64), x, y))
    if op == "gemm":
        while True:
            c = _matmul("", kind, _logu(rng, 9, 2048), _size(rng, 512, 8192, 64), _size(rng, 512, 16384, 64), x, y)
            if c["m"] * c["k"] * c["n"] <= 3e10:
                return _unnamed(c)
    if op == "glu":
        return _unnamed(_glu("", kind, _logu(rng, 1, 1024), _size(rng, 1024, 2048, 64), _size(rng, 1024, 6144, 64),
                             rng.choice(("silu", "silu", "gelu"))))
    hd = rng.choice((64, 128, 128))
    n_kv = rng.choice((2, 4, 8, 16))
    n_head = n_kv * rng.choice([g for g in (1, 2, 4, 8) if n_kv * g <= 32])
    gated, norm, neox = (rng.random() < 0.5 for _ in range(3))
    if op == "attn1":
        return _unnamed(_attn("", 1, _logu(rng, 64, 60000), n_head, n_kv, hd, gated, norm, rng.choice((hd, hd // 2)), neox))
    if op == "attnm":
        return _unnamed(_attn("", _logu(rng, 2, 2048), rng.choice((0, 0, _logu(rng, 16, 6000))), min(n_head, 16),
                              min(n_kv, 16), hd, gated, norm, rng.choice((hd, hd // 2)), neox))
    hidden = rng.choice((1024, 1536, 2048))
    n_head = hidden // hd
    n_kv = n_head // rng.choice([g for g in (1, 2, 4) if n_head % g == 0])
    c = _model("", kind, rng.randint(2, 12), 1 if op == "token" else _logu(rng, 2, 500), 0, hidden,
               _size(rng, 2048, 6144, 64), n_head, n_kv, hd, _size(rng, 32000, VOCAB, 16), gated,
               rng.choice(("silu", "silu", "gelu")))
    c["pos"] = rng.choice((0, _logu(rng, 16, 1500)))
    return _unnamed(c)


def _unnamed(c):
    return {k: v for k, v in c.items() if k != "name"}


# --------------------------------------------------------------------------
# weights: drawn on the GPU, handed to the engine as the host planes it takes
# --------------------------------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _u16(t: torch.Tensor) -> np.ndarray:
    return t.to(torch.float16).contiguous().view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1)


def _scales(shape, g):
    return (torch.rand(shape, generator=g, device=DEV) * 0.018 + 0.002).to(torch.float16)


def _nibbles(rows, kp, cols, pad, g):
    q = torch.randint(0, 16, (rows, kp), generator=g, device=DEV, dtype=torch.uint8)
    if kp != cols:
        q[:, cols:] = pad
    return q


class Weight:
    """One packed matrix: its host form for the engine, its f64 values for
    ``exact``, and the bytes of its packed planes."""

    def __init__(self, kind, rows, cols, g, centred=False, exact=False):
        self.rows, self.cols = rows, cols
        make = {"cb4": self._cb4, "g64": self._g64, "q8": self._q8, "q4_0": self._q40}[kind]
        make(rows, cols, g, centred, exact)

    def _g64(self, rows, cols, g, centred, exact):
        kp = (cols + 63) // 64 * 64
        q = _nibbles(rows, kp, cols, 0, g)
        lut = (torch.randn((rows, kp // 64, 16), generator=g, device=DEV) * 0.02).sort(dim=-1).values.to(torch.float16)
        if exact:
            self.values = lut.double().gather(2, q.view(rows, kp // 64, 64).long()).view(rows, kp)[:, :cols]
        else:
            self.host = Cb4G64Matrix(rows, cols, kp, (q[:, 0::2] | (q[:, 1::2] << 4)).cpu().numpy().reshape(-1), _u16(lut))

    def _cb4(self, rows, cols, g, centred, exact):
        kp = (cols + 255) // 256 * 256
        q = _nibbles(rows, kp, cols, 0, g)
        cent = torch.randn(16, generator=g, device=DEV).sort().values
        if centred:
            cent = cent - cent.mean()
        sc = _scales((rows, kp // 128), g)
        hit = torch.rand((rows, cols), generator=g, device=DEV) < OUTLIERS
        at = hit.nonzero()
        res = (torch.randn(at.shape[0], generator=g, device=DEV) * 0.02).to(torch.float16)
        if exact:
            w = cent.double()[q.long()] * sc.double().repeat_interleave(128, dim=1)
            w[at[:, 0], at[:, 1]] += res.double()
            self.values = w[:, :cols]
            return
        ptr = np.zeros(rows + 1, np.uint32)
        ptr[1:] = hit.sum(dim=1).cumsum(0).cpu().numpy().astype(np.uint32)
        packed = at[:, 1].cpu().numpy().astype(np.uint32) | (_u16(res).astype(np.uint32) << 16)
        words = (q[:, 0::2] | (q[:, 1::2] << 4)).contiguous().cpu().numpy().view(np.uint32).reshape(-1)
        self.host = CodebookMatrix(rows, cols, kp, cent.cpu().numpy(), _u16(sc), words, ptr, packed)

    def _q8(self, rows, cols, g, centred, exact):
        kb = (cols + 31) // 32
        q = torch.randint(-127, 128, (rows, kb * 32), generator=g, device=DEV, dtype=torch.int8)
        if kb * 32 != cols:
            q[:, cols:] = 0
        sc = _scales((rows, kb), g)
        if exact:
            self.values = (q.double().view(rows, kb, 32) * sc.double()[..., None]).view(rows, -1)[:, :cols]
        else:
            self.host = q8_from_planes(rows, cols, q.cpu().numpy(), _u16(sc))

    def _q40(self, rows, cols, g, centred, exact):
        kb = (cols + 31) // 32
        q = _nibbles(rows, kb * 32, cols, 8, g).view(rows, kb, 32)
        sc = _scales((rows, kb), g)
        if exact:
            self.values = ((q.double() - 8) * sc.double()[..., None]).view(rows, -1)[:, :cols]
        else:
            words = (q[..., :16] | (q[..., 16:] << 4)).contiguous().cpu().numpy().view(np.uint32).reshape(-1)
            self.host = Q4_0Matrix(rows, cols, kb * 32, _u16(sc), words)


def _packed_bytes(kind, rows, cols):
    if kind == "g64":
        return rows * ((cols + 63) // 64) * (32 + 32)
    if kind == "cb4":
        return rows * ((cols + 127) // 128) * (64 + 2) + 4 * rows * (1 + OUTLIERS * cols)
    return rows * ((cols + 31) // 32) * (34 if kind == "q8" else 18)


def _parts(kind, sizes, cols, g, centred=False, exact=False):
    """Matrices of `sizes` rows each (the parts of a concatenated tensor;
    Q4_0 is uploaded as one)."""
    if kind == "q4_0":
        sizes = (sum(sizes),)
    return [Weight(kind, r, cols, g, centred, exact) for r in sizes]


def _upload(parts):
    if len(parts) == 1:
        return engine().upload_packed(parts[0].host)
    return engine().upload_concat([p.host for p in parts])


# --------------------------------------------------------------------------
# states
# --------------------------------------------------------------------------

class State:
    """What a program holds between calls."""

    def __init__(self, case):
        self.case = case


class Owned:
    """An engine object that has to be freed by hand, freed with its last
    holder: the state, or a torch view of its memory."""

    def __init__(self, obj):
        self.obj = obj

    def __del__(self):
        try:
            torch.cuda.synchronize()
            self.obj.free()
        except Exception:
            pass


class _Region:
    """A device buffer of the engine, for a torch view of it without a copy;
    the view holds this object, and with it the buffer's owner."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def _view(owner, buf, shape, typestr):
    return torch.as_tensor(_Region(owner, buf.ptr, shape, typestr), device=DEV)


def _torch_dtype(name):
    return torch.bfloat16 if name == "bf16" else torch.float32


def _abi_dtype(name):
    return E.DTYPE_BF16 if name == "bf16" else E.DTYPE_F32


def _quantise(t):
    """Q8_0 blocks of 32 along the last axis: int8 values, f16 scales."""
    b = t.float().unflatten(-1, (-1, 32))
    d = (b.abs().amax(-1) / 127.0).to(torch.float16)
    inv = torch.where(d > 0, 1.0 / d.float(), torch.zeros_like(d, dtype=torch.float32))
    q = (b * inv[..., None]).round().clamp(-127, 127).to(torch.int8)
    return q.flatten(-2), d


def _randn(shape, g, scale=1.0):
    return torch.randn(shape, generator=g, device=DEV) * scale


def _cases_attn_inputs(case, seed):
    c, g = case, _gen(seed)
    hd, per, seq = c["hd"], c["n_kv"] * c["hd"], c["pos"] + c["batch"]
    q_rows = c["n_head"] * hd * (2 if c["gated"] else 1)
    d = {"q": _randn((c["batch"], q_rows), g), "k": _randn((c["batch"], per), g), "v": _randn((c["batch"], per), g)}
    d["qn"], d["kn"] = (1 + _randn(hd, g, 0.1) for _ in range(2))
    d["k_cache"], d["v_cache"] = (_quantise(_randn((c["pos"], per), g)) for _ in range(2))
    d["seq"], d["per"], d["q_rows"] = seq, per, q_rows
    return d


def _prepare_attn(case, seed):
    c, eng = case, engine()
    d = _cases_attn_inputs(c, seed)
    s = State(c)
    s.cache = eng.kv_q8_cache(d["seq"], c["n_kv"], c["hd"])
    own = s.own = Owned(s.cache)
    per, pos = d["per"], c["pos"]
    s.rows = []
    for (qs, dd), which in ((d["k_cache"], "k"), (d["v_cache"], "v")):
        vq = _view(own, getattr(s.cache, which + "_qs"), (d["seq"], per), "|i1")
        vd = _view(own, getattr(s.cache, which + "_d"), (d["seq"], per // 32), "<f2")
        vq.zero_()
        vd.zero_()
        vq[:pos] = qs
        vd[:pos] = dd
        s.rows += [vq[pos:], vd[pos:]]
    s.q, s.k, s.v, s.qn, s.kn = (d[n].contiguous() for n in ("q", "k", "v", "qn", "kn"))
    s.out = torch.zeros((c["batch"], c["n_head"] * c["hd"]), device=DEV)
    s.params = E.GqaParams(s.qn.data_ptr() if c["norm"] else 0, s.kn.data_ptr() if c["norm"] else 0, 0, 0, 0,
                           c["n_head"], int(c["gated"]), c["rope"], int(c["neox"]), 1e6, 1e-6)
    return s


def _run_attn(s):
    c = s.case
    s.cache.step(s.params, s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(), c["pos"], c["pos"], s.out.data_ptr(),
                 batch_m=c["batch"], q_stride=s.q.shape[1], kv_stride=s.k.shape[1])
    return {"out": s.out, "k_qs": s.rows[0], "k_d": s.rows[1], "v_qs": s.rows[2], "v_d": s.rows[3]}


def _model_weights(case, seed, exact=False):
    """Two layers' matrices drawn; a decoder's layers use them in turn (each
    layer with memory of its own)."""
    c, g = case, _gen(seed)
    H, per = c["hidden"], c["n_kv"] * c["hd"]
    aw = c["n_head"] * c["hd"]
    qr = aw * (2 if c["gated"] else 1)
    layers = []
    for _ in range(min(2, c["layers"])):
        layers.append({"in": _parts(c["kind"], (qr, per, per), H, g, True, exact),
                       "out": _parts(c["kind"], (H,), aw, g, True, exact),
                       "gu": _parts(c["kind"], (c["ffn"], c["ffn"]), H, g, True, exact),
                       "dn": _parts(c["kind"], (H,), c["ffn"], g, True, exact)})
    head = Weight("q8", c["vocab"], H, g, False, exact)
    norms = [1 + _randn(H, g, 0.1) for _ in range(2 * c["layers"] + 1)]
    qk = [1 + _randn(c["hd"], g, 0.1) for _ in range(2)]
    ids = torch.randint(0, c["vocab"], (c["pos"] + c["batch"],), generator=g, device=DEV).cpu().numpy().astype(np.uint32)
    return layers, head, norms, qk, ids


def _prepare_model(case, seed):
    c, eng = case, engine()
    layers, head, norms, qk, ids = _model_weights(c, seed)
    s = State(c)
    up = [{k: _upload(v) for k, v in L.items()} for L in layers]
    s.weights = list(up)
    for i in range(len(up), c["layers"]):
        s.weights.append({k: t.clone() for k, t in up[i % len(up)].items()})
    s.head = _upload([head])
    s.norms, s.qk = norms, qk
    rl = [E.RunnerLayer(L["in"].handle, L["out"].handle, L["gu"].handle, L["dn"].handle, norms[2 * i].data_ptr(),
                        norms[2 * i + 1].data_ptr(), qk[0].data_ptr(), qk[1].data_ptr())
          for i, L in enumerate(s.weights)]
    cfg = E.RunnerConfig(c["layers"], c["hidden"], c["n_head"], c["n_kv"], c["hd"], c["ffn"], c["vocab"],
                         int(c["gated"]), c["hd"], 1, E.ACT_GELU_TANH if c["act"] == "gelu" else E.ACT_SILU,
                         c["pos"] + c["batch"] + 64, max(c["batch"], c["pos"], 1), 1e6, 1e-6, 1.0)
    torch.cuda.synchronize()
    s.runner = eng.runner(cfg, rl, norms[-1].data_ptr(), s.head, s.head)
    s.own = Owned(s.runner)
    if c["pos"]:
        s.runner.step(ids[:c["pos"]], 0, want_logits=False)
    s.ids = ids[c["pos"]:]
    return s


def _matmul_rows(case):
    return (case["n"],) if case["op"] == "matmul" else (case["ffn"], case["ffn"])


def _matmul_inputs(case, seed, exact=False):
    g = _gen(seed)
    w = _parts(case["kind"], _matmul_rows(case), case["k"], g, False, exact)
    # the activation is N(0, 1); a gated product gets a smaller one where the
    # weights would push every gate far into saturation
    gain = 1.0 if case["op"] == "matmul" else 2.0 / {"g64": 0.02, "cb4": 0.012, "q8": 0.88, "q4_0": 0.056}[case["kind"]] / case["k"] ** 0.5
    x = _randn((case["m"], case["k"]), g, gain).to(_torch_dtype(case.get("x", "bf16")))
    return w, x


def prepare(case, seed):
    if case["op"] == "attn":
        return _prepare_attn(case, seed)
    if case["op"] == "model":
        return _prepare_model(case, seed)
    w, x = _matmul_inputs(case, seed)
    s = State(case)
    s.w = _upload(w)
    s.x = x
    s.y = torch.zeros((case["m"], case.get("n") or case["ffn"]), device=DEV, dtype=_torch_dtype(case.get("y", "bf16")))
    return s


def run(s):
    c = s.case
    if c["op"] == "attn":
        return _run_attn(s)
    if c["op"] == "model":
        return s.runner.step(s.ids, c["pos"])
    if c["op"] == "glu":
        engine().ffn_glu_dev(s.w, s.x.data_ptr(), E.DTYPE_BF16, c["m"], s.y.data_ptr(), E.DTYPE_BF16,
                             activation=E.ACT_GELU_TANH if c["act"] == "gelu" else E.ACT_SILU)
        return s.y
    engine().matmul_dev(s.w, s.x.data_ptr(), _abi_dtype(c["x"]), c["m"], s.y.data_ptr(), _abi_dtype(c["y"]))
    return s.y


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------

def _attn_work(batch, pos, n_head, n_kv, hd, gated):
    per = n_kv * hd
    pairs = batch * pos + batch * (batch + 1) / 2
    return {"bytes": 2 * (pos + batch) * per * 34 / 32 + batch * 4 * (2 * per + n_head * hd * (3 if gated else 2)),
            "flops": 4 * n_head * hd * pairs}


def work(case):
    c = case
    if c["op"] == "attn":
        return _attn_work(c["batch"], c["pos"], c["n_head"], c["n_kv"], c["hd"], c["gated"])
    if c["op"] == "model":
        H, F, per, aw = c["hidden"], c["ffn"], c["n_kv"] * c["hd"], c["n_head"] * c["hd"]
        shapes = [(aw * (2 if c["gated"] else 1) + 2 * per, H), (H, aw), (2 * F, H), (H, F)]
        a = _attn_work(c["batch"], c["pos"], c["n_head"], c["n_kv"], c["hd"], c["gated"])
        kv = 2 * (c["pos"] + c["batch"]) * per * 34 / 32
        return {"bytes": c["layers"] * (sum(_packed_bytes(c["kind"], r, k) for r, k in shapes) + kv)
                + _packed_bytes("q8", c["vocab"], H) + 4 * c["vocab"],
                "flops": c["layers"] * (sum(2 * c["batch"] * r * k for r, k in shapes) + a["flops"]) + 2 * c["vocab"] * H}
    rows = sum(_matmul_rows(c))
    out = c.get("n") or c["ffn"]
    size = {"bf16": 2, "f32": 4}
    return {"bytes": _packed_bytes(c["kind"], rows, c["k"]) + c["m"] * c["k"] * size[c.get("x", "bf16")]
            + c["m"] * out * size[c.get("y", "bf16")],
            "flops": 2 * c["m"] * rows * c["k"]}


# --------------------------------------------------------------------------
# what the outputs are in 64 bits, and how far another implementation may be
# --------------------------------------------------------------------------

def _norm64(x, w, eps=1e-6):
    return x * (x.square().mean(-1, keepdim=True) + eps).rsqrt() * w.double()


def _rope64(x, pos0, rope, neox):
    """x [tokens, heads, hd], token t at position pos0 + t; the angle is the
    f32 product of the position and the f32 frequency, as the path defines it."""
    half = rope // 2
    i = np.arange(half, dtype=np.float32)
    freq = np.power(np.float32(1e6), -(np.float32(2) * i) / np.float32(rope), dtype=np.float32)
    ang = np.arange(pos0, pos0 + x.shape[0], dtype=np.float32)[:, None] * freq[None]
    ang = torch.from_numpy(ang.astype(np.float32)).to(DEV).double()[:, None, :]
    cos, sin = ang.cos(), ang.sin()
    out = x.clone()
    a, b = (slice(0, half), slice(half, rope)) if neox else (slice(0, rope, 2), slice(1, rope, 2))
    out[..., a] = x[..., a] * cos - x[..., b] * sin
    out[..., b] = x[..., a] * sin + x[..., b] * cos
    return out


def _attn64(q, k, v, qn, kn, k_cache, v_cache, pos, n_head, n_kv, hd, gated, rope, neox):
    """The attention step in 64 bits over a cache kept in its Q8_0 form:
    (out, rows of the cache written)."""
    m = q.shape[0]
    qd = q.double().view(m, n_head, 2 if gated else 1, hd)
    qh, gate = qd[:, :, 0], qd[:, :, 1] if gated else None
    kh, vh = k.double().view(m, n_kv, hd), v.double().view(m, n_kv, hd)
    if qn is not None:
        qh, kh = _norm64(qh, qn), _norm64(kh, kn)
    qh, kh = _rope64(qh, pos, rope, neox), _rope64(kh, pos, rope, neox)
    new = [*_quantise(kh.reshape(m, -1)), *_quantise(vh.reshape(m, -1))]
    K, V = (torch.cat([cq[:pos].double().unflatten(-1, (-1, 32)) * cd[:pos].double()[..., None],
                       nq.double().unflatten(-1, (-1, 32)) * nd.double()[..., None]]).view(pos + m, n_kv, hd)
            for (cq, cd), (nq, nd) in ((k_cache, new[:2]), (v_cache, new[2:])))
    out = torch.empty((m, n_head, hd), device=DEV, dtype=torch.float64)
    t = torch.arange(pos + m, device=DEV)
    for h in range(n_head):
        kv = h // (n_head // n_kv)
        for r in range(0, m, 512):
            rows = slice(r, min(r + 512, m))
            s = qh[rows, h] @ K[:, kv].T / hd ** 0.5
            s.masked_fill_(t[None] > (torch.arange(r, rows.stop, device=DEV) + pos)[:, None], -math.inf)
            out[rows, h] = s.softmax(-1) @ V[:, kv]
    if gated:
        out = out * gate.sigmoid()
    return out.view(m, -1), new


def _act64(g, act):
    return torch.nn.functional.gelu(g, approximate="tanh") if act == "gelu" else torch.nn.functional.silu(g)


def _model64(case, seed):
    c = case
    layers, head, norms, qk, ids = _model_weights(c, seed, exact=True)
    emb = torch.from_numpy(ids.astype(np.int64)).to(DEV)
    cur = head.values[emb]
    H, per, aw = c["hidden"], c["n_kv"] * c["hd"], c["n_head"] * c["hd"]
    qr = aw * (2 if c["gated"] else 1)
    mats = [{k: torch.cat([p.values for p in v]) for k, v in L.items()} for L in layers]
    for i in range(c["layers"]):
        W = mats[i % len(mats)]
        qkv = _norm64(cur, norms[2 * i]) @ W["in"].T
        none = (torch.zeros((0, per), device=DEV, dtype=torch.int8), torch.zeros((0, per // 32), device=DEV, dtype=torch.float16))
        a, _ = _attn64(qkv[:, :qr], qkv[:, qr:qr + per], qkv[:, qr + per:], qk[0], qk[1], none, none, 0, c["n_head"],
                       c["n_kv"], c["hd"], c["gated"], c["hd"], True)
        cur = cur + a @ W["out"].T
        gu = _norm64(cur, norms[2 * i + 1]) @ W["gu"].T
        cur = cur + (_act64(gu[:, :c["ffn"]], c["act"]) * gu[:, c["ffn"]:]) @ W["dn"].T
    return (_norm64(cur[-1:], norms[-1]) @ head.values.T)[0].cpu().numpy()


def exact(case, seed):
    c = case
    if c["op"] == "model":
        return _model64(c, seed)
    if c["op"] == "attn":
        d = _cases_attn_inputs(c, seed)
        out, new = _attn64(d["q"], d["k"], d["v"], d["qn"] if c["norm"] else None, d["kn"] if c["norm"] else None,
                           d["k_cache"], d["v_cache"], c["pos"], c["n_head"], c["n_kv"], c["hd"], c["gated"],
                           c["rope"], c["neox"])
        # the cache's rows are codes, not computed numbers
        return {"out": out, "k_qs": None, "k_d": None, "v_qs": None, "v_d": None}
    w, x = _matmul_inputs(c, seed, exact=True)
    # in slices of rows: a vocabulary's values in 64 bits are large
    y = torch.cat([x.double() @ r.T for p in w for r in p.values.split(16384)], dim=1)
    return y if c["op"] == "matmul" else _act64(y[:, :c["ffn"]], c["act"]) * y[:, c["ffn"]:]


def tolerance(case):
    """Relative errors measured against ``exact``, times about four."""
    c = case
    if c["op"] == "model":
        # bf16 between the projections of every layer
        return {"rel": 0.03, "max": 0.15}
    if c["op"] == "attn":
        # f32 sums; the written rows' f16 scales and int8 codes can take the
        # other neighbour where a normed, rotated value lies on a boundary
        return {"rel": 5e-4, "max": 0.02, "differ": 0.01}
    if c["op"] == "glu" or c["y"] == "bf16":
        return {"rel": 7e-3, "max": 0.016}
    return {"rel": 2e-6, "max": 2e-5}
