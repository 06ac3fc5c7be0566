"""Workloads of the MI355X decode backend, each one pass through its public entry points.

A case is a dict of plain values.  Its "kind" names the entry point:

  call     HipBackend.matvec: one matvec with host arrays in and out, as a needle.js host makes it
  matvec   nd_matvec_d: activations and result in HBM, int8 (bits 0) or Cactus-Quant matrices
  matmul   nd_matmul_d: per-row-scaled int8 matrices over many activation rows
  attend   nd_kv_store_d + nd_attention_d for every layer of one decoded token
  select   nd_select_mask_d: constrained greedy selection of a batch
  prefill  HipPrefill.run: a prompt through the 8-layer synthetic decoder
  decode   nd_batch_step: one step of a constrained batch over ragged contexts
  needle   Needle 2 at the shipped geometry: a prompt, then a token at a time

Models and matrices are fixed (a program serves one model); prompts, activations, caches and masks
come from the seed.  Outputs that live in HBM are the state's own buffers.
"""

from __future__ import annotations

import collections
import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parent.parent
for p in (ROOT, ROOT / "needle.js_amd"):
    if str(p) not in sys.path:
        sys.path.insert(0, str(p))

from needle_hip import (CqMatrix, HipBackend, HipKvCache, Int8Matrix, Needle2Geometry,  # noqa: E402
                        Needle2Weights, NeedleModel, pack_codes, synth)
from needle_hip.models import (MASK_P, PREFIX_SCALE, DecoderGeometry, HipBatch,  # noqa: E402
                               HipDecoder, HipPrefill)

DEVICE = "cuda:0"
HD = 64  # head dimension of every model here


def listed():
    return [
        # One product of a host-driven layer (the 512 x 512 output projection): latency only.
        dict(name="call_i8_512", kind="call", bits=0, n=512, k=512, g=512, batch=1),
        # The isolated quantized matvec at a size that streams from HBM, batch 1.
        dict(name="matvec_i8_16384_b1", kind="matvec", bits=0, n=16384, k=4096, g=32, batch=1),
        # The same group-scaled matrix form for the 64 sequences of a decoding batch.
        dict(name="matvec_i8_4096_b64", kind="matvec", bits=0, n=4096, k=4096, g=32, batch=64),
        # The archive's own 4-bit form, batch 1: the logits of a large vocabulary.
        dict(name="matvec_cq4_32768_b1", kind="matvec", bits=4, n=32768, k=2048, g=32, batch=1),
        # The archive's q/k/v/gate rows over a tool prompt's positions (ragged count).
        dict(name="matvec_cq4_1536_b300", kind="matvec", bits=4, n=1536, k=512, g=32, batch=300),
        # A prompt-sized product of the synthetic decoder (feed-forward up), ragged row count.
        dict(name="matmul_2048x512_m2000", kind="matmul", n=2048, k=512, rows=2000),
        # One decoded token's cache work: append and attend in each of 8 layers at 8192 positions.
        dict(name="attend_8x8192", kind="attend", layers=8, kv_heads=8, rep=1, length=8192,
             window=0, sink=0, mode="int8"),
        # Constrained selection of a 64-sequence batch over the synthetic decoder's vocabulary.
        dict(name="select_64x32768", kind="select", batch=64, vocab=32768),
        # The prompt of the synthetic decoder at its named length.
        dict(name="prefill_2048", kind="prefill", tokens=2048),
        # One step of 64 constrained sequences over contexts of 32 to 2048 positions.
        dict(name="decode_b64", kind="decode", batch=64, min_context=32, max_context=2048),
        # A tool prompt through the shipped archive's form, then the first tokens of the answer.
        dict(name="needle_cq4_p640", kind="needle", form="4", prompt=640, steps=2, sink=0),
        # Token-at-a-time decode after a short prompt (int8 weights).
        dict(name="needle_i8_s24", kind="needle", form="0", prompt=48, steps=24, sink=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["call", "matvec", "matvec", "matvec", "matmul", "attend", "select", "prefill",
                       "decode", "needle"])
    if kind == "call":
        k = 1 << rng.randint(7, 12)
        return dict(kind=kind, bits=rng.choice([0, 0, 2, 4]), n=_log(rng, 128, 8192), k=k,
                    g=rng.choice([32, k]) if k <= 2048 else 32, batch=1)
    if kind == "matvec":
        bits = rng.choice([0, 0, 2, 3, 4, 5])
        batch = rng.choice([1, _log(rng, 2, 64), _log(rng, 8, 300)])
        if bits:
            k, g = _log(rng, 256, 4096), rng.choice([32, 32, 64, 128])
        else:
            k, g = 1 << rng.randint(9, 12), rng.choice([32, 32, 64, 128])
        n = _log(rng, 256, 16384)
        return dict(kind=kind, bits=bits, n=min(n, 1 + (1 << 30) // (k * batch)), k=k, g=g, batch=batch)
    if kind == "matmul":
        return dict(kind=kind, n=_log(rng, 256, 4096), k=1 << rng.randint(7, 11),
                    rows=_log(rng, 16, 2048))
    if kind == "attend":
        window = rng.choice([0, 0, 256])
        return dict(kind=kind, layers=rng.randint(2, 8), kv_heads=rng.choice([2, 4, 8]),
                    rep=rng.choice([1, 1, 2, 4]), length=_log(rng, 64, 8192), window=window,
                    sink=rng.choice([0, 3]) if window else 0,
                    mode=rng.choice(["int8", "int8", "int8", "float32"]))
    if kind == "select":
        return dict(kind=kind, batch=_log(rng, 1, 64), vocab=_log(rng, 2000, 40000))
    if kind == "prefill":
        return dict(kind=kind, tokens=_log(rng, 64, 2048))
    if kind == "decode":
        return dict(kind=kind, batch=_log(rng, 2, 64), min_context=32,
                    max_context=_log(rng, 128, 2048))
    return dict(kind=kind, form=rng.choice(["0", "4", "4", "2", "mixed"]),
                prompt=_log(rng, 8, 640), steps=rng.randint(1, 8), sink=rng.choice([0, 3]))


# ------------------------------------------------------------------ shared program state

_cache: dict = {}


def _once(key, make):
    if key not in _cache:
        _cache[key] = make()
    return _cache[key]


def _backend() -> HipBackend:
    return _once("backend", lambda: HipBackend(device=0))


def _rng(*key) -> np.random.Generator:
    return np.random.default_rng([2026, *key])


def _int8_matrix(n, k, g, *key) -> Int8Matrix:
    r = _rng(n, k, g, *key)
    return Int8Matrix(r.integers(-127, 128, (n, k), dtype=np.int8),
                      r.uniform(0.001, 0.02, (n, k // g)).astype(np.float32), g)


def _cq_matrix(n, k, g, bits) -> CqMatrix:
    r = _rng(n, k, g, bits)
    kpad = -(-k // g) * g
    if bits == 5:
        codes = np.array([0, 1, 3])[r.integers(0, 3, (n, kpad))]
    else:
        codes = r.integers(0, 1 << bits, (n, kpad))
    cb = synth.cq_codebook()
    books = {2: cb[0:4], 3: cb[4:12], 4: cb[12:28]}
    norms = r.uniform(0.01, 0.05, (n, kpad // g)).astype(np.float16).view(np.uint16)
    m = CqMatrix(pack_codes(codes, bits), norms, books, n, k, g, bits)
    m.codes = codes.astype(np.int8)  # for exact() only
    return m


def _matrix(case):
    n, k, g, bits = (case[f] for f in ("n", "k", "g", "bits"))
    return _once(("mat", n, k, g, bits), lambda: _cq_matrix(n, k, g, bits) if bits
                 else _int8_matrix(n, k, g))


class _DecoderWeights:
    """The synthetic 8-layer decoder's weights, in the attributes HipDecoder reads."""

    def __init__(self):
        g = self.geometry = DecoderGeometry()
        qr, kr = g.heads * HD, g.kv_heads * HD

        def mats(role, n, k):
            return [_int8_matrix(n, k, k, role, layer) for layer in range(g.layers)]

        self.embedding = _int8_matrix(g.vocab, g.dim, g.dim, 99)
        self.wq, self.wk, self.wv = mats(1, qr, g.dim), mats(2, kr, g.dim), mats(3, kr, g.dim)
        self.wo = mats(4, g.dim, qr)
        self.wup, self.wdown = mats(5, g.ffn, g.dim), mats(6, g.dim, g.ffn)
        r = _rng(7)

        def vec(*shape):
            return r.uniform(-0.1, 0.1, shape).astype(np.float32)

        self.attn_norm, self.ffn_norm = vec(g.layers, g.dim), vec(g.layers, g.dim)
        self.q_norm, self.k_norm = vec(g.layers, HD), vec(g.layers, HD)
        self.final_norm = vec(g.dim)


def _decoder() -> HipDecoder:
    return _once("decoder", lambda: HipDecoder(_backend(), _DecoderWeights()))


def _needle(form: str):
    def make():
        bits = form if form == "mixed" else int(form)
        weights = Needle2Weights(Needle2Geometry(), 2026, cq_bits=bits)
        return NeedleModel(_backend(), weights).create_resident_runtime()

    return _once(("needle", form), make)


class _Hbm:
    """A view of a cache's device memory for torch.as_tensor, which keeps this object (and with it
    the cache) for as long as the tensor lives."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr,
                                         "version": 2, "strides": None}


class _Cache(HipKvCache):
    """A cache given back when nothing refers to it any more."""

    def __del__(self):
        if getattr(self, "handle", None) is not None:
            self.free()


def _kv_views(cache: _Cache):
    """The cache's arrays in HBM as tensors: K and V codes, K and V scales."""
    alloc, kc, vc, ks, vs = C.c_uint32(), C.c_void_p(), C.c_void_p(), C.c_void_p(), C.c_void_p()
    cache.lib.nd_kv_info(cache.handle, C.byref(alloc), C.byref(kc), C.byref(vc), C.byref(ks),
                         C.byref(vs))
    rows = (cache.layers, cache.kv_heads, cache.alloc)
    codes = "|i1" if cache.mode == 0 else "<f4"
    views = [_Hbm(cache, kc.value, rows + (HD,), codes), _Hbm(cache, vc.value, rows + (HD,), codes)]
    if cache.mode == 0:
        views += [_Hbm(cache, ks.value, rows, "<f4"), _Hbm(cache, vs.value, rows, "<f4")]
    return [torch.as_tensor(v, device=DEVICE) for v in views]


_recent: collections.deque = collections.deque(maxlen=8)


class _State:
    """What the program holds.  Batches and prompt sessions go back with the state; the last
    states are kept, so that outputs in their caches outlive the call that made them."""

    def __init__(self, case, **held):
        self.case = case
        self.__dict__.update(held)
        _recent.append(self)

    def __del__(self):
        for owned in ("batch", "prefill"):
            if hasattr(self, owned):
                getattr(self, owned).free()


def _normal(seed, shape, salt=0):
    r = torch.Generator(device=DEVICE).manual_seed(1000003 * salt + seed)
    return torch.randn(shape, generator=r, device=DEVICE, dtype=torch.float32)


# ------------------------------------------------------------------------------ prepare

def prepare(case, seed):
    hip, kind = _backend(), case["kind"]
    if kind == "call":
        m = _matrix(case)
        hip.upload(m)
        return _State(case, hip=hip, matrix=m, x=_normal(seed, case["k"]).cpu().numpy())
    if kind == "matvec":
        return _State(case, hip=hip, handle=hip.upload(_matrix(case)),
                      x=_normal(seed, (case["batch"], case["k"])),
                      y=torch.empty((case["batch"], case["n"]), device=DEVICE))
    if kind == "matmul":
        m = _once(("mm", case["n"], case["k"]),
                  lambda: _int8_matrix(case["n"], case["k"], case["k"], 3))
        return _State(case, hip=hip, handle=hip.upload(m), x=_normal(seed, (case["rows"], case["k"])),
                      y=torch.empty((case["rows"], case["n"]), device=DEVICE))
    if kind == "attend":
        cache = _Cache(hip, case["layers"], case["kv_heads"], case["length"], case["sink"],
                           case["window"], case["mode"])
        rows = (case["length"], case["kv_heads"], HD)
        new = []
        for layer in range(case["layers"]):
            k, v = _normal(seed, rows, 2 * layer + 1), _normal(seed, rows, 2 * layer + 2)
            torch.cuda.synchronize()
            hip._check(hip.lib.nd_kv_store_d(hip.ctx, cache.handle, layer, 0, case["length"],
                                             k.data_ptr(), v.data_ptr(), None))
            hip._check(hip.lib.nd_sync(hip.ctx))
            new.append((k[-1].clone(), v[-1].clone()))  # the token's own K and V
        q = _normal(seed, (case["layers"], case["kv_heads"] * case["rep"] * HD), 99)
        return _State(case, hip=hip, cache=cache, new=new, q=q, out=torch.empty_like(q),
                      views=_kv_views(cache))
    if kind == "select":
        b, v = case["batch"], case["vocab"]
        words = (v + 31) // 32
        allowed = _normal(seed, (b, words * 32), 5) < -2.0537  # about 2% of the ids
        allowed[:, v:] = False
        allowed[torch.arange(b), torch.randint(0, v, (b,), generator=torch.Generator().manual_seed(
            seed))] = True
        bits = (allowed.view(b, words, 32).long() << torch.arange(32, device=DEVICE)).sum(-1)
        mask = torch.where(bits >= 1 << 31, bits - (1 << 32), bits).to(torch.int32)
        return _State(case, hip=hip, logits=_normal(seed, (b, v)) * 20, mask=mask,
                      ids=torch.empty(b, dtype=torch.int32, device=DEVICE),
                      lps=torch.empty(b, dtype=torch.float64, device=DEVICE))
    if kind == "prefill":
        n, dec = case["tokens"], _decoder()
        g = dec.geometry
        cache = _Cache(hip, g.layers, g.kv_heads, n)
        return _State(case, prefill=HipPrefill(dec, n, n), cache=cache, views=_kv_views(cache),
                      prompt=_rng(seed, 11).integers(0, g.vocab, n).astype(np.uint32))
    if kind == "decode":
        dec, b, r = _decoder(), case["batch"], _rng(seed, 12)
        lengths = r.integers(case["min_context"], case["max_context"] + 1, b).astype(np.uint32)
        batch = HipBatch(dec, b, case["max_context"] + 8)
        for s in range(b):
            sk, sv = (int(z) for z in r.integers(0, 1 << 62, 2))
            batch.fill_synthetic(s, sk, sv, int(lengths[s]), batch.max_length, *PREFIX_SCALE)
        pin = dict(pin_memory=True)
        return _State(case, hip=hip, batch=batch, lengths=lengths, mask_seed=seed,
                      start=r.integers(0, dec.geometry.vocab, b).astype(np.uint32),
                      tokens=torch.empty(b, dtype=torch.int32, **pin),
                      positions=torch.empty(b, dtype=torch.int32, **pin),
                      lps=torch.empty(b, dtype=torch.float64, **pin),
                      logits=torch.empty((b, dec.geometry.vocab), **pin))
    runtime = _needle(case["form"])
    ids = _rng(seed, 13).integers(0, 8192, case["prompt"] + case["steps"]).astype(np.uint32)
    return _State(case, runtime=runtime, prompt=ids[:case["prompt"]], tokens=ids[case["prompt"]:])


# ---------------------------------------------------------------------------------- run

def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "call":
        return s.hip.matvec(s.matrix, s.x)
    if kind == "matvec":
        s.hip._check(s.hip.lib.nd_matvec_d(s.hip.ctx, s.handle, s.x.data_ptr(), case["batch"], 0,
                                           case["n"], s.y.data_ptr(), None))
        return s.y
    if kind == "matmul":
        s.hip._check(s.hip.lib.nd_matmul_d(s.hip.ctx, s.handle, s.x.data_ptr(), case["rows"],
                                           s.y.data_ptr(), 0, None))
        return s.y
    if kind == "attend":
        lib, ctx, kv = s.hip.lib, s.hip.ctx, s.cache.handle
        at = case["length"] - 1
        for layer, (k, v) in enumerate(s.new):
            s.hip._check(lib.nd_kv_store_d(ctx, kv, layer, at, 1, k.data_ptr(), v.data_ptr(), None))
            s.hip._check(lib.nd_attention_d(ctx, kv, layer, at, s.q[layer].data_ptr(),
                                            case["kv_heads"] * case["rep"], s.out[layer].data_ptr(),
                                            None))
        return [s.out, *s.views]
    if kind == "select":
        s.hip._check(s.hip.lib.nd_select_mask_d(s.hip.ctx, s.logits.data_ptr(), case["batch"],
                                                case["vocab"], s.mask.data_ptr(), s.ids.data_ptr(),
                                                s.lps.data_ptr(), None))
        return [s.ids, s.lps]
    if kind == "prefill":
        return [s.prefill.run(s.cache, s.prompt), *s.views]
    if kind == "decode":
        s.batch.set_state(s.start, s.lengths, 0)
        s.batch.step(int(s.lengths.max()), mask_seed=s.mask_seed)
        s.hip._check(s.hip.lib.nd_batch_read(s.hip.ctx, s.batch.handle, s.tokens.data_ptr(),
                                             s.positions.data_ptr(), s.lps.data_ptr(),
                                             s.logits.data_ptr()))
        return [s.tokens, s.positions, s.lps, s.logits]
    s.runtime.reset(len(s.prompt) + len(s.tokens) + 1, case["sink"])
    logits = [s.runtime.prefill(s.prompt)]
    logits += [s.runtime.step(int(t)) for t in s.tokens]
    return logits


# ------------------------------------------------------------------- what a pass has to do

def _matrix_bytes(case):
    n, k, g, bits = (case[f] for f in ("n", "k", "g", "bits"))
    if not bits:
        return n * k + n * (k // g) * 4
    kpad = -(-k // g) * g
    return n * kpad * (2 if bits == 5 else bits) // 8 + n * (kpad // g) * 2


def _visible(case):
    if not case["window"]:
        return case["length"]
    return min(case["length"], case["sink"] + case["window"])


def work(case):
    kind = case["kind"]
    if kind in ("call", "matvec"):
        n, k, b = case["n"], case["k"], case["batch"]
        return {"bytes": _matrix_bytes(case) + 4 * b * (n + k), "flops": 2 * n * k * b}
    if kind == "matmul":
        n, k, m = case["n"], case["k"], case["rows"]
        return {"bytes": n * (k + 4) + 4 * m * (n + k), "flops": 2 * n * k * m}
    if kind == "attend":
        per = 2 * HD + 8 if case["mode"] == "int8" else 8 * HD
        heads, seen = case["kv_heads"], _visible(case)
        q = heads * case["rep"] * HD
        return {"bytes": case["layers"] * (heads * (seen * per + 8 * HD) + 8 * q),
                "flops": case["layers"] * 4 * q * seen}
    if kind == "select":
        b, v = case["batch"], case["vocab"]
        return {"bytes": b * (4 * v + v // 8 + 12), "flops": 4 * b * v}
    if kind in ("prefill", "decode"):
        g = DecoderGeometry()
        rows = (g.heads + 2 * g.kv_heads) * HD
        layer = rows * g.dim + g.dim * g.dim + 2 * g.ffn * g.dim
        weights = g.layers * (layer + 4 * (rows + 2 * g.dim + g.ffn)) + g.vocab * (g.dim + 4)
        if kind == "prefill":
            m = case["tokens"]
            return {"bytes": weights + m * g.layers * g.kv_heads * (2 * HD + 8) + 4 * g.vocab,
                    "flops": g.layers * (2 * m * layer + 2 * g.heads * HD * m * (m + 1))
                    + 2 * g.vocab * g.dim}
        b = case["batch"]
        seen = b * (case["min_context"] + case["max_context"]) / 2
        return {"bytes": weights + seen * g.layers * g.kv_heads * (2 * HD + 8) + b * g.vocab * 4.125,
                "flops": 2 * b * (g.layers * layer + g.vocab * g.dim)
                + seen * g.layers * g.heads * HD * 4}
    g = Needle2Geometry()
    rows = (2 * g.heads + 2 * g.kv_heads) * HD
    mix = (2 * g.lanes + g.lanes * g.lanes) * g.lanes * g.dim
    layer = rows * g.dim + g.dim * g.heads * HD + mix
    engram = len(g.sites) * 2 * g.dim * g.engram_tables * g.engram_sub
    head = g.vocab * g.dim
    per = {"0": 1.0, "2": 0.3125, "4": 0.5625, "mixed": 0.4}[case["form"]]  # bytes a weight
    p, n = case["prompt"], case["steps"]

    def cache(m):  # positions read by a token that sees m of them
        return min(m, g.kv_window + case["sink"])

    steps = sum(cache(p + i + 1) for i in range(n))
    prompt = sum(cache(i + 1) for i in range(p))
    kv = g.layers * g.kv_heads * (2 * HD + 8)
    weights = per * (g.layers * layer + engram + head)
    return {"bytes": (1 + n) * (weights + 4 * g.vocab) + kv * (p + steps),
            "flops": 2 * (p + n) * (g.layers * layer + engram) + 2 * (1 + n) * head
            + 4 * g.layers * g.heads * HD * (steps + prompt)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("call", "matvec", "matmul"):
        return {"rel": 2e-6, "max": 1e-4}  # 32-bit sums of up to 4096 products (seen: 3e-7)
    if kind == "attend":  # fp32 softmax sums; codes and scales are the quantizer's, bit for bit
        return {"rel": 2.5e-5, "max": 1e-3}  # seen: 6e-6 at 8192 positions
    if kind == "select":  # ids are exact; the log-sum-exp is taken in 64 bits
        return {"rel": 1e-12, "max": 1e-11}
    # Whole models: a K or V element within rounding of a half-integer takes the neighbouring
    # code, which later layers and positions see (one code of 127 steps).
    return {"rel": 2e-3, "max": 5e-2, "differ": 5e-3}


# -------------------------------------------------------------------------------- exact

def _hadamard_rows(x, g):
    """Walsh-Hadamard transform of every group of g columns (natural order)."""
    h = torch.ones((1, 1), dtype=torch.float64, device=x.device)
    while h.shape[0] < g:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.view(x.shape[0], -1, g) @ h).reshape(x.shape)


def _exact_product(m, x):
    x = x.double()
    if getattr(m, "kind", None) == "cq":
        pad, g = m.input_size_padded, m.group_size
        x = torch.nn.functional.pad(x, (0, pad - m.input_size))
        x = _hadamard_rows(x, g)
        if m.bits == 5:
            levels = np.array([0.0, 1.2240064, 0.0, -1.2240064]) / math.sqrt(g)
        else:
            levels = np.asarray(m.codebook, np.float64)
        x = x / math.sqrt(g)
        w = torch.from_numpy(levels).to(DEVICE)[torch.from_numpy(m.codes).to(DEVICE).long()]
        norms = torch.from_numpy(m.norms.view(np.float16).astype(np.float64)).to(DEVICE)
        w = w * norms.repeat_interleave(g, 1)
    else:
        w = torch.from_numpy(m.codes).to(DEVICE).double()
        w = w * torch.from_numpy(m.scales).to(DEVICE).double().repeat_interleave(m.group_size, 1)
    return x @ w.t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "call":
        return _exact_product(_matrix(case), _normal(seed, case["k"])[None])[0].cpu().numpy()
    if kind == "matvec":
        return _exact_product(_matrix(case), _normal(seed, (case["batch"], case["k"])))
    if kind == "matmul":
        m = _once(("mm", case["n"], case["k"]),
                  lambda: _int8_matrix(case["n"], case["k"], case["k"], 3))
        return _exact_product(m, _normal(seed, (case["rows"], case["k"])))
    if kind == "attend":
        rows = (case["length"], case["kv_heads"], HD)
        heads, rep = case["kv_heads"], case["rep"]
        at = case["length"] - 1
        first = 0 if not case["window"] else max(0, at + 1 - case["window"])
        seen = torch.tensor([p for p in range(at + 1) if p >= first or p < case["sink"]])
        outs = []

        def dequantized(x):
            x = x.double()[seen.to(DEVICE)]
            if case["mode"] != "int8":
                return x
            s = x.abs().amax(-1, keepdim=True).clamp_min(1e-12) / 127
            return torch.round(x / s) * s.float().double()  # half to even, scales stored in 32 bits

        for layer in range(case["layers"]):
            k = dequantized(_normal(seed, rows, 2 * layer + 1)).transpose(0, 1)
            v = dequantized(_normal(seed, rows, 2 * layer + 2)).transpose(0, 1)
            q = _normal(seed, (case["layers"], heads * rep * HD), 99)[layer].double()
            q = q.view(heads, rep, HD)
            p = torch.softmax((q[:, :, None] * k[:, None]).sum(-1) / 8, -1)
            outs.append((p[..., None] * v[:, None]).sum(2).reshape(-1))
        return [torch.stack(outs)] + [None] * (4 if case["mode"] == "int8" else 2)
    if kind == "select":
        s = prepare(case, seed)
        bits = (s.mask.long()[:, :, None] >> torch.arange(32, device=DEVICE)) & 1
        allowed = bits.reshape(case["batch"], -1)[:, :case["vocab"]].bool()
        ids = s.logits.masked_fill(~allowed, -math.inf).argmax(-1)
        lps = torch.log_softmax(s.logits.double(), -1).gather(1, ids[:, None])[:, 0]
        return [ids.int(), lps]
    # Whole models quantize their cache between layers: a pass in 64 bits takes other codes at the
    # rounding boundaries, so its logits are no nearer the quantized model's own.
    return None


assert MASK_P == 0.02  # the batched step's masks have the selection case's density
