"""The work that a user of juno_amd has it do, as measurable cases.

Every case is one block of a Llama-style model on packed GGUF weights (or a
whole call of the decoder or the batch pipeline), at the shapes of the three
models this repository is benchmarked on: TinyLlama-1.1B, Llama-3-8B and
Phi-3-mini.  ``listed`` names twelve of them, ``draw`` gives others of the same
ranges.  The kinds:

  host     one host-pointer matVec, HipMatVec.sgemv_quant: Juno's own interface,
           a host float[] in and a host float[] out per call
  proj     one projection on device vectors, HipMatVec.sgemv_dev, for a batch
  qkv      residual add + rmsNorm + the [q, k, v] projections, as LlamaDecoder
           (one request) and LlamaBatchPipeline (several) issue them
  mlp      residual add + rmsNorm + [gate, up] + SwiGLU + down, likewise
  head     the final norm and the output projection, likewise
  attn     rope + KV append + grouped-query attention + output projection
  merge    a LoRA merge of one matrix: dequantize, add the delta, requantize
  step     LlamaDecoder: one decode step from a token, its captured graph
           replayed
  serve    LlamaBatchPipeline.forward_batch: tokens in, host logits out

Weights are packed blocks drawn from the seed with the quants, scales and
minima that weights of N(0, 0.02) have; activations are N(0, 1) with a few
strong channels; caches hold N(0, 1) keys and values.  ``exact`` unpacks the
same bytes and computes in 64 bits with plain torch.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from juno_amd import _lib
from juno_amd import matvec as mv
from juno_amd.decode import LlamaConfig, LlamaDecoder, LlamaLayerWeights, LlamaWeights
from juno_amd.pipeline import LlamaBatchPipeline

TYPES = {"q8_0": 8, "q2_k": 10, "q3_k": 11, "q4_k": 12, "q5_k": 13, "q6_k": 14}
BLOCK = {"q8_0": (32, 34), "q2_k": (256, 84), "q3_k": (256, 110), "q4_k": (256, 144), "q5_k": (256, 176),
         "q6_k": (256, 210)}
# a model file's quantization: the type of most matrices, and of attn_v, ffn_down and the output projection
MIX = {"q4_k_m": ("q4_k", "q6_k"), "q5_k_m": ("q5_k", "q6_k"), "q8_0": ("q8_0", "q8_0"), "q6_k": ("q6_k", "q6_k"),
       "q3_k": ("q3_k", "q3_k"), "q2_k": ("q2_k", "q3_k")}
EPS, STD = 1e-5, 0.02
# hidden, ffn, heads, kv heads, head_dim, vocab, rope theta
TINYLLAMA = dict(hidden=2048, ffn=5632, heads=32, kv=4, hd=64, vocab=32000, theta=10000.0)
LLAMA8B = dict(hidden=4096, ffn=14336, heads=32, kv=8, hd=128, vocab=128256, theta=500000.0)
PHI3 = dict(hidden=3072, ffn=8192, heads=32, kv=32, hd=96, vocab=32064, theta=10000.0)


def listed():
    m8, mt, mp = LLAMA8B, TINYLLAMA, PHI3
    return [
        # the smallest call: a k projection through Juno's host interface; latency and copies
        {"name": "host-k-tinyllama", "kind": "host", "type": "q4_k", "rows": 256, "cols": 2048, "row0": 0},
        # one request's attention input of an 8B layer: three small matrices of two formats in one launch
        {"name": "qkv-8b-b1", "kind": "qkv", "mix": "q4_k_m", "hidden": m8["hidden"], "kvdim": 1024, "batch": 1},
        # one request's feed-forward of an 8B layer: most of a decode step's bytes
        {"name": "mlp-8b-b1", "kind": "mlp", "mix": "q4_k_m", "hidden": m8["hidden"], "ffn": m8["ffn"], "batch": 1},
        # two requests on the fused QKV of a Phi-3 file in Q8_0
        {"name": "proj-phi3-qkv-b2", "kind": "proj", "type": "q8_0", "rows": 9216, "cols": mp["hidden"], "row0": 0,
         "batch": 2},
        # a serving node's feed-forward at a ragged batch of requests
        {"name": "mlp-8b-b20", "kind": "mlp", "mix": "q4_k_m", "hidden": m8["hidden"], "ffn": m8["ffn"], "batch": 20},
        # the same at a full node: more requests than one tile of columns
        {"name": "mlp-8b-b128", "kind": "mlp", "mix": "q4_k_m", "hidden": m8["hidden"], "ffn": m8["ffn"],
         "batch": 128},
        # the output projection for a few requests: the largest matrix of the model
        {"name": "head-8b-b8", "kind": "head", "type": "q6_k", "hidden": m8["hidden"], "vocab": m8["vocab"],
         "batch": 8},
        # one request far into a long context
        {"name": "attn-8b-b1-long", "kind": "attn", "type": "q4_k", "heads": 32, "kv": 8, "hd": 128,
         "theta": m8["theta"], "batch": 1, "ctx": 4000, "max_seq": 4096},
        # a batch of requests at positions of their own
        {"name": "attn-8b-b32", "kind": "attn", "type": "q4_k", "heads": 32, "kv": 8, "hd": 128, "theta": m8["theta"],
         "batch": 32, "ctx": 900, "max_seq": 1024},
        # merging an adapter into an attention matrix of an 8B file
        {"name": "merge-8b-q", "kind": "merge", "type": "q4_k", "rows": m8["hidden"], "cols": m8["hidden"]},
        # a whole decode step, one request, 512 positions of context
        {"name": "step-tinyllama", "kind": "step", "mix": "q4_k_m", "layers": 22, "pos": 511, "max_seq": 512,
         "batch": 1},
        # a whole serving call: tokens in, logits on the host
        {"name": "serve-tinyllama-b24", "kind": "serve", "mix": "q4_k_m", "layers": 22, "pos": 400, "max_seq": 512,
         "batch": 24},
    ]


def _log_int(rng, lo, hi, step=1):
    """A multiple of step in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step * ((lo + step - 1) // step), step * int(v / step))


def draw(rng):
    kind = rng.choice(["host", "proj", "proj", "qkv", "mlp", "mlp", "head", "attn", "attn", "merge"])
    typ = rng.choice(["q4_k", "q4_k", "q6_k", "q8_0", "q5_k", "q3_k", "q2_k"])
    mix = rng.choice(["q4_k_m", "q4_k_m", "q4_k_m", "q8_0", "q5_k_m", "q6_k", "q3_k", "q2_k"])
    batch = _log_int(rng, 1, 128)
    if kind in ("host", "proj"):
        # any rows of any matrix, row ranges among them (the fused QKV of a Phi-3 file); K-quant columns come in
        # blocks of 256, Q8_0 columns in blocks of 32
        c = {"kind": kind, "type": typ, "rows": _log_int(rng, 250, 20000),
             "cols": _log_int(rng, 512, 14336, 32 if typ == "q8_0" and rng.random() < 0.3 else 256),
             "row0": rng.choice([0, 0, 0, rng.randrange(1, 700)])}
        return c if kind == "host" else dict(c, batch=batch)
    if kind == "qkv":
        hidden = _log_int(rng, 1024, 8192, 256)
        return {"kind": kind, "mix": mix, "hidden": hidden, "kvdim": hidden // rng.choice([1, 4, 8]), "batch": batch}
    if kind == "mlp":
        return {"kind": kind, "mix": mix, "hidden": _log_int(rng, 1024, 4096, 256),
                "ffn": _log_int(rng, 2560, 14336, 256), "batch": batch}
    if kind == "head":
        hidden = rng.choice([2048, 3072, 4096])
        return {"kind": kind, "type": rng.choice(["q6_k", "q6_k", "q8_0", "q4_k"]), "hidden": hidden,
                "vocab": _log_int(rng, 32000, 128256), "batch": _log_int(rng, 1, 32)}
    if kind == "attn":
        m = rng.choice([LLAMA8B, LLAMA8B, TINYLLAMA, PHI3])
        batch = rng.choice([1, _log_int(rng, 1, 64)])
        # positions: all of a batch's KV within 32768 positions of an 8B layer
        most = min(8192, 32768 * 1024 // (batch * m["kv"] * m["hd"]))
        ctx = _log_int(rng, 20, most)
        return {"kind": kind, "type": rng.choice(["q4_k", "q4_k", "q6_k", "q8_0"]), "heads": m["heads"], "kv": m["kv"],
                "hd": m["hd"], "theta": m["theta"], "batch": batch, "ctx": ctx,
                "max_seq": min(max(512, 2 * ctx), 8192)}
    return {"kind": kind, "type": rng.choice(["q4_k", "q4_k", "q6_k", "q8_0", "q5_k"]),
            "rows": _log_int(rng, 256, 14336), "cols": _log_int(rng, 1024, 8192, 256)}


# ------------------------------------------------------------------ packed weights from a seed
def _f16(v):
    """fp16 bytes [..., 2] of a float tensor."""
    return v.to(torch.float16).contiguous().view(torch.uint8).reshape(*v.shape, 2)


def _quants(g, n, per, mean, std, hi):
    q = torch.empty(n, per, device="cuda").normal_(mean, std, generator=g)
    return q.round_().clamp_(0, hi).to(torch.uint8)


def _packed(g, typ, rows, cols):
    """Packed bytes [blocks, block_bytes] of a matrix of that type, on the GPU."""
    qk, _ = BLOCK[typ]
    n = rows * cols // qk
    u = lambda *s: torch.rand(*s, device="cuda", generator=g)  # noqa: E731
    ints = lambda lo, hi, *s: torch.randint(lo, hi, s, device="cuda", generator=g, dtype=torch.int32)  # noqa: E731
    b8 = lambda v: v.to(torch.uint8)  # noqa: E731
    jitter = 0.8 + 0.4 * u(n)
    if typ == "q8_0":
        q = torch.empty(n, 32, device="cuda").normal_(0, 42.0, generator=g).round_().clamp_(-127, 127)
        return torch.cat([_f16(STD / 42.0 * jitter), q.to(torch.int8).view(torch.uint8)], 1)
    if typ in ("q4_k", "q5_k"):
        top = 15 if typ == "q4_k" else 31
        ls = ints(36, 64, n, 8)
        lm = (ls + ints(-3, 4, n, 8)).clamp_(0, 63)
        step = 4.0 * STD / top / 50.0 * jitter  # d: one quant step over a scale of about 50
        sc = torch.cat([(ls[:, :4] | ((ls[:, 4:] & 0x30) << 2)), (lm[:, :4] | ((lm[:, 4:] & 0x30) << 2)),
                        ((ls[:, 4:] & 15) | ((lm[:, 4:] & 15) << 4))], 1)
        q = _quants(g, n, 256, top / 2.0, top / 4.0, top).view(n, 4, 2, 32)
        parts = [_f16(step), _f16(step * (top / 2.0)), b8(sc)]
        if typ == "q5_k":
            bit = (q >> 4).view(n, 8, 32)
            qh = bit[:, 0].clone()
            for j in range(1, 8):
                qh |= bit[:, j] << j
            parts.append(qh)
        parts.append(((q[:, :, 0] & 15) | ((q[:, :, 1] & 15) << 4)).reshape(n, 128))
        return torch.cat(parts, 1)
    if typ == "q6_k":
        q = _quants(g, n, 256, 32.0, 10.0, 63).view(n, 2, 4, 32)
        ql = ((q[:, :, :2] & 15) | ((q[:, :, 2:] & 15) << 4)).reshape(n, 128)
        qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
        sc = ints(60, 128, n, 16) * (1 - 2 * ints(0, 2, n, 16))
        return torch.cat([ql, qh.reshape(n, 64), sc.to(torch.int8).view(torch.uint8), _f16(STD / 950.0 * jitter)], 1)
    if typ == "q3_k":
        q = _quants(g, n, 256, 4.0, 1.6, 7).view(n, 2, 4, 2, 16)  # half, 32-column group j, sub-block r, column
        low = q & 3
        qs = low[:, :, 0] | (low[:, :, 1] << 2) | (low[:, :, 2] << 4) | (low[:, :, 3] << 6)
        hi = (q >> 2).view(n, 8, 32)
        hm = hi[:, 0].clone()
        for j in range(1, 8):
            hm |= hi[:, j] << j
        top = 3 * ints(0, 2, n, 4, 4)  # the scales' two high bits: -32..-17 or 16..31
        sc = torch.cat([ints(0, 256, n, 8), top[..., 0] | (top[..., 1] << 2) | (top[..., 2] << 4) | (top[..., 3] << 6)],
                       1)
        return torch.cat([hm, qs.reshape(n, 64), b8(sc), _f16(STD / 40.0 * jitter)], 1)
    assert typ == "q2_k", typ
    q = _quants(g, n, 256, 1.5, 1.0, 3).view(n, 2, 4, 2, 16)
    qs = q[:, :, 0] | (q[:, :, 1] << 2) | (q[:, :, 2] << 4) | (q[:, :, 3] << 6)
    s = ints(8, 16, n, 16)
    sc = s | ((s + ints(-1, 2, n, 16)).clamp_(0, 15) << 4)
    return torch.cat([b8(sc), qs.reshape(n, 64), _f16(STD / 12.0 * jitter), _f16(1.5 * STD / 12.0 * jitter)], 1)


def _half(b):
    return b.contiguous().view(torch.float16).to(torch.float64)


def _unpack(b, typ, rows, cols):
    """The 64-bit weights [rows, cols] that packed bytes mean (the GGUF block layouts)."""
    n = b.shape[0]
    i64 = lambda v: v.to(torch.int16)  # noqa: E731
    if typ == "q8_0":
        w = _half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif typ in ("q4_k", "q5_k"):
        d, dm = _half(b[:, :2]), _half(b[:, 2:4])
        s = i64(b[:, 4:16])
        ls = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] & 0xC0) >> 2)], 1)
        lm = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] & 0xC0) >> 2)], 1)
        qs = b[:, -128:].view(n, 4, 1, 32)
        q = i64(torch.cat([qs & 15, qs >> 4], 2).view(n, 8, 32))
        if typ == "q5_k":
            qh = b[:, 16:48].view(n, 1, 32)
            sh = torch.arange(8, device=b.device, dtype=torch.uint8).view(1, 8, 1)
            q = q | (i64((qh >> sh) & 1) << 4)
        w = (d * ls.double()).unsqueeze(2) * q.double() - (dm * lm.double()).unsqueeze(2)
    elif typ == "q6_k":
        ql, qh = i64(b[:, :128]).view(n, 2, 2, 32), i64(b[:, 128:192]).view(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int16).view(1, 1, 4, 1)
        q = (lo | (((qh >> sh) & 3) << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _half(b[:, 208:210])
        w = q.view(n, 16, 16).double() * sc.unsqueeze(2)
    elif typ == "q3_k":
        sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int16).view(1, 1, 4, 1)
        low = (i64(b[:, 32:96]).view(n, 2, 1, 32) >> sh) & 3
        bit = torch.arange(8, device=b.device, dtype=torch.int16).view(1, 8, 1)
        hi = ((i64(b[:, :32]).view(n, 1, 32) >> bit) & 1).view(n, 2, 4, 32)
        q = (low | (hi << 2)) - 4
        s = i64(b[:, 96:108])
        lo4 = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
        hi2 = torch.cat([(s[:, 8:] >> (2 * k)) & 3 for k in range(4)], 1)
        sc = ((lo4 | (hi2 << 4)) - 32).double() * _half(b[:, 108:110])
        w = q.reshape(n, 16, 16).double() * sc.unsqueeze(2)
    else:
        sh = torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int16).view(1, 1, 4, 1)
        q = ((i64(b[:, 16:80]).view(n, 2, 1, 32) >> sh) & 3).reshape(n, 16, 16).double()
        s = i64(b[:, :16])
        w = q * (_half(b[:, 80:82]) * (s & 15).double()).unsqueeze(2) \
            - (_half(b[:, 82:84]) * (s >> 4).double()).unsqueeze(2)
    return w.reshape(rows, cols)


def _packed_size(typ, rows, cols):
    return rows * cols // BLOCK[typ][0] * BLOCK[typ][1]


class _Inputs:
    """A case's inputs, in the order the kinds ask for them: the same for prepare and for exact."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def vec(self, *shape):
        """Activations: N(0, 1), one channel in 256 stronger."""
        x = torch.empty(*shape, device="cuda").normal_(0, 1, generator=self.g)
        x[..., 17::256] *= 6.0
        return x

    def normal(self, *shape, std=1.0):
        return torch.empty(*shape, device="cuda").normal_(0, std, generator=self.g)

    def norm(self, n):
        return 1.0 + self.normal(n, std=0.1)

    def mat(self, typ, rows, cols):
        return _packed(self.g, typ, rows, cols), typ, rows, cols


def _upload(m):
    b, typ, rows, cols = m
    be = mv.GpuContext.shared(0).create_mat_vec()
    return be.upload_quant(TYPES[typ], rows, cols, b.cpu().numpy())


def _w64(m):
    b, typ, rows, cols = m
    return _unpack(b, typ, rows, cols)


def _qkv_mats(case):
    a, b = MIX[case["mix"]]
    return [(a, case["hidden"]), (a, case["kvdim"]), (b, case["kvdim"])]


# ------------------------------------------------------------------ inputs per kind
def _inputs(case, seed):
    """The kind's inputs as torch tensors on the GPU, by name."""
    i, k = _Inputs(seed), case["kind"]
    B = case.get("batch", 1)
    if k in ("host", "proj"):
        return {"x": i.vec(B, case["cols"]), "w": i.mat(case["type"], case["rows"] + case["row0"], case["cols"])}
    if k == "qkv":
        H = case["hidden"]
        return {"x": i.vec(B, H), "res": i.vec(B, H), "norm": i.norm(H),
                "mats": [i.mat(t, r, H) for t, r in _qkv_mats(case)]}
    if k == "mlp":
        H, F = case["hidden"], case["ffn"]
        a, b = MIX[case["mix"]]
        return {"x": i.vec(B, H), "res": i.vec(B, H), "norm": i.norm(H), "gate": i.mat(a, F, H), "up": i.mat(a, F, H),
                "down": i.mat(b, H, F)}
    if k == "head":
        H = case["hidden"]
        return {"x": i.vec(B, H), "res": i.vec(B, H), "norm": i.norm(H), "w": i.mat(case["type"], case["vocab"], H)}
    if k == "attn":
        D, KV = case["heads"] * case["hd"], case["kv"] * case["hd"]
        lo = max(0, case["ctx"] - 1 if B == 1 else case["ctx"] // 2)
        pos = torch.randint(lo, case["ctx"], (B,), device="cuda", generator=i.g, dtype=torch.int32)
        return {"q": i.normal(B, D), "k": i.normal(B, KV), "v": i.normal(B, KV), "pos": pos,
                "slot": torch.randperm(B, device="cuda", generator=i.g).to(torch.int32),
                "kc": i.normal(B, case["max_seq"], KV), "vc": i.normal(B, case["max_seq"], KV),
                "wo": i.mat(case["type"], D, D)}
    if k == "merge":
        return {"w": i.mat(case["type"], case["rows"], case["cols"]),
                "delta": i.normal(case["rows"], case["cols"], std=0.002)}
    m, (a, b) = TINYLLAMA, MIX[case["mix"]]
    H, F, KV = m["hidden"], m["ffn"], m["kv"] * m["hd"]
    layers = []
    for _ in range(case["layers"]):
        layers.append({"attn_norm": i.norm(H), "ffn_norm": i.norm(H), "q": i.mat(a, H, H), "k": i.mat(a, KV, H),
                       "v": i.mat(b, KV, H), "o": i.mat(a, H, H), "gate": i.mat(a, F, H), "up": i.mat(a, F, H),
                       "down": i.mat(b, H, F)})
    return {"layers": layers, "out_norm": i.norm(H), "out": i.mat(b, m["vocab"], H), "embd": i.mat("q6_k", m["vocab"], H),
            "tokens": torch.randint(0, m["vocab"], (B,), device="cuda", generator=i.g, dtype=torch.int32),
            "pos": case["pos"] - torch.randint(0, 1 if k == "step" else 100, (B,), device="cuda", generator=i.g,
                                               dtype=torch.int32),
            "kc": i.normal(case["layers"], B, case["max_seq"], KV, std=0.5),
            "vc": i.normal(case["layers"], B, case["max_seq"], KV, std=0.5)}


def _model(inp, case):
    """The uploaded weights of a step or serve case."""
    m = TINYLLAMA
    cfg = LlamaConfig(m["hidden"], case["layers"], m["heads"], m["kv"], m["hd"], m["ffn"], m["vocab"], EPS, m["theta"])
    layers = [LlamaLayerWeights(lw["attn_norm"], lw["ffn_norm"],
                                {n: _upload(lw[n]) for n in ("q", "k", "v", "o", "gate", "up", "down")})
              for lw in inp["layers"]]
    return LlamaWeights(cfg, layers, inp["out_norm"], _upload(inp["out"]), token_embd=_upload(inp["embd"]))


# ------------------------------------------------------------------ a user's program
_P = ctypes.c_void_p


def _ptr(t):
    return _P(t.data_ptr())


def _check(rc):
    if rc:
        raise RuntimeError(_lib.last_error())


def _ptrs(ts):
    return (_P * len(ts))(*[t.data_ptr() for t in ts])


def prepare(case, seed):
    k, B = case["kind"], case.get("batch", 1)
    inp = _inputs(case, seed)
    s = {"case": case, "B": B, "L": _lib.load(), "stream": _P(torch.cuda.current_stream().cuda_stream)}
    f = dict(device="cuda", dtype=torch.float32)
    if k == "host":
        s.update(be=mv.GpuContext.shared(0).create_mat_vec(), w=_upload(inp["w"]), x=inp["x"][0].cpu().numpy())
    elif k == "proj":
        s.update(be=mv.GpuContext.shared(0).create_mat_vec(), w=_upload(inp["w"]), x=inp["x"],
                 y=torch.empty(B, case["rows"], **f))
    elif k == "qkv":
        mats = [_upload(m) for m in inp["mats"]]
        ys = [torch.empty(B, m.rows, **f) for m in mats]
        s.update(x=inp["x"], res=inp["res"], norm=inp["norm"], mats=mats, ys=ys, x_out=torch.empty_like(inp["x"]),
                 xn=torch.empty_like(inp["x"]), hs=(_P * 3)(*[m.handle for m in mats]), yp=_ptrs(ys))
        s["xp"] = _ptrs([s["xn"]] * 3)
    elif k == "mlp":
        F = case["ffn"]
        s.update(x=inp["x"], res=inp["res"], norm=inp["norm"], gate=_upload(inp["gate"]), up=_upload(inp["up"]),
                 down=_upload(inp["down"]), x_out=torch.empty_like(inp["x"]), xn=torch.empty_like(inp["x"]),
                 g=torch.empty(B, F, **f), u=torch.empty(B, F, **f), hid=torch.empty(B, F, **f),
                 y=torch.empty(B, case["hidden"], **f))
        s.update(hs=(_P * 1)(s["down"].handle), xp=_ptrs([s["hid"]]), yp=_ptrs([s["y"]]))
    elif k == "head":
        s.update(x=inp["x"], res=inp["res"], norm=inp["norm"], w=_upload(inp["w"]), x_out=torch.empty_like(inp["x"]),
                 xn=torch.empty_like(inp["x"]), y=torch.empty(B, case["vocab"], **f))
    elif k == "attn":
        s.update({n: inp[n] for n in ("q", "k", "v", "pos", "slot", "kc", "vc")}, wo=_upload(inp["wo"]),
                 att=torch.empty_like(inp["q"]), y=torch.empty_like(inp["q"]))
    elif k == "merge":
        b = inp["w"][0]
        s.update(be=mv.GpuContext.shared(0).create_mat_vec(), w=_upload(inp["w"]), delta=inp["delta"],
                 full=torch.empty_like(inp["delta"]), packed=torch.empty(b.numel(), device="cuda", dtype=torch.uint8))
    elif k == "step":
        dec = LlamaDecoder(_model(inp, case), case["max_seq"])
        dec.token.copy_(inp["tokens"])
        dec.pos.copy_(inp["pos"])
        torch.cuda.synchronize()
        graph = dec.capture(torch.cuda.Stream(), from_token=True)
        dec.k_cache.copy_(inp["kc"][:, 0])
        dec.v_cache.copy_(inp["vc"][:, 0])
        s.update(dec=dec, graph=graph, tokens=inp["tokens"], pos=inp["pos"])
    else:
        pipe = LlamaBatchPipeline(_model(inp, case), case["max_seq"], max_batch=B)
        s.update(pipe=pipe, ids=["r%d" % b for b in range(B)], tokens=[[int(t)] for t in inp["tokens"].tolist()],
                 pos=inp["pos"].tolist())
        pipe.forward_batch(s["ids"], s["tokens"], s["pos"])  # the requests take their cache slots, 0 first
        pipe.k_cache.copy_(inp["kc"])
        pipe.v_cache.copy_(inp["vc"])
    torch.cuda.synchronize()
    return s


def run(s):
    case, B, L, st = s["case"], s["B"], s["L"], s["stream"]
    k = case["kind"]
    if k == "host":
        return s["be"].sgemv_quant(s["w"], s["x"], case["row0"], case["row0"] + case["rows"])
    if k == "proj":
        s["be"].sgemv_dev(s["w"], s["x"].data_ptr(), s["y"].data_ptr(), case["row0"], case["row0"] + case["rows"],
                          st.value or 0, B)
        return s["y"]
    if k == "qkv":
        if B == 1:  # as LlamaDecoder
            _check(L.jh_rmsnorm_qmatvec_group_dev(3, s["hs"], _ptr(s["x"]), _ptr(s["res"]), _ptr(s["norm"]), EPS,
                                                  _ptr(s["x_out"]), _ptr(s["xn"]), s["yp"], st))
        else:  # as LlamaBatchPipeline
            _check(L.jh_rmsnorm_rows_dev(_ptr(s["x"]), _ptr(s["res"]), _ptr(s["norm"]), case["hidden"], B, EPS,
                                         _ptr(s["x_out"]), _ptr(s["xn"]), st))
            _check(L.jh_qmatvec_batched_group_dev(3, s["hs"], s["xp"], B, s["yp"], st))
        return [s["x_out"], *s["ys"]]
    if k == "mlp":
        if B == 1:
            _check(L.jh_rmsnorm_qmatvec_swiglu_dev(s["gate"].handle, s["up"].handle, _ptr(s["x"]), _ptr(s["res"]),
                                                   _ptr(s["norm"]), EPS, _ptr(s["x_out"]), _ptr(s["xn"]),
                                                   _ptr(s["hid"]), st))
            _check(L.jh_qmatvec_group_dev(1, s["hs"], s["xp"], s["yp"], st))
        else:
            _check(L.jh_rmsnorm_rows_dev(_ptr(s["x"]), _ptr(s["res"]), _ptr(s["norm"]), case["hidden"], B, EPS,
                                         _ptr(s["x_out"]), _ptr(s["xn"]), st))
            _check(L.jh_qmatvec_batched_swiglu_dev(s["gate"].handle, s["up"].handle, _ptr(s["xn"]), B, _ptr(s["hid"]),
                                                   _ptr(s["g"]), _ptr(s["u"]), st))
            _check(L.jh_qmatvec_batched_dev(s["down"].handle, _ptr(s["hid"]), B, _ptr(s["y"]), 0, case["hidden"], st))
        return [s["x_out"], s["hid"], s["y"]]
    if k == "head":
        if B == 1:
            _check(L.jh_rmsnorm_qmatvec_dev(s["w"].handle, _ptr(s["x"]), _ptr(s["res"]), _ptr(s["norm"]), EPS,
                                            _ptr(s["x_out"]), _ptr(s["xn"]), _ptr(s["y"]), st))
        else:
            _check(L.jh_rmsnorm_rows_dev(_ptr(s["x"]), _ptr(s["res"]), _ptr(s["norm"]), case["hidden"], B, EPS,
                                         _ptr(s["x_out"]), _ptr(s["xn"]), st))
            _check(L.jh_qmatvec_batched_dev(s["w"].handle, _ptr(s["xn"]), B, _ptr(s["y"]), 0, case["vocab"], st))
        return [s["x_out"], s["y"]]
    if k == "attn":
        h, kv, hd = case["heads"], case["kv"], case["hd"]
        if B == 1:
            _check(L.jh_rope_attention_qmatvec_dev(_ptr(s["q"]), _ptr(s["k"]), _ptr(s["v"]), h, kv, hd, _ptr(s["pos"]),
                                                   case["max_seq"], case["theta"], _ptr(s["kc"]), _ptr(s["vc"]),
                                                   s["wo"].handle, _ptr(s["att"]), _ptr(s["y"]), st))
        else:
            _check(L.jh_rope_attention_batched_dev(_ptr(s["q"]), _ptr(s["k"]), _ptr(s["v"]), B, h, kv, hd,
                                                   _ptr(s["pos"]), _ptr(s["slot"]), B, case["max_seq"], case["theta"],
                                                   _ptr(s["kc"]), _ptr(s["vc"]), _ptr(s["att"]), st))
            _check(L.jh_qmatvec_batched_dev(s["wo"].handle, _ptr(s["att"]), B, _ptr(s["y"]), 0, h * hd, st))
        return [s["att"], s["y"], s["kc"], s["vc"]]
    if k == "merge":
        cur = st.value or 0
        s["be"].dequantize_dev(s["w"], s["full"].data_ptr(), cur)
        torch.add(s["full"], s["delta"], out=s["full"])
        mv.quantize_dev(TYPES[case["type"]], s["full"].data_ptr(), s["full"].numel(), s["packed"].data_ptr(), cur)
        return [s["full"], s["packed"]]
    if k == "step":
        dec = s["dec"]
        dec.token.copy_(s["tokens"])
        dec.pos.copy_(s["pos"])
        s["graph"].replay()
        return [dec.logits, dec.k_cache, dec.v_cache]
    return s["pipe"].forward_batch(s["ids"], s["tokens"], s["pos"])


# ------------------------------------------------------------------ 64 bits
def _rms64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, pos, hd, theta):
    """Adjacent pairs of x [B, heads * hd] rotated by each row's position."""
    p = torch.arange(hd // 2, device="cuda", dtype=torch.float64)
    ang = pos.double().view(-1, 1, 1) * theta ** (-2.0 * p / hd)
    v = x.view(x.shape[0], -1, hd // 2, 2)
    a, b = v[..., 0], v[..., 1]
    c, s = ang.cos(), ang.sin()
    return torch.stack([a * c - b * s, a * s + b * c], -1).reshape(x.shape)


def _attend64(q, k, v, pos, slot, kc, vc, heads, kv, hd, theta):
    """The attention output [B, heads * hd]; kc and vc (64-bit copies are made per request) get the new rows."""
    q, k, v = _rope64(q, pos, hd, theta), _rope64(k, pos, hd, theta), v
    out = []
    for b, (p, z) in enumerate(zip(pos.tolist(), slot.tolist())):
        kc[z, p], vc[z, p] = k[b].to(kc.dtype), v[b].to(vc.dtype)
        K, V = kc[z, :p + 1].double().view(p + 1, kv, hd), vc[z, :p + 1].double().view(p + 1, kv, hd)
        K[p], V[p] = k[b].view(kv, hd), v[b].view(kv, hd)
        s = torch.matmul(q[b].view(kv, heads // kv, hd), K.permute(1, 2, 0).contiguous()) / math.sqrt(hd)
        out.append(torch.matmul(s.softmax(-1), V.permute(1, 0, 2).contiguous()).reshape(-1))
    return torch.stack(out)


def _silu64(x):
    return x / (1.0 + torch.exp(-x))


def exact(case, seed):
    i, k = _inputs(case, seed), case["kind"]
    if k in ("host", "proj"):
        w = _w64(i["w"])[case["row0"]:]
        y = i["x"].double() @ w.T
        return y[0] if k == "host" else y
    if k in ("qkv", "mlp", "head"):
        h = i["x"].double() + i["res"].double()
        xn = _rms64(h, i["norm"])
        if k == "qkv":
            return [h, *[xn @ _w64(m).T for m in i["mats"]]]
        if k == "head":
            return [h, xn @ _w64(i["w"]).T]
        hid = _silu64(xn @ _w64(i["gate"]).T) * (xn @ _w64(i["up"]).T)
        return [h, hid, hid @ _w64(i["down"]).T]
    if k == "attn":
        slot = torch.zeros_like(i["slot"]) if i["slot"].numel() == 1 else i["slot"]
        att = _attend64(i["q"].double(), i["k"].double(), i["v"].double(), i["pos"], slot, i["kc"], i["vc"],
                        case["heads"], case["kv"], case["hd"], case["theta"])
        return [att, att @ _w64(i["wo"]).T, i["kc"], i["vc"]]
    if k == "merge":
        return [_w64(i["w"]) + i["delta"].double(), None]
    m, B = TINYLLAMA, case["batch"]
    slot = torch.arange(B, device="cuda")
    x = _w64(i["embd"])[i["tokens"].long()]
    for li, lw in enumerate(i["layers"]):
        xn = _rms64(x, lw["attn_norm"])
        att = _attend64(xn @ _w64(lw["q"]).T, xn @ _w64(lw["k"]).T, xn @ _w64(lw["v"]).T, i["pos"], slot, i["kc"][li],
                        i["vc"][li], m["heads"], m["kv"], m["hd"], m["theta"])
        x = x + att @ _w64(lw["o"]).T
        xn = _rms64(x, lw["ffn_norm"])
        x = x + (_silu64(xn @ _w64(lw["gate"]).T) * (xn @ _w64(lw["up"]).T)) @ _w64(lw["down"]).T
    logits = _rms64(x, i["out_norm"]) @ _w64(i["out"]).T
    return [logits[0], i["kc"][:, 0], i["vc"][:, 0]] if k == "step" else list(logits)


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    k, B = case["kind"], case.get("batch", 1)
    if k in ("host", "proj"):
        r, c = case["rows"], case["cols"]
        return {"bytes": _packed_size(case["type"], r, c) + 4 * B * (r + c), "flops": 2 * B * r * c}
    if k == "qkv":
        H = case["hidden"]
        n = sum(r for _, r in _qkv_mats(case))
        return {"bytes": sum(_packed_size(t, r, H) for t, r in _qkv_mats(case)) + 4 * B * (3 * H + n) + 4 * H,
                "flops": 2 * B * n * H}
    if k == "mlp":
        H, F = case["hidden"], case["ffn"]
        a, b = MIX[case["mix"]]
        return {"bytes": 2 * _packed_size(a, F, H) + _packed_size(b, H, F) + 4 * B * (4 * H + F) + 4 * H,
                "flops": 6 * B * H * F}
    if k == "head":
        H, V = case["hidden"], case["vocab"]
        return {"bytes": _packed_size(case["type"], V, H) + 4 * B * (3 * H + V) + 4 * H, "flops": 2 * B * H * V}
    if k == "attn":
        D, KV = case["heads"] * case["hd"], case["kv"] * case["hd"]
        n = case["ctx"] if B == 1 else B * case["ctx"] * 3 // 4  # positions attended over
        return {"bytes": _packed_size(case["type"], D, D) + 4 * (2 * n * KV + B * (3 * D + 4 * KV)),
                "flops": 2 * B * D * D + 4 * n * D}
    if k == "merge":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * _packed_size(case["type"], case["rows"], case["cols"]) + 8 * n, "flops": 8 * n}
    m, (a, b) = TINYLLAMA, MIX[case["mix"]]
    H, F, KV, V = m["hidden"], m["ffn"], m["kv"] * m["hd"], m["vocab"]
    per = _packed_size(a, 2 * H + KV + 2 * F, H) + _packed_size(b, KV, H) + _packed_size(b, H, F)
    n = case["layers"] * (2 * H * H + 2 * KV * H + 3 * F * H) + V * H
    return {"bytes": case["layers"] * (per + 8 * B * case["pos"] * KV) + _packed_size(b, V, H) + 4 * B * V,
            "flops": 2 * B * n + 4 * B * case["layers"] * case["pos"] * H}


def tolerance(case):
    # 32-bit sums of a few thousand terms in another order
    k = case["kind"]
    if k == "merge":
        return "exact"
    if k in ("step", "serve"):
        return {"rel": 1e-4}
    return {"rel": 1e-5}
