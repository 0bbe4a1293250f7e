"""Timed cases of the decode framework: what its users run, through its public entry points.

Three kinds of case.

- ``linear``: one projection over activation rows, as a program that binds the launch seam calls it: the rows are
  packed (``cj_q8k_pack``; Q4_0 and MXFP4 read f32 rows) and multiplied with a prepared weight (``cj_matvec``,
  ``cj_matvec_mxfp4_q8`` for one row, ``cj_matmul`` for several).
- ``attend``: one layer's decode attention of one token: QK prep (RoPE, K/V append) and the attend over the paged
  fp16 K/V.
- ``generate``: a whole call: prompts prefilled into sequence slots, then greedy decoding, one slot (``decode``) or
  several at once (``decodeBatch``), with the logits the caller reads.

Inputs are made on the GPU from the seed alone: weights as GGUF blocks of the named format whose values are close to
N(0, 0.02), activations N(0, 1) (what a norm leaves), uniformly random prompt ids.
"""
import ctypes
import importlib.util
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F32, Q4_0, Q8_0, Q4_K, Q6_K, MXFP4 = 0, 2, 8, 12, 14, 39
TYPES = {"f32": F32, "q4_0": Q4_0, "q8_0": Q8_0, "q4_k": Q4_K, "q6_k": Q6_K, "mxfp4": MXFP4}
BLOCK = {F32: (1, 4), Q4_0: (32, 18), Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210), MXFP4: (32, 17)}

# hidden, query heads, kv heads, head size, FFN width, layers, experts, experts used, projection type, expert type,
# embedding type, head type, window, vocabulary
MODELS = {
    # the tiny Q8_0 model, whole
    "tiny": (512, 8, 2, 64, 1408, 4, 0, 0, "q8_0", "", "f32", "q8_0", 0, 32000),
    # two layers of the Llama-3-8B shape in its 4-bit K-quant form (Q6_K head)
    "dense": (4096, 32, 8, 128, 14336, 2, 0, 0, "q4_k", "", "q4_k", "q6_k", 0, 32000),
    # two layers of the gpt-oss-20b shape: one with a 128-position window, one without
    "moe": (2880, 64, 8, 64, 2880, 2, 32, 4, "q8_0", "mxfp4", "q8_0", "q8_0", 128, 32000),
}


def listed():
    def linear(name, type, rows, cols, n):
        return {"name": name, "kind": "linear", "type": type, "rows": rows, "cols": cols, "n": n}

    def attend(name, heads, kv, hd, count):
        return {"name": name, "kind": "attend", "heads": heads, "kv": kv, "hd": hd, "count": count}

    def generate(name, model, slots, prompt, steps):
        return {"name": name, "kind": "generate", "model": model, "slots": slots, "prompt": prompt, "steps": steps}

    return [
        # the smallest call: one token's k or v projection at the 8B shape
        linear("kv_proj_q4k_1", "q4_k", 1024, 4096, 1),
        # one token's down projection at the 8B shape, the ordinary decode GEMV
        linear("down_q4k_1", "q4_k", 4096, 14336, 1),
        # one token's output head: the largest GEMV of a step
        linear("head_q6k_1", "q6_k", 128256, 4096, 1),
        # a batch of 32 decoding sequences through the gate (or up) projection
        linear("gate_q80_32", "q8_0", 14336, 4096, 32),
        # a whole prefill chunk through the gate and the down projection, 8-bit and 4-bit weights
        linear("gate_q80_512", "q8_0", 14336, 4096, 512),
        linear("down_q4k_512", "q4_k", 4096, 14336, 512),
        # the ragged end of a prompt through a down projection kept at 6 bits, as K-quant mixes do
        linear("down_q6k_203", "q6_k", 4096, 14336, 203),
        # one token's attention at a 2049-position context, 8B shape (split-K form)
        attend("attend_h128_2049", 32, 8, 128, 2049),
        # one token's attention at a 4097-position context, gpt-oss shape (two-pass form)
        attend("attend_h64_4097", 64, 8, 64, 4097),
        # one short request on the tiny model: the launch-bound whole call
        generate("tiny_1x16+64", "tiny", 1, 16, 64),
        # a batch of long, ragged prompts answered together: prefill chunks, then batched decode steps
        generate("dense_8x1100+32", "dense", 8, 1100, 32),
        generate("moe_16x300+16", "moe", 16, 300, 16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("linear", "attend", "generate"), (7, 2, 1))[0]
    if kind == "linear":
        type = rng.choice(("q4_k", "q4_k", "q8_0", "q8_0", "q6_k", "q4_0", "mxfp4"))
        step = BLOCK[TYPES[type]][0]
        rows, cols = _log(rng, 256, 32768), step * max(1, _log(rng, 1024, 14336) // step)
        n = 1 if type == "mxfp4" or rng.random() < 0.3 else _log(rng, 2, 16 if type == "q4_0" else 512)
        while rows * cols * n > 2.5e10:
            n //= 2
        return {"kind": kind, "type": type, "rows": rows, "cols": cols, "n": max(1, n)}
    if kind == "attend":
        heads, kv, hd = rng.choice(((32, 8, 128), (64, 8, 128), (64, 8, 64), (8, 2, 64), (16, 8, 128)))
        return {"kind": kind, "heads": heads, "kv": kv, "hd": hd, "count": _log(rng, 16, 6000)}
    model = rng.choice(("tiny", "dense", "moe"))
    slots = rng.choice((1, 2, 3, 5, 8))
    return {"kind": kind, "model": model, "slots": slots, "prompt": _log(rng, 16, 1000), "steps": _log(rng, 4, 32)}


# ------------------------------------------------------------------ inputs

def _gen(seed, k=0):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + 7919 * k) % (1 << 62))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _half(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def _blocks(g, type, rows, cols):
    """Random weight rows as GGUF blocks of `type`: uint8 [rows, row bytes]."""
    if type == F32:
        return (_randn(g, rows, cols) / math.sqrt(cols)).view(torch.uint8)
    per, size = BLOCK[type]
    nb = cols // per
    out = torch.empty(rows, nb, size, dtype=torch.uint8, device="cuda")
    step = max(1, (1 << 25) // max(1, cols))   # rows made at a time
    for r in range(0, rows, step):
        n = min(step, rows - r)
        z, wob = _randn(g, n, nb, per), 1.0 + 0.1 * _randn(g, n, nb).clamp(-3, 3)
        o = out[r:r + n]
        if type == Q8_0:
            o[..., :2] = _half(0.02 / 42 * wob)
            o[..., 2:] = (z * 42).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        elif type == Q4_0:
            c = (z * 2.7 + 8).round().clamp(0, 15).to(torch.uint8)
            o[..., :2] = _half(0.02 / 2.7 * wob)
            o[..., 2:] = c[..., :16] | (c[..., 16:] << 4)
        elif type == MXFP4:
            value = torch.tensor([0, 1, 2, 3, 4, 6, 8, 12], device="cuda", dtype=torch.float32)
            edge = (value[1:] + value[:-1]) / 2
            c = torch.bucketize((z * 4.5).abs(), edge).to(torch.uint8) | ((z < 0).to(torch.uint8) << 3)
            o[..., 0] = 120 + (torch.rand(n, nb, generator=g, device="cuda") < 0.3)
            o[..., 1:] = c[..., :16] | (c[..., 16:] << 4)
        elif type == Q4_K:
            c = (z * 2.6 + 7.5).round().clamp(0, 15).to(torch.uint8).reshape(n, nb, 4, 2, 32)
            sc = torch.randint(40, 64, (n, nb, 8), generator=g, device="cuda", dtype=torch.uint8)
            mn = torch.randint(40, 64, (n, nb, 8), generator=g, device="cuda", dtype=torch.uint8)
            o[..., 0:2] = _half(0.02 / 2.6 / 52 * wob)
            o[..., 2:4] = _half(0.02 * 7.5 / 2.6 / 52 * wob)
            o[..., 4:8] = sc[..., :4] | ((sc[..., 4:] >> 4) << 6)
            o[..., 8:12] = mn[..., :4] | ((mn[..., 4:] >> 4) << 6)
            o[..., 12:16] = (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)
            o[..., 16:] = (c[..., 0, :] | (c[..., 1, :] << 4)).reshape(n, nb, 128)
        else:
            c = ((z * 10.5).round().clamp(-32, 31) + 32).to(torch.uint8).reshape(n, nb, 2, 4, 32)
            sc = torch.randint(80, 128, (n, nb, 16), generator=g, device="cuda", dtype=torch.int16)
            sc = sc * (1 - 2 * torch.randint(0, 2, (n, nb, 16), generator=g, device="cuda", dtype=torch.int16))
            lo, hi = c & 15, c >> 4
            o[..., :128] = torch.cat((lo[..., 0, :] | (lo[..., 2, :] << 4), lo[..., 1, :] | (lo[..., 3, :] << 4)), -1).reshape(n, nb, 128)
            o[..., 128:192] = (hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)).reshape(n, nb, 64)
            o[..., 192:208] = sc.to(torch.int8).view(torch.uint8)
            o[..., 208:] = _half(0.02 / 10.5 / 104 * wob)
    return out.reshape(rows, nb * size)


def _values(raw, type, cols):
    """The weight rows that the blocks hold, in 64 bits."""
    rows = raw.shape[0]
    if type == F32:
        return raw.view(torch.float32).double()
    per, size = BLOCK[type]
    b = raw.reshape(rows, cols // per, size)

    def half(x):
        return x.contiguous().view(torch.float16).double()

    if type == Q8_0:
        v = half(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).double()
    elif type == Q4_0:
        c = torch.cat((b[..., 2:] & 15, b[..., 2:] >> 4), -1).double() - 8
        v = half(b[..., :2]) * c
    elif type == MXFP4:
        t = torch.tensor([0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12], device="cuda", dtype=torch.float64)
        c = torch.cat((b[..., 1:] & 15, b[..., 1:] >> 4), -1)
        v = torch.exp2(b[..., :1].double() - 128) * t[c.long()]
    elif type == Q4_K:
        s = b[..., 4:16]
        sc = torch.cat((s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)), -1).double()
        mn = torch.cat((s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)), -1).double()
        q = b[..., 16:].reshape(rows, -1, 4, 1, 32)
        c = torch.cat((q & 15, q >> 4), 3).reshape(rows, -1, 8, 32).double()
        v = c * (half(b[..., 0:2]) * sc).unsqueeze(-1) - (half(b[..., 2:4]) * mn).unsqueeze(-1)
    else:
        lo, hi = b[..., :128].reshape(rows, -1, 2, 2, 32), b[..., 128:192].reshape(rows, -1, 2, 1, 32)
        c = torch.cat((lo & 15, lo >> 4), 3) | (torch.cat((hi, hi >> 2, hi >> 4, hi >> 6), 3) & 3) << 4
        sc = b[..., 192:208].contiguous().view(torch.int8).double()
        v = (c.reshape(rows, -1, 16, 16).double() - 32) * (half(b[..., 208:]) * sc).unsqueeze(-1)
    return v.reshape(rows, cols)


def _packed(x, per):
    """Activation rows as an int8 pack holds them: codes and a scale for each `per` values."""
    x = x.float()
    rows, n = x.shape
    pad = (-n) % per
    b = torch.nn.functional.pad(x, (0, pad)).reshape(rows, -1, per)
    top = b.abs().amax(-1, keepdim=True)
    v = (b * torch.where(top > 0, torch.full_like(top, 127.0) / top, top)).double()
    q = torch.sign(v) * torch.floor(v.abs() + 0.5)
    return (q * (top / 127.0).double()).reshape(rows, -1)[:, :n]


# ------------------------------------------------------- the framework's side

def _package():
    name = "cajeta_llm_amd"
    if name not in sys.modules:
        d = os.path.join(ROOT, "cajeta-llm_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(d, "__init__.py"), submodule_search_locations=[d])
        m = importlib.util.module_from_spec(spec)
        sys.modules[name] = m
        spec.loader.exec_module(m)
        pkg = m
        pkg.native.init(0)
        try:   # the registry's lookup of an optional kernel leaves the runtime's last error set; torch would report it
            torch.zeros(1, device="cuda")
        except RuntimeError:
            pass
    return sys.modules[name]


class _View:
    """A device buffer's memory, as torch takes it."""

    def __init__(self, buf, shape, dtype):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": dtype, "data": (buf.h, False), "version": 2}


def _view(buf, shape, dtype="<f4"):
    t = torch.as_tensor(_View(buf, shape, dtype), device="cuda")
    t._held = buf
    return t


def _buffer(pkg, t):
    """A device buffer of the framework holding the tensor's values."""
    flat = t.contiguous().view(torch.uint8).reshape(-1)
    buf = pkg.Buffer(max(16, flat.numel()))
    _view(buf, flat.shape, "|u1").copy_(flat)
    torch.cuda.synchronize()
    return buf


def _status(pkg, rc):
    pkg.native.check(rc, "call")


# ----------------------------------------------------------------- linear

def _linear_inputs(case, seed):
    type = TYPES[case["type"]]
    raw = _blocks(_gen(seed, 1), type, case["rows"], case["cols"])
    return type, raw, _randn(_gen(seed, 2), case["n"], case["cols"])


def _prepare_linear(case, seed):
    pkg = _package()
    L = pkg.native.lib()
    type, raw, x = _linear_inputs(case, seed)
    rows, cols, n = case["rows"], case["cols"], case["n"]
    src = _buffer(pkg, raw)
    w = pkg.Buffer(rows * L.cj_prepared_row_bytes(type, cols))
    _status(pkg, L.cj_prepare_weight(w.h, src.h, type, rows, cols))
    pkg.native.sync()
    src.free()
    stride = (cols + 255) // 256 * 320
    s = {"pkg": pkg, "L": L, "type": type, "rows": rows, "cols": cols, "n": n, "w": w, "x": _buffer(pkg, x),
         "y": pkg.Buffer(n * rows * 4)}
    if type in (Q4_0, MXFP4):
        s["stride"] = cols * 4
    else:
        s["stride"], s["xp"] = stride, pkg.Buffer(n * stride)
    s["out"] = _view(s["y"], (n, rows))
    return s


def _run_linear(s):
    L, type, rows, cols, n = s["L"], s["type"], s["rows"], s["cols"], s["n"]
    x = s["x"].h
    if "xp" in s:
        _status(s["pkg"], L.cj_q8k_pack(s["xp"].h, x, n, cols, (cols + 255) // 256 * 256, 1 if type == Q8_0 else 0))
        x = s["xp"].h
    if type == MXFP4:
        rc = L.cj_matvec_mxfp4_q8(s["y"].h, s["w"].h, x, rows, cols, 0, 0)
    elif n == 1:
        rc = L.cj_matvec(type, s["y"].h, s["w"].h, x, rows, cols, 0, 0)
    else:
        rc = L.cj_matmul(type, s["y"].h, s["w"].h, x, rows, cols, n, s["stride"], rows, 0, 0)
    _status(s["pkg"], rc)
    return s["out"]


def _exact_linear(case, seed):
    type, raw, x = _linear_inputs(case, seed)
    rows, cols = case["rows"], case["cols"]
    x = x.double() if type == Q4_0 else _packed(x, 32 if type in (Q8_0, MXFP4) else 256)
    out = torch.empty(case["n"], rows, dtype=torch.float64, device="cuda")
    for r in range(0, rows, 8192):
        out[:, r:r + 8192] = x @ _values(raw[r:r + 8192], type, cols).t().contiguous()
    return out


# ----------------------------------------------------------------- attend

THETA = 500000.0


def _attend_inputs(case, seed):
    kv, hd, count = case["kv"], case["hd"], case["count"]
    pages = (count + 63) // 64
    g = _gen(seed, 3)
    k, v = _randn(g, pages, kv, 64, hd).half(), _randn(g, pages, kv, 64, hd).half()
    order = torch.randperm(pages, generator=g, device="cuda").to(torch.int32)   # the pool's pages as a slot drew them
    qkv = _randn(g, case["heads"] + 2 * kv, hd)
    return k, v, order, qkv


def _prepare_attend(case, seed):
    pkg = _package()
    L = pkg.native.lib()
    heads, kv, hd, count = (case[n] for n in ("heads", "kv", "hd", "count"))
    k, v, order, qkv = _attend_inputs(case, seed)
    s = {"pkg": pkg, "L": L, "case": case, "kc": _buffer(pkg, k), "vc": _buffer(pkg, v), "pg": _buffer(pkg, order),
         "q0": _buffer(pkg, qkv[:heads]), "k0": _buffer(pkg, qkv[heads:heads + kv]), "v0": _buffer(pkg, qkv[heads + kv:]),
         "q": pkg.Buffer(heads * hd * 4), "k": pkg.Buffer(kv * hd * 4), "part": pkg.Buffer(heads * max(64 * (hd + 2), count) * 4),
         "rope": pkg.Buffer(count * hd * 4), "counters": pkg.Buffer(max(16, kv * 4)), "y": pkg.Buffer(heads * hd * 4)}
    _status(pkg, L.cj_rope_table(s["rope"].h, hd, THETA, count))
    s["counters"].zero()
    pkg.native.sync()
    s["out"] = _view(s["y"], (heads, hd))
    return s


def _run_attend(s):
    L, c = s["L"], s["case"]
    heads, kv, hd, count = c["heads"], c["kv"], c["hd"], c["count"]
    # the projections' fresh q and k of this token, rotated in place by the prep
    _status(s["pkg"], L.cj_buf_copy(s["q"].h, s["q0"].h, heads * hd * 4))
    _status(s["pkg"], L.cj_buf_copy(s["k"].h, s["k0"].h, kv * hd * 4))
    _status(s["pkg"], L.cj_qk_prep(s["q"].h, s["k"].h, s["v0"].h, s["kc"].h, s["vc"].h, 0, 0, s["rope"].h, s["pg"].h, 0,
                                   heads, kv, hd, 0, ctypes.c_float(1e-5), 0, count - 1))
    _status(s["pkg"], L.cj_attend(s["part"].h, s["y"].h, s["q"].h, s["kc"].h, s["vc"].h, s["pg"].h, 0, s["counters"].h, heads,
                                  kv, hd, count, 0, 512, ctypes.c_float(1.0 / math.sqrt(hd))))
    return s["out"]


def _rope(x, pos, theta, half_split):
    """x [..., hd] at positions pos: the pairs (d, d + hd/2), or (2d, 2d + 1) as GGUF orders them."""
    hd = x.shape[-1]
    inv = torch.pow(torch.tensor(theta, dtype=torch.float32), -torch.arange(0, hd, 2, dtype=torch.float32) / hd).cuda()
    ang = (pos.float().reshape(-1, 1, 1) * inv).double()
    a, b = (x[..., :hd // 2], x[..., hd // 2:]) if half_split else (x[..., 0::2], x[..., 1::2])
    u, v = a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()
    return torch.cat((u, v), -1) if half_split else torch.stack((u, v), -1).flatten(-2)


def _attention(q, k, v, first, grp):
    """Causal attention of rows at positions first.. : q [n, heads, hd], k and v [positions, kv, hd]."""
    n, heads, hd = q.shape
    out = torch.empty(n, heads, hd, dtype=torch.float64, device="cuda")
    seen = torch.arange(k.shape[0], device="cuda")[None, :] <= first + torch.arange(n, device="cuda")[:, None]
    for h in range(heads):
        s = (q[:, h] @ k[:, h // grp].t().contiguous()) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v[:, h // grp].contiguous()
    return out


def _exact_attend(case, seed):
    heads, kv, hd, count = (case[n] for n in ("heads", "kv", "hd", "count"))
    k, v, order, qkv = _attend_inputs(case, seed)

    def rows(p):
        return p[order.long()].permute(0, 2, 1, 3).reshape(-1, kv, hd)[:count].double()

    k, v, qkv = rows(k), rows(v), qkv.double()
    pos = torch.tensor([count - 1], device="cuda")
    k[count - 1] = _rope(qkv[heads:heads + kv][None], pos, THETA, True)[0].half().double()
    v[count - 1] = qkv[heads + kv:].half().double()
    return _attention(_rope(qkv[:heads][None], pos, THETA, True), k, v, count - 1, heads // kv)[0]


# --------------------------------------------------------------- generate

def _tensors(model):
    """(name, type, rows, cols, shape) of the model's tensors."""
    h, nq, nk, hd, ffn, layers, experts, _, wt, et, emb, head, _, vocab = MODELS[model]
    yield "token_embd.weight", TYPES[emb], vocab, h, (h, vocab)
    for l in range(layers):
        p = "blk.%d." % l
        for name, rows, cols in (("attn_norm", 1, h), ("attn_q", nq * hd, h), ("attn_k", nk * hd, h), ("attn_v", nk * hd, h),
                                 ("attn_output", h, nq * hd), ("ffn_norm", 1, h)):
            yield p + name + ".weight", F32 if rows == 1 else TYPES[wt], rows, cols, (cols,) if rows == 1 else (cols, rows)
        if experts:
            yield p + "ffn_gate_inp.weight", F32, experts, h, (h, experts)
        for name, rows, cols in (("ffn_gate", ffn, h), ("ffn_up", ffn, h), ("ffn_down", h, ffn)):
            if experts:
                yield p + name + "_exps.weight", TYPES[et], experts * rows, cols, (cols, rows, experts)
            else:
                yield p + name + ".weight", TYPES[wt], rows, cols, (cols, rows)
    yield "output_norm.weight", F32, 1, h, (h,)
    yield "output.weight", TYPES[head], vocab, h, (h, vocab)


def _tensor(seed, k, name, type, rows, cols):
    g = _gen(seed, 100 + k)
    return (1 + 0.02 * _randn(g, 1, cols)).view(torch.uint8) if name.endswith("norm.weight") else _blocks(g, type, rows, cols)


def _write_model(model, seed, path):
    h, nq, nk, hd, ffn, layers, experts, used, _, _, _, _, window, vocab = MODELS[model]

    def text(s):
        return struct.pack("<Q", len(s)) + s.encode()

    kv = [("general.architecture", 8, text("llama")), ("general.alignment", 4, struct.pack("<I", 32))]
    for key, v in (("context_length", 8192), ("embedding_length", h), ("block_count", layers), ("feed_forward_length", ffn),
                   ("attention.head_count", nq), ("attention.head_count_kv", nk), ("attention.key_length", hd),
                   ("attention.value_length", hd), ("rope.dimension_count", hd), ("vocab_size", vocab)):
        kv.append(("llama." + key, 4, struct.pack("<I", v)))
    if experts:
        for key, v in (("expert_count", experts), ("expert_used_count", used), ("expert_feed_forward_length", ffn),
                       ("expert_weights_norm", 1), ("expert_gating_func", 1), ("attention.sliding_window", window),
                       ("attention.sliding_window_pattern", 2)):
            kv.append(("llama." + key, 4, struct.pack("<I", v)))
    kv.append(("llama.rope.freq_base", 6, struct.pack("<f", THETA)))
    kv.append(("llama.attention.layer_norm_rms_epsilon", 6, struct.pack("<f", 1e-5)))
    tensors = list(_tensors(model))
    head = b"GGUF" + struct.pack("<IQQ", 3, len(tensors), len(kv)) + b"".join(text(k) + struct.pack("<I", t) + v for k, t, v in kv)
    at = 0
    for name, type, rows, cols, shape in tensors:
        head += text(name) + struct.pack("<I%dQIQ" % len(shape), len(shape), *shape, type, at)
        per, size = BLOCK[type]
        at += (rows * (cols // per) * size + 31) // 32 * 32
    with open(path, "wb") as f:
        f.write(head + bytes((-len(head)) % 32))
        for k, (name, type, rows, cols, _) in enumerate(tensors):
            raw = _tensor(seed, k, name, type, rows, cols).cpu().numpy()
            f.write(raw.data)
            f.write(bytes((-raw.nbytes) % 32))


def _prompts(case, seed):
    """Ragged prompts: the longest first, each a few tokens shorter than the one before."""
    rng = np.random.default_rng(int(seed))
    vocab = MODELS[case["model"]][13]
    return [rng.integers(0, vocab, max(2, case["prompt"] - 37 * i), dtype=np.int32) for i in range(case["slots"])]


def _prepare_generate(case, seed):
    pkg = _package()
    opts = pkg.EngineOptions("")
    opts.ctx = (case["prompt"] + case["steps"] + 64) // 64 * 64
    opts.maxSeqs = case["slots"]
    shm = "/dev/shm" if os.path.isdir("/dev/shm") else None
    fd, opts.model = tempfile.mkstemp(suffix=".gguf", dir=shm)
    os.close(fd)
    try:
        _write_model(case["model"], seed, opts.model)
        eng = pkg.LlmEngine.load(opts)
    finally:
        os.unlink(opts.model)
    return {"engine": eng, "prompts": _prompts(case, seed), "steps": case["steps"]}


def _run_generate(s):
    eng, steps = s["engine"], s["steps"]
    for slot, p in enumerate(s["prompts"]):
        eng.reset(slot)
        eng.prefill(p, slot)
        if slot == 0:
            first = eng.logits(slot)
    if len(s["prompts"]) == 1:
        return {"prompt": first, "tokens": eng.decode(steps), "last": eng.logits(0)}
    return {"prompt": first, "tokens": eng.decodeBatch(range(len(s["prompts"])), steps), "last": eng.batchLogits()}


def _exact_generate(case, seed):
    """The first prompt's logits; what follows depends on the tokens picked and has no value of its own."""
    h, nq, nk, hd, _, layers, experts, _, wt, _, emb, head, _, _ = MODELS[case["model"]]
    if experts:
        return None
    at = {name: (k, name, type, rows, cols) for k, (name, type, rows, cols, _) in enumerate(_tensors(case["model"]))}

    def weight(name):
        return _values(_tensor(seed, *at[name]), at[name][2], at[name][4])

    def norm(x, name):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5) * weight(name)

    def linear(x, name):
        return _packed(x, 32 if at[name][2] == Q8_0 else 256) @ weight(name).t().contiguous()

    def silu(x):
        return x / (1 + torch.exp(-x))

    ids = torch.from_numpy(_prompts(case, seed)[0]).cuda().long()
    pos = torch.arange(len(ids), device="cuda")
    x = weight("token_embd.weight")[ids]
    for l in range(layers):
        p = "blk.%d." % l
        n = norm(x, p + "attn_norm.weight")
        q, k, v = (linear(n, p + "attn_%s.weight" % c).reshape(len(ids), -1, hd) for c in "qkv")
        q, k = _rope(q, pos, THETA, False), _rope(k, pos, THETA, False).half().double()
        a = _attention(q, k, v.half().double(), 0, nq // nk)
        x = x + linear(a.reshape(len(ids), -1), p + "attn_output.weight")
        n = norm(x, p + "ffn_norm.weight")
        x = x + linear(silu(linear(n, p + "ffn_gate.weight")) * linear(n, p + "ffn_up.weight"), p + "ffn_down.weight")
    logits = linear(norm(x[-1:], "output_norm.weight"), "output.weight")[0]
    return {"prompt": logits, "tokens": None, "last": None}


# ------------------------------------------------------------------ the rest

def prepare(case, seed):
    return {"linear": _prepare_linear, "attend": _prepare_attend, "generate": _prepare_generate}[case["kind"]](case, seed)


def run(state):
    return _run_generate(state) if "engine" in state else _run_attend(state) if "kc" in state else _run_linear(state)


def exact(case, seed):
    return {"linear": _exact_linear, "attend": _exact_attend, "generate": _exact_generate}[case["kind"]](case, seed)


def _weight_bytes(type, rows, cols):
    per, size = BLOCK[type]
    return rows * (cols // per) * size


def work(case):
    if case["kind"] == "linear":
        rows, cols, n = case["rows"], case["cols"], case["n"]
        return {"bytes": _weight_bytes(TYPES[case["type"]], rows, cols) + 4 * n * (rows + cols), "flops": 2 * rows * cols * n}
    if case["kind"] == "attend":
        heads, kv, hd, count = (case[n] for n in ("heads", "kv", "hd", "count"))
        return {"bytes": 4 * count * kv * hd + 4 * hd * (2 * heads + 2 * kv), "flops": 4 * heads * hd * count}
    h, nq, nk, hd, _, layers, experts, used, _, _, _, _, window, vocab = MODELS[case["model"]]
    sizes = [(name, _weight_bytes(t, r, c), r * c) for name, t, r, c, _ in _tensors(case["model"])]
    head = sizes[-1][2]
    body = sum(e * (used / experts if "_exps" in n else 1) for n, _, e in sizes[1:-1])
    lens = [max(2, case["prompt"] - 37 * i) for i in range(case["slots"])]
    steps, rows = case["steps"], sum(lens) + case["slots"] * case["steps"]
    # weights once a prompt chunk of 512 rows and once a step, K/V read once a step
    passes = sum((p + 511) // 512 for p in lens) + steps
    total = passes * sum(b for _, b, _ in sizes[1:-1]) + (len(lens) + steps) * sizes[-1][1]
    flops = 2 * body * rows + 2 * head * case["slots"] * (1 + steps)
    for l in range(layers):
        near = window if window and (l + 1) % 2 else 1 << 30
        total += sum(4 * nk * hd * min(near, p + i) for p in lens for i in range(steps))
        flops += sum(4 * nq * hd * min(near, p) for n in lens for p in range(1, n + steps))
    if experts:   # a step of few rows reads the experts that its rows picked, at most
        bank = sum(b for n, b, _ in sizes if "_exps" in n)
        total -= steps * bank * max(0.0, 1 - case["slots"] * used / experts)
    return {"bytes": total, "flops": flops}


def tolerance(case):
    if case["kind"] == "linear":     # 32-bit sums over exact integer block products
        return {"rel": 2e-6}
    if case["kind"] == "attend":     # 32-bit softmax and sums
        return {"rel": 5e-6}
    # whole calls: a code of an activation pack that rounds the other way in one layer moves what follows
    return {"rel": 0.03, "differ": 0.01}
