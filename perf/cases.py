"""What is measured of this engine: whole calls of its C ABI as a serving program makes them (decode
steps at a context, verify of drafts, prefill of a prompt, the reference's teacher-forced token loop)
and the one layer that a program can call by itself, the decode attention on its own buffers.

    listed()  the cases by name            prepare(case, seed)  what a program holds before the call
    draw(rng) one more of the same ranges  run(state)           one pass
    work, tolerance, exact                 bytes and operations, the bound, the result in 64 bits

Weights are the seeded archives of libchpe_pack.so (the workloads of bench.py), one engine per model
and cache type kept for the process, as a server keeps it.  Every call gets new tokens from the seed.
"""
import math
import random
import sys
import tempfile
from pathlib import Path

import numpy as np
import torch

ROOT = Path.cwd()
sys.path.insert(0, str(ROOT / "chpe-qwen-engine_amd"))
import chpe_amd as ca  # noqa: E402

# model: archive kind, architecture id, shapes, cache rows of the engine
MODELS = {
    "3b-w4": dict(kind=ca.PACK_3B_W4, arch=0, V=151936, L=36, H=16, KV=2, hd=128, D=2048, I=11008, rows=4160),
    "3b-fp16": dict(kind=ca.PACK_3B_FP16_RAW, arch=0, V=151936, L=36, H=16, KV=2, hd=128, D=2048, I=11008, rows=2048),
    "9b-hybrid": dict(kind=ca.PACK_9B_W4, arch=3, V=248320, L=32, H=16, KV=4, hd=256, D=4096, I=12288, rows=2304),
    "72b-w4": dict(kind=ca.PACK_72B_W4, arch=2, V=152064, L=80, H=64, KV=8, hd=128, D=8192, I=29568, rows=8320),
}
HEADS = {"3b": (16, 2, 128), "9b": (16, 4, 256), "72b": (64, 8, 128)}  # query heads, kv heads, head dim


def listed():
    return [
        # one layer's decode attention in a program's own step, the f32 cache and 2048 rows that
        # chpe_init gives a 3B model, a third of it filled: the smallest call
        dict(name="attention 3b f32 at 701", op="attention", heads="3b", kv_f16=False, rows=2048, pos=701),
        # the same of the 72B model at the end of an 8192-token prompt
        dict(name="attention 72b f16 at 8255", op="attention", heads="72b", kv_f16=True, rows=8320, pos=8255),
        # a sampling server's steps: every step's logits go to the host; the reference's cache type
        dict(name="decode 3b-w4 f32 at 515", op="decode", model="3b-w4", kv_f16=False, pos=515, n=4),
        # the same at the context of the 3B benchmark with the fp16 cache
        dict(name="decode 3b-w4 f16 at 4099", op="decode", model="3b-w4", kv_f16=True, pos=4099, n=4),
        # speculative decoding with a small draft, mid-context
        dict(name="verify 5 3b-w4 f16 at 1501", op="verify", model="3b-w4", kv_f16=True, pos=1501, n=5),
        # the reference's own caller: its CPU-runnable fp16 archive, a 32-token prompt, last logits
        dict(name="forward 3b-fp16 32", op="forward", model="3b-fp16", kv_f16=False, n=32),
        # the hybrid model's recurrent step, from an empty state (it cannot be rewound)
        dict(name="forward 9b-hybrid 24", op="forward", model="9b-hybrid", kv_f16=True, n=24),
        # a chat turn's prompt on the small and on the hybrid model, odd lengths
        dict(name="prefill 3b-w4 f32 777", op="prefill", model="3b-w4", kv_f16=False, n=777),
        dict(name="prefill 9b-hybrid 501", op="prefill", model="9b-hybrid", kv_f16=True, n=501),
        # the headline model: decode and verify at its 8192-token context, a prompt's prefill
        dict(name="decode 72b-w4 at 8192", op="decode", model="72b-w4", kv_f16=True, pos=8192, n=2),
        dict(name="verify 8 72b-w4 at 8200", op="verify", model="72b-w4", kv_f16=True, pos=8200, n=8),
        dict(name="prefill 72b-w4 300", op="prefill", model="72b-w4", kv_f16=True, n=300),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random):
    op = rng.choice(["attention", "attention", "decode", "decode", "verify", "forward", "prefill", "prefill"])
    if op == "attention":
        heads, f16 = rng.choice(list(HEADS)), rng.random() < 0.6
        rows = 16 * _log(rng, 8, 520 if heads == "72b" else 260)
        return dict(op=op, heads=heads, kv_f16=f16, rows=rows, pos=_log(rng, 1, rows - 1))
    if op == "decode":
        if rng.random() < 0.35:
            return dict(op=op, model="72b-w4", kv_f16=True, pos=_log(rng, 33, 8300), n=rng.randint(1, 3))
        return dict(op=op, model="3b-w4", kv_f16=rng.random() < 0.5, pos=_log(rng, 33, 4100), n=rng.randint(1, 8))
    if op == "verify":
        if rng.random() < 0.5:
            return dict(op=op, model="72b-w4", kv_f16=True, pos=_log(rng, 33, 8280), n=_log(rng, 2, 32))
        return dict(op=op, model="3b-w4", kv_f16=rng.random() < 0.5, pos=_log(rng, 33, 4100), n=_log(rng, 2, 32))
    if op == "forward":
        if rng.random() < 0.5:
            return dict(op=op, model="3b-fp16", kv_f16=rng.random() < 0.5, n=_log(rng, 3, 100))
        return dict(op=op, model="9b-hybrid", kv_f16=True, n=_log(rng, 3, 100))
    model = rng.choice(["3b-w4", "9b-hybrid", "72b-w4"])
    top = {"3b-w4": 1500, "9b-hybrid": 1300, "72b-w4": 290}[model]
    return dict(op=op, model=model, kv_f16=model != "3b-w4" or rng.random() < 0.5, n=_log(rng, 9, top))


# ------------------------------------------------------------------ what a program holds
def _archive(kind):
    try:
        return ca.ensure_archive(kind, seed=0)
    except PermissionError:  # another user's folder: one of our own
        own = Path(tempfile.gettempdir()) / "chpe_archives_own"
        return ca.ensure_archive(kind, seed=0, directory=own)


class _Served:
    """An engine and the document that fills its cache: decode and verify calls go on from row P of
    it.  Calls overwrite rows; ensure(P) computes rows again that a call has overwritten."""

    def __init__(self, model, kv_f16):
        m = MODELS[model]
        self.e = ca.Engine(_archive(m["kind"]), arch=m["arch"], max_seq_len=m["rows"], kv_f16=kv_f16)
        self.doc = _tokens(model, m["rows"], 7)
        self.built, self.dirty = 0, None

    def ensure(self, upto):
        if self.dirty and self.dirty[0] < upto:
            lo, hi = self.dirty
            self._rows(lo, min(hi, self.built))
        if self.dirty and self.dirty[0] >= upto:  # (rows past what is needed: built anew when asked for)
            self.built = min(self.built, self.dirty[0])
        self.dirty = None
        if self.built < upto:
            self._rows(self.built, upto)
            self.built = upto

    def _rows(self, lo, hi):
        if lo == 0 and hi > 0:
            self.e.prefill(self.doc[:hi])
        else:
            for i in range(lo, hi, 32):
                self.e.verify(self.doc[i:min(i + 32, hi)], i)

    def touch(self, lo, hi):
        self.dirty = (lo, hi) if not self.dirty else (min(lo, self.dirty[0]), max(hi, self.dirty[1]))


_engines = {}


def _served(model, kv_f16):
    if (model, kv_f16) not in _engines:
        _engines[model, kv_f16] = _Served(model, kv_f16)
    return _engines[model, kv_f16]


def _tokens(model, n, seed):
    return np.random.default_rng(seed).integers(0, MODELS[model]["V"], n).astype(np.uint32)


def _attention_inputs(case, seed):
    """Rotated queries and cache rows as a layer meets them: unit-variance keys and values, queries
    whose scores spread over a few units; the engine's cache layout (include/chpe.h)."""
    H, KV, hd = HEADS[case["heads"]]
    rows, f16 = case["rows"], case["kv_f16"]
    g = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.randn(H, hd, generator=g, device="cuda") * 2.0
    dt = torch.float16 if f16 else torch.float32
    k = torch.randn(KV, rows, hd, generator=g, device="cuda").to(dt)
    v = torch.randn(KV, rows, hd, generator=g, device="cuda").to(dt)
    return q, k, v


def prepare(case, seed):
    if case["op"] == "attention":
        H, KV, hd = HEADS[case["heads"]]
        q, k, v = _attention_inputs(case, seed)
        if case["kv_f16"]:
            v = v.reshape(KV, case["rows"] // 4, 4, hd).transpose(2, 3).contiguous()
        out = torch.empty(H, hd, device="cuda")
        return dict(case=case, lib=ca.load_engine_lib(), q=q, k=k, v=v, out=out)
    s = _served(case["model"], case["kv_f16"])
    n, P = case["n"], case.get("pos", 0)
    if P:
        s.ensure(P)
    s.touch(P, P + n)
    return dict(case=case, e=s.e, tokens=_tokens(case["model"], n, seed + 1000003))


def run(st):
    c = st["case"]
    if c["op"] == "attention":
        H, KV, hd = HEADS[c["heads"]]
        rc = st["lib"].chpe_attention_noalloc(hd, H, KV, int(c["kv_f16"]), c["pos"], c["rows"], st["q"].data_ptr(),
                                              st["k"].data_ptr(), st["v"].data_ptr(), st["out"].data_ptr(),
                                              torch.cuda.current_stream().cuda_stream)
        if rc:
            raise RuntimeError(f"chpe_attention_noalloc: {rc}")
        return st["out"]
    e, toks = st["e"], st["tokens"]
    if c["op"] == "decode":
        return [e.decode_step(int(t), c["pos"] + i)[1] for i, t in enumerate(toks)]
    if c["op"] == "verify":
        drafts = e.verify(toks, c["pos"])
        # with the fp16 cache a row that rounds the other way can turn a near tie of two logits, so
        # the drafts' argmaxes are compared where the cache is exact
        return [e.logits()] if c["kv_f16"] else [e.logits(), drafts]
    if c["op"] == "forward":
        return [e.forward_tokens(toks, want_logits=True)[1]]
    return [e.prefill(toks, want_logits=True)[1]]


# ------------------------------------------------------------------ bytes and operations
def _weights(model):
    """(bytes, weights) of one pass over every projection and the LM head: codes, group scales."""
    m = MODELS[model]
    D, I, L, V, kvd = m["D"], m["I"], m["L"], m["V"], m["KV"] * m["hd"]
    if model == "9b-hybrid":  # 24 DeltaNet layers and 8 gated attention layers
        n = 24 * (8192 * D + 4096 * D + 64 * D + D * 4096) + 8 * (8192 * D + 2 * kvd * D + D * 4096) + L * 3 * D * I
    else:
        n = L * (2 * D * D + 2 * kvd * D + 3 * D * I)
    n += V * D
    return n * (2.0 if model == "3b-fp16" else 0.5 + 2 / 128), n


def work(case):
    if case["op"] == "attention":
        H, KV, hd = HEADS[case["heads"]]
        ctx = case["pos"] + 1
        return dict(bytes=2 * KV * hd * ctx * (2 if case["kv_f16"] else 4) + 8 * H * hd, flops=4 * H * hd * ctx)
    m, n, P = MODELS[case["model"]], case["n"], case.get("pos", 0)
    wb, wn = _weights(case["model"])
    att = 8 if case["model"] == "9b-hybrid" else m["L"]
    row = 2 * m["KV"] * m["hd"] * (2 if case["kv_f16"] else 4) * att
    passes = n if case["op"] == "decode" else 1  # one call per step; elsewhere one call has all tokens
    b = passes * wb + row * n + row * P * passes + 4 * m["V"] * passes
    pairs = n * P + n * (n + 1) / 2
    f = 2.0 * (wn - m["V"] * m["D"]) * n + 2.0 * m["V"] * m["D"] * (1 if case["op"] in ("forward", "prefill") else n)
    f += 4.0 * m["H"] * m["hd"] * att * pairs
    if case["model"] == "9b-hybrid":  # the delta rule's state, read and written once; its products
        b += 24 * 2 * (32 * 128 * 128 + 8192 * 3) * 4
        f += 24 * n * 32 * 128 * 128 * 7
    return dict(bytes=b, flops=f)


def tolerance(case):
    # about four times the distance from the 64-bit result (f32 sums; with the fp16 cache, rows that
    # round the other way, over 36, 8 or 80 layers)
    if case["op"] == "attention":
        return dict(rel=2.5e-6)
    if not case["kv_f16"]:
        return dict(rel=4e-5, differ=0.0)
    return dict(rel=5e-3, max=5e-2) if case["model"] == "72b-w4" else dict(rel=4e-4, max=8e-3)


# ------------------------------------------------------------------ the results in 64 bits
class _Archive:
    """Tensors of an archive in 64 bits on the GPU, from its bytes (17408-byte cells: 64 header, 16384
    codes, 960 payload with the metadata first; raw archives: 16384-byte tiles of fp16)."""

    def __init__(self, model):
        m = MODELS[model]
        self.raw = model == "3b-fp16"
        self.stride = 16384 if self.raw else 17408
        self.b = np.memmap(_archive(m["kind"]), dtype=np.uint8, mode="r")

    def _cells(self, rec, n):
        o = 4096 + rec * self.stride
        a = np.ascontiguousarray(self.b[o:o + n * self.stride]).reshape(n, self.stride)
        return torch.from_numpy(a).cuda()

    @staticmethod
    def _view(c, at, n, dt):
        return c[:, at:at + n * dt.itemsize].contiguous().view(dt)

    def matrix(self, rec, rows, cols, tied=False):
        n = -(-rows * cols // (8192 if self.raw else 32768))
        c = self._cells(rec, n)
        if self.raw:
            return c.view(torch.float16).reshape(-1)[:rows * cols].reshape(rows, cols).double()
        code = c[:, 64:64 + 16384]
        w = (torch.stack((code & 15, code >> 4), -1).reshape(n, 256, 128).double() - 8.0)
        w *= self._view(c, 16448 + 48, 256, torch.float16).double()[:, :, None]
        w = w.reshape(n, 32768)
        if cols > 2048:  # flat tiles: single outliers replace weights
            cnt = self._view(c, 16448 + 560, 1, torch.int16).long()
            val = self._view(c, 16448 + 562, 64, torch.float16).double()
            off = self._view(c, 16448 + 690, 64, torch.int16).long() & 0xFFFF
            t, j = torch.nonzero(torch.arange(64, device="cuda")[None, :] < cnt, as_tuple=True)
            w[t, off[t, j]] = val[t, j]
        else:  # 16-row cells: outlier columns, added (replacing in the tied embedding)
            w = w.reshape(n, 16, cols)
            col = self._view(c, 16448 + 816, 8, torch.int16).long()[:, None, :].expand(n, 16, 8)
            val = self._view(c, 16448 + 560, 128, torch.float16).double().reshape(n, 16, 8)
            w = w.scatter(2, col, val) if tied else w.scatter_add(2, col, val)
        return w.reshape(-1)[:rows * cols].reshape(rows, cols)

    def vector(self, rec, n, dt=np.float32):
        o = 4096 + rec * self.stride + (0 if self.raw else 64)
        a = np.frombuffer(self.b[o:o + n * np.dtype(dt).itemsize].tobytes(), dt)
        return a

    def gain(self, rec, n):
        g = self.vector(rec, n)
        return torch.from_numpy((g if np.isfinite(g).all() and g.any() else np.ones(n, np.float32)).astype(np.float64)).cuda()

    def bias(self, rec, n):
        v = self.vector(rec, n)
        return torch.from_numpy(np.where(np.isfinite(v), v, 0).astype(np.float64)).cuda()

    def bf16(self, rec, n):
        v = np.concatenate([self.vector(rec + i, min(8192, n - 8192 * i), np.uint16) for i in range(-(-n // 8192))])
        return torch.from_numpy((v.astype(np.uint32) << 16).view(np.float32).astype(np.float64)).cuda()

    def embed(self, toks, D):
        rows = []
        for t in toks.tolist():
            if self.raw:
                o = 4096 + t * D * 2
                rows.append(np.frombuffer(self.b[o:o + 2 * D].tobytes(), np.float16).astype(np.float64))
                continue
            o = 4096 + t // 16 * self.stride
            cell, r = self.b[o:o + self.stride], t % 16
            code = np.asarray(self.b[o + 64 + r * (D // 2):o + 64 + (r + 1) * (D // 2)])
            w = np.stack((code & 15, code >> 4), -1).reshape(-1).astype(np.float64) - 8.0
            pay = cell[16448:].tobytes()
            if D > 2048:  # one scale and bias per tile, rows running past the cell
                sc, bi = np.frombuffer(pay, np.float32, 2, 32)
                rows.append(w * float(sc) + float(bi))
                continue
            w *= np.repeat(np.frombuffer(pay, np.float16, 16, 48 + 32 * r).astype(np.float64), 128)
            w[np.frombuffer(pay, np.uint16, 8, 816)] = np.frombuffer(pay, np.float16, 8, 560 + 16 * r)
            rows.append(w)
        return torch.from_numpy(np.stack(rows)).cuda()


def _map(model, l):
    """First records of layer l's tensors (the archive layouts of the reference's tensor maps)."""
    if model == "3b-fp16":
        b = 37984 + l * 9413
        return dict(n1=b, q=b + 1, qb=b + 513, k=b + 514, kb=b + 578, v=b + 579, vb=b + 643, o=b + 644, n2=b + 1156,
                    g=b + 1157, u=b + 3909, d=b + 6661)
    if model == "72b-w4":
        b = 38016 + l * 26789
        return dict(n1=b, q=b + 1, qb=b + 2049, k=b + 2050, kb=b + 2306, v=b + 2307, vb=b + 2563, o=b + 2564,
                    n2=b + 4612, g=b + 4613, u=b + 12005, d=b + 19397)
    if model == "9b-hybrid":
        b = 62080 + sum(12804 if i % 4 == 3 else 13337 for i in range(l))
        r = dict(n1=b, q=b + 1, k=b + 2049, v=b + 2305, o=b + 2561, qn=b + 3585, kn=b + 3586, n2=b + 3587)
        if l % 4 != 3:
            r = dict(n1=b, qkv=b + 1, z=b + 2049, a=b + 3073, b=b + 3081, conv=b + 3089, alog=b + 3093, dt=b + 3094,
                     ln=b + 3095, o=b + 3096, n2=b + 4120)
        return dict(r, g=r["n2"] + 1, u=r["n2"] + 3073, d=r["n2"] + 6145)
    # the 3B cell archive: blocks of 2357 records in an irregular order, layer 21's down projection apart
    if l == 21:
        b = 42494
        return dict(n1=b, g=b + 1, u=b + 689, n2=b + 1377, kb=b + 1378, k=b + 1379, o=b + 1395, qb=b + 1523, q=b + 1524,
                    vb=b + 1652, v=b + 1653, d=60662)
    first = {0: 9496, 1: 11853, 2: 37780, 20: 40137}
    b = first.get(l) or (44163 + 2357 * (l - 3) if l < 10 else 14210 + 2357 * (l - 10) if l < 20 else 61350 + 2357 * (l - 22))
    return dict(n1=b, d=b + 1, g=b + 689, u=b + 1377, n2=b + 2065, kb=b + 2066, k=b + 2067, o=b + 2083, qb=b + 2211,
                q=b + 2212, vb=b + 2340, v=b + 2341)


_TAIL = {"3b-w4": (94348, 0), "3b-fp16": (376852, 0), "9b-hybrid": (484600, 484601), "72b-w4": (2181136, 2181137)}


def _rms(x, g, eps=float(np.float32(1e-6))):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * g


def _rope(x, n, rot):
    """Rotary embedding of [n][heads][hd] at positions 0..n-1 over the first `rot` dims, pairs (i, i + rot/2);
    the angles are the 32-bit ones that the model is defined with."""
    i = np.arange(rot // 2, dtype=np.float32)
    f = np.float32(1.0) / np.power(np.float32(1e6), np.float32(2.0) * i / np.float32(rot))
    a = torch.from_numpy((np.arange(n, dtype=np.float32)[:, None] * f[None]).astype(np.float64)).cuda()[:, None]
    c, s = a.cos(), a.sin()
    x0, x1 = x[..., :rot // 2], x[..., rot // 2:rot]
    return torch.cat((x0 * c - x1 * s, x0 * s + x1 * c, x[..., rot:]), -1)


def _attend(q, k, v):
    """Causal attention of [n][H][hd] over [n][KV][hd] in blocks of queries."""
    n, H, hd = q.shape
    KV = k.shape[1]
    out = torch.empty_like(q)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    for a in range(0, n, 512):
        z = min(n, a + 512)
        for h in range(H):
            s = q[a:z, h] @ kt[h // (H // KV)] / math.sqrt(hd)
            s.masked_fill_(torch.arange(n, device="cuda")[None] > torch.arange(a, z, device="cuda")[:, None], -math.inf)
            out[a:z, h] = s.softmax(-1) @ vt[h // (H // KV)]
    return out


def _delta_layer(A, r, x):
    """A gated DeltaNet layer over positions 0..n-1 of normalised inputs x, from an empty state."""
    n, D = x.shape
    silu = torch.nn.functional.silu
    mix, z = x @ A.matrix(r["qkv"], 8192, D).T, (x @ A.matrix(r["z"], 4096, D).T).reshape(n, 32, 128)
    w = A.bf16(r["conv"], 8192 * 4).reshape(8192, 4)
    pad = torch.cat((torch.zeros(3, 8192, dtype=torch.float64, device="cuda"), mix))
    mix = silu(sum(pad[t:t + n] * w[:, t] for t in range(4)))
    q, k, v = mix[:, :2048].reshape(n, 16, 128), mix[:, 2048:4096].reshape(n, 16, 128), mix[:, 4096:].reshape(n, 32, 128)
    unit = lambda t: t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6)  # noqa: E731
    q = unit(q).repeat_interleave(2, 1) / math.sqrt(128)
    k = unit(k).repeat_interleave(2, 1)
    beta = (x @ A.matrix(r["b"], 32, D).T).sigmoid()
    step = torch.nn.functional.softplus(x @ A.matrix(r["a"], 32, D).T + A.bf16(r["dt"], 32))
    decay = (-A.bf16(r["alog"], 32).exp() * step).exp()
    S = torch.zeros(32, 128, 128, dtype=torch.float64, device="cuda")
    o = torch.empty(n, 32, 128, dtype=torch.float64, device="cuda")
    for t in range(n):
        S = S * decay[t][:, None, None]
        d = (v[t] - (S * k[t][:, :, None]).sum(1)) * beta[t][:, None]
        S = S + k[t][:, :, None] * d[:, None]
        o[t] = (S * q[t][:, :, None]).sum(1)
    return (_rms(o, A.bf16(r["ln"], 128)) * silu(z)).reshape(n, 4096)


def _model64(model, toks, kv_f16, keep):
    """Logits of the last `keep` of positions 0..n-1."""
    m, A, n = MODELS[model], _Archive(model), len(toks)
    D, I, H, KV, hd, hyb = m["D"], m["I"], m["H"], m["KV"], m["hd"], model == "9b-hybrid"
    cache = (lambda t: t.half().double()) if kv_f16 else (lambda t: t)
    h = A.embed(toks, D)
    for l in range(m["L"]):
        r = _map(model, l)
        x = _rms(h, A.gain(r["n1"], D))
        if "qkv" in r:
            y = _delta_layer(A, r, x)
        else:
            lin = lambda w, b, rows: x @ A.matrix(r[w], rows, D).T + (A.bias(r[b], rows) if b in r else 0)  # noqa: E731
            q, k = lin("q", "qb", 8192 if hyb else D).reshape(n, H, -1), lin("k", "kb", KV * hd).reshape(n, KV, hd)
            v = lin("v", "vb", KV * hd).reshape(n, KV, hd)
            if hyb:  # per head 256 query values, then 256 output gates
                q, gate = q[..., :hd], q[..., hd:]
                q, k = _rms(q, A.bf16(r["qn"], hd)), _rms(k, A.bf16(r["kn"], hd))
            rot = 64 if hyb else hd
            y = _attend(_rope(q, n, rot), cache(_rope(k, n, rot)), cache(v))
            y = (y * gate.sigmoid() if hyb else y).reshape(n, H * hd)
        h = h + y @ A.matrix(r["o"], D, H * hd).T
        x = _rms(h, A.gain(r["n2"], D))
        a = torch.nn.functional.silu(x @ A.matrix(r["g"], I, D).T) * (x @ A.matrix(r["u"], I, D).T)
        h = h + a @ A.matrix(r["d"], D, I).T
    norm, head = _TAIL[model]
    return _rms(h[-keep:], A.gain(norm, D)) @ A.matrix(head, m["V"], D, tied=head == 0).T


def exact(case, seed):
    if case["op"] == "attention":
        q, k, v = _attention_inputs(case, seed)
        H, KV, hd = HEADS[case["heads"]]
        ctx = case["pos"] + 1
        k, v = k[:, :ctx].double(), v[:, :ctx].double()
        s = torch.matmul(q.double().reshape(KV, H // KV, hd), k.transpose(1, 2).contiguous()) / math.sqrt(hd)
        return torch.matmul(s.softmax(-1), v).reshape(H, hd)
    model, n, P = case["model"], case["n"], case.get("pos", 0)
    if model == "72b-w4" and P + n > 350:  # (the whole model in 64 bits over that many positions: too long)
        return None
    toks = _tokens(model, n, seed + 1000003)
    if P:
        toks = np.concatenate((_tokens(model, MODELS[model]["rows"], 7)[:P], toks))
    y = _model64(model, toks, case["kv_f16"], n if case["op"] == "decode" else 1)
    if case["op"] == "decode":
        return [y[i] for i in range(n)]
    return [y[0], None] if case["op"] == "verify" and not case["kv_f16"] else [y[0]]
