"""The work that this library's users have it do, as cases that can be timed.

A case is one pass through the public entry points of welvet_amd: the Dense
projections of a decode step (one token, or a batch of sequences), the int8
path of the narrow DTypes, the LM head called on host buffers, Dense's
forward and backward over a training batch, the prefill products of a prompt,
and the decoder's own generate and prefill calls. Widths are those of
bench.py's workloads and of the tests (hidden 4096, FFN 14336, KV 1024, vocab
32000; 2560 x 6912 for the ternary layers), token counts go from one row to
the 2047 tokens that the 2048-position cache takes, ragged ones among them.

prepare() packs N(0, 0.02) weights into the reference's block formats on the
GPU (the same rules as quant.Pack: absmax or min/max scales per block, 8-bit
sub-scales per super-block) and uploads them, as a loader does with the bytes
of a checkpoint. exact() decodes the same bytes' fields in float64 torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import welvet_amd as wv
from welvet_amd.decode import Config, Decoder

SIGMA = 0.02  # of the weights, as in the bench workloads
BITS = {"Q4_0": 5.0, "Q8_0": 9.0, "Q4_K": 5.25, "Q6_K": 6.75, "NativeTernary": 2.0}  # stored bits per weight
FMTS = ("Q4_K", "Q6_K", "Q8_0", "Q4_0")


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # A decode step's attention projections: Q, K, V on one row, O on another (grouped-query, 8 KV heads).
        # The smallest calls of a token: launches and latency count as much as bytes.
        dict(name="decode_qkvo", kind="attn", fmt="Q4_K", hidden=4096, kv=1024, batch=1),
        # A decode step's SwiGLU: gate with its SiLU, up, down. Three quarters of the bytes of a token.
        dict(name="decode_mlp", kind="mlp", fmt="Q4_K", hidden=4096, ffn=14336, batch=1),
        # The LM head on host buffers (MatVecPackedBlob), what a Go caller does after its last norm.
        dict(name="decode_head", kind="head", fmt="Q6_K", rows=32000, cols=4096),
        # A BitNet layer's projections: ternary codes, activations quantized to int8, exact int32 sums.
        dict(name="ternary_mlp", kind="ternary", hidden=2560, ffn=6912, batch=1),
        # The SwiGLU of a decode step that serves 8 sequences at once, at the precision of the one-row path.
        dict(name="batch8_mlp", kind="mlp", fmt="Q4_K", hidden=4096, ffn=14336, batch=8),
        # Dense.Forward of a training batch: 32 rows, bias, GELU.
        dict(name="forward32", kind="dense", fmt="Q8_0", rows=4096, cols=4096, batch=32, act="gelu", block=False),
        # Dense's input gradient of a small batch: gx += W^T gy for 8 rows.
        dict(name="grad8", kind="grad", fmt="Q4_K", rows=14336, cols=4096, batch=8),
        # A prompt's projections: one short block, a ragged one of the wide-K shape in a 6-bit format, and the
        # longest prompt of a 2048-position cache through Dense's block entry with bias and SiLU.
        dict(name="block32", kind="block", fmt="Q4_K", rows=14336, cols=4096, batch=32),
        dict(name="block509", kind="block", fmt="Q6_K", rows=4096, cols=14336, batch=509),
        dict(name="block2047", kind="dense", fmt="Q4_K", rows=14336, cols=4096, batch=2047, act="silu", block=True),
        # Greedy decoding of 8 tokens at the end of a 2048-position cache (4 of the 32 layers of the bench's model).
        dict(name="generate", kind="generate", fmt="Q4_K", layers=4, hidden=4096, heads=32, kv_heads=8, hd=128,
             ffn=14336, vocab=32000, seq=2048, pos=2032, steps=8),
        # A 512-token prompt through the same layers: the projections, causal attention, the last row's logits.
        dict(name="prompt512", kind="prompt", fmt="Q4_K", layers=4, hidden=4096, heads=32, kv_heads=8, hd=128,
             ffn=14336, vocab=32000, seq=2048, tokens=512),
    ]


def _log_int(rng, lo, hi, step=1):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def _rows(rng, lo, hi):
    """Output rows: whole 64-row groups or not."""
    return _log_int(rng, lo, hi, rng.choice((64, 64, 1)))


def draw(rng):
    kind = rng.choice(("attn", "mlp", "mlp", "head", "ternary", "dense", "dense", "grad", "block", "block", "generate",
                       "prompt"))
    fmt = rng.choice(FMTS)
    if kind == "attn":
        hidden = _log_int(rng, 1024, 5120, 256)
        return dict(kind=kind, fmt=fmt, hidden=hidden, kv=rng.choice((hidden, hidden // 4, 512)),
                    batch=_log_int(rng, 1, 32))
    if kind == "mlp":
        return dict(kind=kind, fmt=fmt, hidden=_log_int(rng, 1024, 5120, 256), ffn=_log_int(rng, 2560, 14336, 256),
                    batch=rng.choice((1, 1, _log_int(rng, 2, 32))))
    if kind == "head":
        return dict(kind=kind, fmt=fmt, rows=_rows(rng, 2000, 32000), cols=_log_int(rng, 1024, 5120, 256))
    if kind == "ternary":
        return dict(kind=kind, hidden=_log_int(rng, 1024, 4096, 256), ffn=_log_int(rng, 2560, 14336, 256),
                    batch=rng.choice((1, 1, _log_int(rng, 2, 16))))
    if kind == "dense":
        block = rng.random() < 0.5
        cols = _log_int(rng, 512, 14336, 256)
        if fmt in ("Q8_0", "Q4_0") and rng.random() < 0.25:
            cols = _log_int(rng, 512, 6144, 32)  # 32-column blocks, not whole super-blocks
        return dict(kind=kind, fmt=fmt, rows=_rows(rng, 1024, 14336), cols=cols,
                    batch=_log_int(rng, 2, 512 if block and cols % 256 == 0 else 48),
                    act=rng.choice(("linear", "relu", "silu", "gelu")), block=block)
    if kind == "grad":
        return dict(kind=kind, fmt=fmt, rows=_rows(rng, 1024, 14336), cols=_log_int(rng, 1024, 14336, 256),
                    batch=_log_int(rng, 1, 32))
    if kind == "block":
        return dict(kind=kind, fmt=fmt, rows=_rows(rng, 1024, 14336), cols=_log_int(rng, 1024, 14336, 256),
                    batch=_log_int(rng, 2, 2047))
    hd = rng.choice((64, 128))
    kv_heads = rng.choice((4, 8))
    heads = kv_heads * rng.choice((1, 2, 4))
    base = dict(kind=kind, fmt=fmt, layers=2, hidden=_log_int(rng, 1024, 4096, 256), heads=heads, kv_heads=kv_heads,
                hd=hd, ffn=_log_int(rng, 2560, 14336, 256), vocab=_log_int(rng, 4000, 32000))
    if kind == "generate":
        base.update(seq=2048, pos=_log_int(rng, 16, 2040), steps=8)
    else:
        base.update(seq=2048, tokens=_log_int(rng, 9, 2047))
    return base


# ------------------------------------------------------------- the weights

class _Weights:
    """One projection: the packed bytes (host) and the float64 decode of the same fields."""

    def __init__(self, gen, fmt, rows, cols):
        self.fmt, self.rows, self.cols = fmt, rows, cols
        if fmt == "NativeTernary":  # per-tensor absmean scale, P(0) about 1/3
            self.q = torch.randint(0, 3, (rows, cols), generator=gen, device="cuda", dtype=torch.uint8)
            self.scale = SIGMA
            return
        w = torch.randn(rows * cols, generator=gen, device="cuda") * SIGMA
        if fmt in ("Q4_0", "Q8_0"):
            b = w.view(-1, 32)
            top = 7.0 if fmt == "Q4_0" else 127.0
            self.scale = b.abs().amax(1, keepdim=True) / top
            self.q = torch.round(b / self.scale).clamp_(-8.0 if fmt == "Q4_0" else -127.0, top).to(torch.int8)
            return
        b = w.view(-1, 16, 16)  # super-blocks of 16 groups of 16
        if fmt == "Q4_K":
            lo, hi = b.amin(2), b.amax(2)
            gs = (hi - lo) / 15.0
            self.q = torch.round((b - lo[..., None]) / gs[..., None]).clamp_(0, 15).to(torch.uint8)
            self.dmin = lo.abs().amax(1)
            self.m = torch.round(lo / self.dmin[:, None] * 127.0).clamp_(-127, 127).to(torch.int8)
        else:  # Q6_K
            gs = b.abs().amax(2) / 32.0
            self.q = (torch.round(b / gs[..., None]) + 32).clamp_(0, 63).to(torch.uint8)
            self.dmin = torch.zeros(b.shape[0], device="cuda")
        self.d = gs.amax(1)
        self.u = torch.round(gs / self.d[:, None] * 255.0).clamp_(0, 255).to(torch.uint8)

    def packed(self):
        f = lambda t: t.contiguous().view(torch.uint8)  # noqa: E731  (the little-endian bytes of a tensor)
        if self.fmt == "NativeTernary":
            q = self.q.view(-1, 4)
            raw = q[:, 0] | q[:, 1] << 2 | q[:, 2] << 4 | q[:, 3] << 6
            return wv.PackedBlob(self.fmt, self.rows, self.cols, raw.cpu().numpy(), tensor_scale=self.scale)
        if self.fmt == "Q8_0":
            raw = torch.cat((f(self.scale), f(self.q)), 1)
        elif self.fmt == "Q4_0":
            q = f(self.q) & 15
            raw = torch.cat((f(self.scale), q[:, 0::2] | q[:, 1::2] << 4), 1)
        else:
            q = self.q.view(-1, 256)
            if self.fmt == "Q4_K":
                codes = q[:, 0::2] | q[:, 1::2] << 4
                raw = torch.cat((f(self.d[:, None]), f(self.dmin[:, None]), self.u, f(self.m), codes), 1)
            else:  # a stream of 6-bit codes, four to three bytes
                a, b, c, e = (q[:, k::4] for k in range(4))
                codes = torch.stack((a | b << 6, b >> 2 | c << 4, c >> 4 | e << 2), 2).reshape(-1, 192)
                raw = torch.cat((f(self.d[:, None]), f(self.dmin[:, None]), self.u, codes), 1)
        return wv.PackedBlob(self.fmt, self.rows, self.cols, raw.reshape(-1).cpu().numpy(),
                             block_weights=wv.pack_sizes(self.fmt, self.rows, self.cols)[4])

    def upload(self):
        return wv.upload(self.packed())

    def f64(self):
        if self.fmt == "NativeTernary":
            return (self.q.double() - 1.0) * float(np.float32(self.scale))
        if self.fmt in ("Q4_0", "Q8_0"):
            w = self.q.double() * self.scale.double()
        else:
            sc = self.d.double()[:, None] * self.u.double().clamp_(min=1) / 255.0  # sub-scale 0 decodes as d/255
            if self.fmt == "Q4_K":
                mn = self.dmin.double()[:, None] * self.m.double() / 127.0
                w = self.q.double() * sc[..., None] + mn[..., None]
            else:
                w = (self.q.double() - 32.0) * sc[..., None]
        return w.reshape(self.rows, self.cols)


def _gen(seed, part):
    return torch.Generator("cuda").manual_seed(seed * 1009 + part)


def _shapes(c):
    """(rows, cols) of the case's projections, in the order that run() calls them."""
    k = c["kind"]
    if k == "attn":
        return [(c["hidden"], c["hidden"]), (c["kv"], c["hidden"]), (c["kv"], c["hidden"]), (c["hidden"], c["hidden"])]
    if k in ("mlp", "ternary"):
        return [(c["ffn"], c["hidden"]), (c["ffn"], c["hidden"]), (c["hidden"], c["ffn"])]
    if k in ("generate", "prompt"):
        q, kv, h, f = c["heads"] * c["hd"], c["kv_heads"] * c["hd"], c["hidden"], c["ffn"]
        return [(q, h), (kv, h), (kv, h), (h, q), (f, h), (f, h), (h, f)] * c["layers"] + [(c["vocab"], h)]
    return [(c["rows"], c["cols"])]


def _fmt(c):
    return c.get("fmt", "NativeTernary")


def _weights(c, seed, i):
    rows, cols = _shapes(c)[i]
    return _Weights(_gen(seed, 10 + i), _fmt(c), rows, cols)


def _input(seed, part, *shape):
    return torch.randn(*shape, generator=_gen(seed, 500 + part), device="cuda")


def _norms(c, seed):
    """Gammas of 2 norms per layer and of the final one, about 1."""
    return 1.0 + 0.1 * _input(seed, 0, 2 * c["layers"] + 1, c["hidden"])


def _cache(c, seed, layer):
    return _input(seed, 100 + layer, 2, c["pos"], c["kv_heads"] * c["hd"])


def _tokens(c, seed):
    n = c["tokens"] if c["kind"] == "prompt" else 1
    return torch.randint(0, c["vocab"], (n,), generator=_gen(seed, 900), device="cuda")


# ------------------------------------------------------- the state and a pass

_stream = None


def _the_stream():
    """The program's stream: every device-pointer call and torch operation of a pass goes there."""
    global _stream
    if _stream is None:
        wv.init(0)
        _stream = torch.cuda.Stream()
    return _stream


def prepare(case, seed):
    c, k = case, case["kind"]
    st = _the_stream()
    s = {"case": c, "stream": st, "sh": st.cuda_stream}
    dev = dict(device="cuda", dtype=torch.float32)
    if k in ("generate", "prompt"):
        cfg = Config(n_layers=c["layers"], hidden=c["hidden"], n_heads=c["heads"], n_kv_heads=c["kv_heads"],
                     head_dim=c["hd"], ffn=c["ffn"], vocab=c["vocab"], max_seq=c["seq"])
        dec = Decoder(cfg)
        norms = _norms(c, seed).cpu().numpy()
        for i in range(c["layers"]):
            blobs = [_weights(c, seed, 7 * i + j).upload() for j in range(7)]
            dec.set_layer(i, blobs, norms[2 * i], norms[2 * i + 1])
            if k == "generate":
                kv = _cache(c, seed, i).cpu().numpy()
                dec.set_kv(i, 0, kv[0], kv[1])
        head = _weights(c, seed, 7 * c["layers"]).upload()
        dec.set_output(head, norms[-1], _input(seed, 1, c["vocab"], c["hidden"]).cpu().numpy())
        if k == "generate":
            dec.use_graph(True)
        s.update(dec=dec, ids=_tokens(c, seed).cpu().numpy().astype(np.int32))
        torch.cuda.synchronize()
        return s
    s["blobs"] = [_weights(c, seed, i).upload() for i in range(len(_shapes(c)))]
    if k == "head":
        s["x"] = _input(seed, 0, c["cols"]).cpu().numpy()
        s["y"] = np.zeros(c["rows"], np.float32)
        return s
    b = c["batch"]
    if k == "attn":
        s["x"], s["a"] = _input(seed, 0, b, c["hidden"]), _input(seed, 1, b, c["hidden"])
        s["y"] = [torch.zeros(b, r, **dev) for r, _ in _shapes(c)]
    elif k in ("mlp", "ternary"):
        s["x"], s["h"] = _input(seed, 0, b, c["hidden"]), _input(seed, 1, b, c["ffn"])
        s["pre"], s["gate"], s["up"] = (torch.zeros(b, c["ffn"], **dev) for _ in range(3))
        s["y"] = torch.zeros(b, c["hidden"], **dev)
    elif k == "dense":
        s["x"] = _input(seed, 0, b, c["cols"])
        s["bias"] = _input(seed, 1, c["rows"]).double() * 0.1
        s["pre"], s["post"] = torch.zeros(b, c["rows"], **dev), torch.zeros(b, c["rows"], **dev)
    elif k == "grad":
        s["gy"] = _input(seed, 0, b, c["rows"])
        s["gx"] = torch.zeros(b, c["cols"], **dev)
    else:  # block
        s["x"] = _input(seed, 0, b, c["cols"])
        s["y"] = torch.zeros(b, c["rows"], **dev)
    torch.cuda.synchronize()
    return s


def run(state):
    s, c, sh = state, state["case"], state["sh"]
    k = c["kind"]
    if k == "generate":
        toks, logits = s["dec"].generate(int(s["ids"][0]), c["pos"], c["steps"], want_logits=True)
        return {"tokens": toks, "logits": logits}
    if k == "prompt":
        _, logits = s["dec"].prefill(s["ids"], 0, want_logits=True)
        return {"logits": logits}
    w = s["blobs"]
    if k == "head":
        w[0].matvec_packed_blob(s["x"], s["y"])
        return s["y"]
    b = c["batch"]
    if k == "attn":
        x, y = s["x"].data_ptr(), s["y"]
        for i in range(3):
            w[i].matvec_dev(x, y[i].data_ptr(), b, sh)
        w[3].matvec_dev(s["a"].data_ptr(), y[3].data_ptr(), b, sh)
        return y
    if k == "mlp":
        x = s["x"].data_ptr()
        w[0].dense_forward_dev(x, s["pre"].data_ptr(), s["gate"].data_ptr(), b, None, "silu", sh)
        w[1].matvec_dev(x, s["up"].data_ptr(), b, sh)
        with torch.cuda.stream(s["stream"]):
            torch.mul(s["gate"], s["up"], out=s["h"])
        w[2].matvec_dev(s["h"].data_ptr(), s["y"].data_ptr(), b, sh)
        return {"gate": s["gate"], "up": s["up"], "y": s["y"]}
    if k == "ternary":  # each projection on its own row: its int8 rounding is not the next one's input
        x = s["x"].data_ptr()
        w[0].matvec_dev(x, s["gate"].data_ptr(), b, sh)
        w[1].matvec_dev(x, s["up"].data_ptr(), b, sh)
        w[2].matvec_dev(s["h"].data_ptr(), s["y"].data_ptr(), b, sh)
        return {"gate": s["gate"], "up": s["up"], "y": s["y"]}
    if k == "dense":
        if c["block"]:
            wv.check(wv.lib().wv_dense_forward_block_dev(w[0].handle, s["x"].data_ptr(), s["pre"].data_ptr(),
                                                         s["post"].data_ptr(), b, s["bias"].data_ptr(),
                                                         wv.ACT[c["act"]], sh))
        else:
            w[0].dense_forward_dev(s["x"].data_ptr(), s["pre"].data_ptr(), s["post"].data_ptr(), b,
                                   s["bias"].data_ptr(), c["act"], sh)
        return {"pre": s["pre"], "post": s["post"]}
    if k == "grad":
        with torch.cuda.stream(s["stream"]):
            s["gx"].zero_()
        w[0].matvec_t_dev(s["gy"].data_ptr(), s["gx"].data_ptr(), b, sh)
        return s["gx"]
    w[0].matmul_dev(s["x"].data_ptr(), s["y"].data_ptr(), b, sh)
    return s["y"]


# -------------------------------------------------- what a pass cannot avoid

def work(case):
    c, k = case, case["kind"]
    sh = _shapes(c)
    bits = BITS[_fmt(c)]
    params = sum(r * n for r, n in sh)
    if k in ("generate", "prompt"):
        head = c["vocab"] * c["hidden"]
        kv_row = 2 * c["kv_heads"] * c["hd"] * 4  # bytes of a position's K and V
        q = c["heads"] * c["hd"]
        if k == "generate":
            n, past = c["steps"], c["pos"] + c["steps"] / 2
            return {"bytes": n * (params * bits / 8 + c["layers"] * kv_row * past + 4 * (c["vocab"] + c["hidden"])),
                    "flops": n * (2.0 * params + c["layers"] * 4.0 * q * past)}
        t = c["tokens"]
        return {"bytes": params * bits / 8 + c["layers"] * kv_row * t + 4 * t * c["hidden"] + 4 * c["vocab"],
                "flops": 2.0 * t * (params - head) + 2.0 * head + c["layers"] * 2.0 * q * t * (t + 1)}
    b = c.get("batch", 1)
    outs = 2 if k == "dense" else 1
    rows_io = sum(n + outs * r for r, n in sh)
    if k == "grad":
        rows_io = sum(2 * n + r for r, n in sh)  # gx is read and written
    return {"bytes": params * bits / 8 + 4.0 * b * rows_io, "flops": 2.0 * b * params}


def tolerance(case):
    """About four times the distance from exact() that each path shows (in brackets)."""
    k = case["kind"]
    if k == "prompt":  # fp16 products through the layers [2.3e-3]
        return {"rel": 8e-3, "max": 4e-2}
    if k == "block" or (k == "dense" and case["block"]):  # fp16 operands, f32 sums [6.6e-4]
        return {"rel": 2.5e-3, "max": 1.5e-2}
    if k == "generate":  # f32 through the layers [2.7e-6]
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}
    if k == "ternary":  # exact integer sums, two f32 scales [4e-8]
        return {"rel": 2e-7, "max": 1e-6}
    return {"rel": 5e-6, "max": 5e-5}  # f32 operands and sums [1.4e-6]


# ------------------------------------------------------- the same in 64 bits

def _act(v, act):
    if act == "relu":
        return v.clamp(min=0)
    if act == "silu":
        return v * torch.sigmoid(v)
    if act == "gelu":  # the tanh form
        return 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v ** 3)))
    return v


def _ternary(w, x):
    """quantizeActsI8 (f32 scale and quotient, ties away from zero), integer sums, the two scales."""
    s = x.abs().amax(1, keepdim=True) / 127.0
    t = (x / s).double()
    q = torch.sign(t) * torch.floor(t.abs() + 0.5)
    return (q @ (w.q.double() - 1.0).T) * s.double() * float(np.float32(w.scale))


def _norm(x, gamma, eps=1e-5):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + eps) * gamma.double()


def _rope(v, pos, hd, theta=5e5):
    half = hd // 2
    d = torch.arange(half, device="cuda", dtype=torch.float64)
    a = pos.double()[:, None] / theta ** (2.0 * d / hd)
    co, si = torch.cos(a)[:, None], torch.sin(a)[:, None]
    v = v.reshape(v.shape[0], -1, hd)
    x, y = v[..., :half], v[..., half:]
    return torch.cat((x * co - y * si, x * si + y * co), 2)


def _forward(c, seed, layers, ids, pos0, caches):
    """The decoder's layers over the rows of `ids` at pos0..; caches[i] = (K, V) of the positions before them."""
    hd, g = c["hd"], c["heads"] // c["kv_heads"]
    norms = _norms(c, seed)
    h = _input(seed, 1, c["vocab"], c["hidden"])[ids].double()
    pos = torch.arange(pos0, pos0 + len(ids), device="cuda")
    for i in range(c["layers"]):
        n = _norm(h, norms[2 * i])
        w = lambda j: layers(7 * i + j)  # noqa: E731
        q = _rope(n @ w(0).T, pos, hd)
        kk, vv = _rope(n @ w(1).T, pos, hd), (n @ w(2).T).reshape(len(ids), -1, hd)
        if caches[i] is not None:
            kk, vv = torch.cat((caches[i][0], kk)), torch.cat((caches[i][1], vv))
        caches[i] = (kk, vv)
        mask = torch.arange(len(kk), device="cuda")[None, :] > pos[:, None]
        out = torch.empty_like(q)
        for a in range(c["heads"]):
            sc = (q[:, a] @ kk[:, a // g].T) / math.sqrt(hd)
            out[:, a] = torch.softmax(sc.masked_fill(mask, -math.inf), 1) @ vv[:, a // g]
        h = h + out.reshape(len(ids), -1) @ w(3).T
        n = _norm(h, norms[2 * i + 1])
        h = h + (_act(n @ w(4).T, "silu") * (n @ w(5).T)) @ w(6).T
    return (_norm(h[-1:], norms[-1]) @ layers(7 * c["layers"]).T)[0]


def exact(case, seed):
    c, k = case, case["kind"]
    if k == "prompt":
        return {"logits": _forward(c, seed, lambda i: _weights(c, seed, i).f64(), _tokens(c, seed), 0,
                                   [None] * c["layers"])}
    if k == "generate":
        kept = {}

        def layers(i):
            if i not in kept:
                kept[i] = _weights(c, seed, i).f64()
            return kept[i]
        caches = []
        for i in range(c["layers"]):
            kv = _cache(c, seed, i).double().reshape(2, c["pos"], c["kv_heads"], c["hd"])
            caches.append((kv[0], kv[1]))
        ids, toks = _tokens(c, seed), []
        for n in range(c["steps"]):
            logits = _forward(c, seed, layers, ids, c["pos"] + n, caches)
            ids = logits.argmax().reshape(1)
            toks.append(int(ids[0]))
        return {"tokens": np.array(toks, np.int32), "logits": logits}
    if k == "head":
        return _weights(c, seed, 0).f64() @ _input(seed, 0, c["cols"]).double()
    b = c["batch"]
    if k == "attn":
        x, a = _input(seed, 0, b, c["hidden"]).double(), _input(seed, 1, b, c["hidden"]).double()
        return [(a if i == 3 else x) @ _weights(c, seed, i).f64().T for i in range(4)]
    if k == "ternary":
        x, h = _input(seed, 0, b, c["hidden"]), _input(seed, 1, b, c["ffn"])
        return {n: _ternary(_weights(c, seed, i), h if i == 2 else x) for i, n in enumerate(("gate", "up", "y"))}
    if k == "mlp":
        x = _input(seed, 0, b, c["hidden"]).double()
        gate = _act(x @ _weights(c, seed, 0).f64().T, "silu")
        up = x @ _weights(c, seed, 1).f64().T
        return {"gate": gate, "up": up, "y": (gate * up) @ _weights(c, seed, 2).f64().T}
    if k == "grad":
        return _input(seed, 0, b, c["rows"]).double() @ _weights(c, seed, 0).f64()
    y = _input(seed, 0, b, c["cols"]).double() @ _weights(c, seed, 0).f64().T
    if k == "dense":
        pre = y + _input(seed, 1, c["rows"]).double() * 0.1
        return {"pre": pre, "post": _act(pre, c["act"])}
    return y
