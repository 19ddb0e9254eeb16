"""The workloads this framework is timed on, with their inputs, their outputs
in 64 bits and their tolerances.

The cases are the calls a GGUF / bitsandbytes inference engine makes on one
GPU: decode GEMVs from the smallest projection to the vocabulary head, decode
steps of whole layers at short and long contexts, the prefill GEMMs from 16 to
2048 tokens, the first half of a prefill block, and the expansion of a packed
weight.  Shapes are those of the repository's own configurations (Llama-3-8B
and Qwen2.5-0.5B layers); ``draw`` spreads sizes, block formats and element
types over the ranges in between.

Weights are made on the device directly in their packed layouts: quants of a
rounded normal distribution and scales that vary from block to block, so that
the decoded weights are about N(0, 0.02^2) as trained projections are.
``_chunks`` makes the quants and scales once; packing them gives the call's
operand and the closed form of the format gives the values ``exact`` uses.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from cima_amd import gguf
from cima_amd.decoder import DecoderConfig, DeviceDecoder, HostModel, PROJECTIONS
from cima_amd.hip import HipCtx
from cima_amd.nf4 import NF4_CODE, HostNf4, Nf4Weight

SIGMA = 0.02          # standard deviation of the weights
SLAB_BYTES = 32 << 20  # the engine's scratch slab
FMT = {t.name: int(t) for t in gguf.DType}
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
IQ4NL = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)

_ctx = None


def _hip() -> HipCtx:
    """The process's context, on torch's current stream as a torch program runs it."""
    global _ctx
    if _ctx is None:
        _ctx = HipCtx(0)
    _ctx.use_torch_stream()
    return _ctx


def _gen(*key) -> torch.Generator:
    g = torch.Generator(device="cuda")
    s = 1469598103934665603
    for v in key:
        s = ((s ^ (int(v) & 0xFFFFFFFF)) * 1099511628211) & 0x7FFFFFFFFFFFFFFF
    g.manual_seed(s)
    return g


def _normal(shape, *key, scale=1.0, mean=0.0, dtype=torch.float32):
    v = torch.randn(shape, generator=_gen(*key), device="cuda", dtype=torch.float32)
    return (v * scale + mean).to(dtype)


# ------------------------------------------------------------ packed weights

def _quants(g, shape, sigma, centre, hi):
    q = torch.randn(shape, generator=g, device="cuda").mul_(sigma).add_(centre).round_().clamp_(0, hi)
    return q.to(torch.uint8)


def _scale(g, shape, mean):
    """f16 block scales within 30% of their mean."""
    return (mean * (0.7 + 0.6 * torch.rand(shape, generator=g, device="cuda"))).to(torch.float16)


def _ints(g, shape, lo, hi):
    return torch.randint(lo, hi + 1, shape, generator=g, device="cuda", dtype=torch.int32)


def _half_bytes(h):
    return h.contiguous().view(torch.uint8).reshape(*h.shape, 2)


def _nibbles(q):
    """[..., 32] quants -> [..., 16] bytes: element j low, element j + 16 high."""
    return (q[..., :16] & 15) | ((q[..., 16:] & 15) << 4)


def _scales_k4(sc, m):
    """Eight 6-bit scales and eight 6-bit mins -> Q4_K / Q5_K's 12 bytes."""
    lo = (sc[..., :4] & 63) | ((sc[..., 4:] >> 4) << 6)
    mid = (m[..., :4] & 63) | ((m[..., 4:] >> 4) << 6)
    hi = (sc[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)
    return torch.cat([lo, mid, hi], -1).to(torch.uint8)


def _bits32(b):
    """[..., 32] zeros and ones -> [..., 4] bytes, bit j of the word = element j."""
    w = torch.tensor([1 << i for i in range(8)], dtype=torch.int32, device=b.device)
    return (b.reshape(*b.shape[:-1], 4, 8).to(torch.int32) * w).sum(-1).to(torch.uint8)


def _blocks32(fmt, g, n, nb):
    """Packed bytes [n, nb, block bytes] and a function giving the values for the 32-element formats."""
    if fmt == "Q8_0":
        d = _scale(g, (n, nb), SIGMA / 42)
        q = torch.randn((n, nb, 32), generator=g, device="cuda").mul_(42).round_().clamp_(-127, 127).to(torch.int8)
        return torch.cat([_half_bytes(d), q.view(torch.uint8)], -1), lambda T: d.to(T)[..., None] * q.to(T)
    bits = 5 if fmt in ("Q5_0", "Q5_1") else 4
    sig, top = (5.8, 31) if bits == 5 else (2.8, 15)
    d = _scale(g, (n, nb), SIGMA / sig)
    mins = fmt in ("Q4_1", "Q5_1")
    q = _quants(g, (n, nb, 32), sig, top / 2 if mins else (top + 1) / 2, top)
    parts = [_half_bytes(d)]
    if mins:
        m = (-(top / 2) * d.float() * (0.9 + 0.2 * torch.rand((n, nb), generator=g, device="cuda"))).to(torch.float16)
        parts.append(_half_bytes(m))
    if bits == 5:
        parts.append(_bits32(q >> 4))
    parts.append(_nibbles(q))
    packed = torch.cat(parts, -1)
    if mins:
        return packed, lambda T: d.to(T)[..., None] * q.to(T) + m.to(T)[..., None]
    return packed, lambda T: d.to(T)[..., None] * (q.to(T) - (16 if bits == 5 else 8))


def _blocks256(fmt, g, n, nb):
    """The same for the 256-element formats."""
    if fmt in ("Q4_K", "Q5_K"):
        sig, top = (2.8, 15) if fmt == "Q4_K" else (5.8, 31)
        d = _scale(g, (n, nb), SIGMA / sig / 44)
        dmin = (d.float() * (top / 2)).to(torch.float16)
        sc = _ints(g, (n, nb, 8), 25, 63)
        m = (sc + _ints(g, (n, nb, 8), -4, 4)).clamp_(0, 63)
        q = _quants(g, (n, nb, 8, 32), sig, top / 2, top)
        parts = [_half_bytes(d), _half_bytes(dmin), _scales_k4(sc, m)]
        if fmt == "Q5_K":
            w = torch.tensor([1 << i for i in range(8)], dtype=torch.int32, device="cuda")
            parts.append(((q >> 4).to(torch.int32) * w[:, None]).sum(-2).to(torch.uint8))
        parts.append(((q[:, :, 0::2] & 15) | ((q[:, :, 1::2] & 15) << 4)).reshape(n, nb, 128))

        def val(T):
            ds, ms = d.to(T)[..., None] * sc.to(T), dmin.to(T)[..., None] * m.to(T)
            return ds[..., None] * q.to(T) - ms[..., None]
        return torch.cat(parts, -1), val
    if fmt == "Q6_K":
        d = _scale(g, (n, nb), SIGMA / 11 / 90)
        sc = _ints(g, (n, nb, 16), 55, 125) * (2 * _ints(g, (n, nb, 16), 0, 1) - 1)
        q = _quants(g, (n, nb, 2, 4, 32), 11, 32, 63)  # half, group, l
        ql = torch.cat([(q[:, :, :, 0] & 15) | ((q[:, :, :, 2] & 15) << 4),
                        (q[:, :, :, 1] & 15) | ((q[:, :, :, 3] & 15) << 4)], -1).reshape(n, nb, 128)
        h = q >> 4
        qh = (h[:, :, :, 0] | (h[:, :, :, 1] << 2) | (h[:, :, :, 2] << 4) | (h[:, :, :, 3] << 6)).reshape(n, nb, 64)
        packed = torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _half_bytes(d)], -1)

        def val(T):
            s = d.to(T)[..., None] * sc.to(T)
            return s[..., None] * (q.to(T).reshape(n, nb, 16, 16) - 32)
        return packed, val
    d = _scale(g, (n, nb), SIGMA / 49 / 22)
    ls = 32 + _ints(g, (n, nb, 8), 12, 31) * (2 * _ints(g, (n, nb, 8), 0, 1) - 1)
    q = _quants(g, (n, nb, 8, 32), 3.2, 7.5, 15)
    two = torch.tensor([1 << (2 * i) for i in range(8)], dtype=torch.int32, device="cuda")
    sh = ((ls >> 4) * two).sum(-1).to(torch.int32)
    shb = torch.stack([sh & 255, sh >> 8], -1).to(torch.uint8)
    sl = ((ls[..., 0::2] & 15) | ((ls[..., 1::2] & 15) << 4)).to(torch.uint8)
    packed = torch.cat([_half_bytes(d), shb, sl, _nibbles(q).reshape(n, nb, 128)], -1)
    code = torch.tensor(IQ4NL, device="cuda")

    def val(T):
        return (d.to(T)[..., None] * (ls - 32).to(T))[..., None] * code.to(T)[q.long()]
    return packed, val


def _nf4_blocks(g, n, nb, bs):
    """bitsandbytes NF4: nibbles (element 2j high), f32 absmax per bs elements."""
    q = _quants(g, (n, nb, bs), 3.3, 7.2, 15)
    a = SIGMA / 0.42 * (0.7 + 0.6 * torch.rand((n, nb), generator=g, device="cuda"))
    packed = (q[..., 0::2] << 4) | q[..., 1::2]
    code = torch.from_numpy(np.asarray(NF4_CODE, np.float32)).cuda()
    return packed, a, lambda T: code.to(T)[q.long()] * a.to(T)[..., None]


def _chunks(fmt, n, k, *key, bs=64):
    """(first row, packed operands, values) over row ranges of an [n, k] weight."""
    step = max(1, (32 << 20) // k)
    for r0 in range(0, n, step):
        r = min(step, n - r0)
        g = _gen(*key, r0, n, k)
        if fmt == "NF4":
            p, a, val = _nf4_blocks(g, r, k // bs, bs)
            yield r0, (p.reshape(-1), a.reshape(-1)), lambda T, v=val, r=r: v(T).reshape(r, k)
        else:
            p, val = (_blocks32 if gguf.block_elems(FMT[fmt]) == 32 else _blocks256)(
                fmt, g, r, k // gguf.block_elems(FMT[fmt]))
            yield r0, p.reshape(-1), lambda T, v=val, r=r: v(T).reshape(r, k)


def _packed(fmt, n, k, *key):
    return torch.cat([p for _, p, _ in _chunks(fmt, n, k, *key)])


def _f16_values(val):
    """The decoded f16 weights (products and sums in f32, one rounding to f16, as the format's decoder)."""
    return val(torch.float32).to(torch.float16)


def _matvec64(fmt, n, k, x, *key, bs=64):
    """W . x in f64, W the format's values unrounded."""
    return torch.cat([v(torch.float64) @ x for _, _, v in _chunks(fmt, n, k, *key, bs=bs)])


def _matmul64(fmt, n, k, x, *key, bs=64):
    """X . W^T in f64 over the f16 operands the prefill contract names: decoded f16 W, X rounded to f16."""
    x = x.to(torch.float16).to(torch.float64)
    return torch.cat([x @ _f16_values(v).to(torch.float64).T for _, _, v in _chunks(fmt, n, k, *key, bs=bs)], 1)


def _row64(fmt, n, k, row, *key):
    """Decoded f16 rows of a table, as f64 (row: a tensor of indices)."""
    out = torch.empty((row.numel(), k), dtype=torch.float64, device="cuda")
    for r0, _, v in _chunks(fmt, n, k, *key):
        r1 = min(n, r0 + max(1, (32 << 20) // k))
        at = (row >= r0) & (row < r1)
        if bool(at.any()):
            out[at] = _f16_values(v).to(torch.float64)[row[at] - r0]
    return out


def _wbytes(fmt, n, k, bs=64):
    return n * k // 2 + n * k // bs * 4 if fmt == "NF4" else n * gguf.row_bytes(FMT[fmt], k)


def _esz(d):
    return 4 if d == "f32" else 2


# --------------------------------------------------------------- the cases

LLAMA8B = dict(hidden=4096, q_heads=32, kv_heads=8, head_dim=128, ffn=14336)
QWEN05B = dict(hidden=896, q_heads=14, kv_heads=2, head_dim=64, ffn=4864)


def listed():
    return [
        # one projection of a 0.5B model: the smallest call, all launch and latency
        dict(name="gemv_q8_0_4864x896", kind="gemv", fmt="Q8_0", n=4864, k=896, act="f16", mode=0),
        # a bitsandbytes checkpoint's decode: the down projection of an 8B layer
        dict(name="gemv_nf4_4096x14336", kind="gemv", fmt="NF4", n=4096, k=14336, act="f16", mode=0),
        # the vocabulary head of an 8B model with its norm and greedy argmax: the largest GEMV
        dict(name="head_q6_k_128256x4096", kind="head", fmt="Q6_K", n=128256, k=4096),
        # four 8B layers of one decode step deep in a long conversation
        dict(name="layers_llama8b_q4_k_ctx8000", kind="decode", model="llama8b", fmt="Q4_K", v_down="Q4_K",
             layers=4, vocab=8192, pos=7999, max_seq=8192, window=0),
        # a whole decode step of a 0.5B model at a medium context
        dict(name="decode_qwen05b_q8_0_ctx2048", kind="decode", model="qwen05b", fmt="Q8_0", v_down="Q8_0",
             layers=24, vocab=151936, pos=2047, max_seq=4096, window=0),
        # the first half of a prefill block: embedding rows, norm, q / k / v projections, RoPE, KV append
        dict(name="prefill_in_q4_k_585", kind="prefill_in", fmt="Q4_K", m=585, vocab=32000, pos=0, max_seq=2048),
        # prefill GEMMs: a short prompt (or a batch of 16 users), a ragged one, chunks of 512 and 2048 tokens
        dict(name="gemm_q4_k_14336x4096_m16", kind="gemm", fmt="Q4_K", n=14336, k=4096, m=16, x="bf16", y="f32",
             slab=True),
        dict(name="gemm_q6_k_4096x14336_m100", kind="gemm", fmt="Q6_K", n=4096, k=14336, m=100, x="f16", y="f16",
             slab=True),
        dict(name="gemm_q4_k_14336x4096_m512", kind="gemm", fmt="Q4_K", n=14336, k=4096, m=512, x="bf16", y="f32",
             slab=False),
        dict(name="gemm_nf4_4096x4096_m300", kind="gemm", fmt="NF4", n=4096, k=4096, m=300, x="f16", y="f16",
             slab=True),
        dict(name="gemm_q8_0_14336x4096_m2048", kind="gemm", fmt="Q8_0", n=14336, k=4096, m=2048, x="f16", y="f16",
             slab=True),
        # a packed weight expanded to f16 for a program's own use of it
        dict(name="dequant_q4_k_14336x4096", kind="dequant", fmt="Q4_K", n=14336, k=4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "head", "decode", "prefill_in", "gemm", "gemm", "gemm", "gemm", "dequant"])
    fmts = sorted(FMT)
    if kind == "gemv":
        fmt = rng.choice(fmts + ["NF4"])
        mode = 0 if fmt == "NF4" else rng.choice([0, 0, 2])
        k = 256 * _log(rng, 2, 56)
        return dict(kind=kind, fmt=fmt, n=_log(rng, 200, 20000 if mode == 0 else 15000), k=k,
                    act=rng.choice(["f16", "f16", "f32"]), mode=mode)
    if kind == "head":
        return dict(kind=kind, fmt=rng.choice(["Q4_K", "Q6_K", "Q8_0", "Q5_K"]), n=_log(rng, 32000, 152064),
                    k=rng.choice([896, 1536, 2048, 3072, 4096]) // 256 * 256)
    if kind == "decode":
        fmt = rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q8_0", "IQ4_XS"])
        return dict(kind=kind, model="llama8b", fmt=fmt, v_down=rng.choice([fmt, "Q6_K"]), layers=rng.randint(1, 4),
                    vocab=_log(rng, 1000, 16000), pos=_log(rng, 1, 8191), max_seq=8192,
                    window=rng.choice([0, 0, 0, 1000]))
    if kind == "prefill_in":
        return dict(kind=kind, fmt=rng.choice(["Q4_K", "Q8_0", "Q6_K"]), m=_log(rng, 2, 1024), vocab=32000,
                    pos=rng.choice([0, 0, rng.randint(1, 1000)]), max_seq=2048)
    if kind == "gemm":
        fmt = rng.choice(fmts + ["NF4", "Q4_K", "Q8_0"])
        n, k = rng.choice([(14336, 4096), (4096, 14336), (4096, 4096), (1024, 4096), (6144, 4096),
                           (_log(rng, 300, 14336), 256 * rng.randint(4, 40)), (_log(rng, 300, 14336), 4096)])
        return dict(kind=kind, fmt=fmt, n=n, k=k, m=_log(rng, 2, 2048), x=rng.choice(["f16", "bf16", "bf16", "f32"]),
                    y=rng.choice(["f16", "f32"]), slab=True if fmt == "NF4" else rng.random() < 0.6)
    return dict(kind=kind, fmt=rng.choice(fmts + ["NF4"]), n=_log(rng, 300, 20000), k=256 * _log(rng, 2, 56))


# ------------------------------------------------------------------- GEMV

def _prep_gemv(c, seed):
    n, k, fmt, dt = c["n"], c["k"], c["fmt"], DTYPES[c["act"]]
    s = dict(case=c, ctx=_hip(), x=_normal(k, seed, 1, dtype=dt), y=torch.empty(n, dtype=dt, device="cuda"))
    if fmt == "NF4":
        s["w"] = _nf4_weight(n, k, seed)
    else:
        rows = 2 * n if c["mode"] == 2 else n
        s["w"] = _packed(fmt, rows, k, seed, 2)
        s["bias"] = _normal(rows, seed, 3, scale=0.1, dtype=dt)
    return s


def _run_gemv(s):
    c, ctx = s["case"], s["ctx"]
    ctx.use_torch_stream()
    if c["fmt"] == "NF4":
        s["w"].gemv(ctx, s["x"], s["y"])
    else:
        ctx.gguf_gemv(FMT[c["fmt"]], s["x"], s["w"], s["bias"], s["y"], c["n"], c["k"], c["mode"])
    return s["y"]


def _exact_gemv(c, seed):
    n, k, dt = c["n"], c["k"], DTYPES[c["act"]]
    x = _normal(k, seed, 1, dtype=dt).to(torch.float64)
    if c["fmt"] == "NF4":
        return _matvec64("NF4", n, k, x, seed, 2)
    rows = 2 * n if c["mode"] == 2 else n
    v = _matvec64(c["fmt"], rows, k, x, seed, 2) + _normal(rows, seed, 3, scale=0.1, dtype=dt).to(torch.float64)
    return v if c["mode"] == 0 else v[:n] * torch.sigmoid(v[:n]) * v[n:]


def _nf4_weight(n, k, seed, bs=64):
    parts = [p for _, p, _ in _chunks("NF4", n, k, seed, 2, bs=bs)]
    host = HostNf4(packed=np.zeros(1, np.uint8), absmax=np.zeros(1, np.float32),
                   qmap=np.asarray(NF4_CODE, np.float32), rows=n, cols=k, blocksize=bs)
    w = Nf4Weight(host)
    w.packed = torch.cat([p for p, _ in parts])
    w.absmax = torch.cat([a for _, a in parts])
    return w


# ------------------------------------------------------------------- head

def _prep_head(c, seed):
    n, k = c["n"], c["k"]
    return dict(case=c, ctx=_hip(), w=_packed(c["fmt"], n, k, seed, 2), x=_normal(k, seed, 1, dtype=torch.float16),
                norm=_normal(k, seed, 4, scale=0.1, mean=1.0, dtype=torch.float16),
                y=torch.empty(n, dtype=torch.float16, device="cuda"),
                slot=torch.zeros(1, dtype=torch.int64, device="cuda"),
                ids=torch.zeros(1, dtype=torch.int32, device="cuda"))


def _run_head(s):
    c, ctx = s["case"], s["ctx"]
    ctx.use_torch_stream()
    ctx.gguf_gemv_argmax(FMT[c["fmt"]], s["x"], s["norm"], 1e-5, s["w"], s["y"], c["n"], c["k"], s["slot"])
    ctx.argmax_to_ids(s["slot"], s["ids"])
    return s["y"], s["ids"]


def _rms64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(torch.float64)


def _exact_head(c, seed):
    n, k = c["n"], c["k"]
    h = _rms64(_normal(k, seed, 1, dtype=torch.float16).to(torch.float64),
               _normal(k, seed, 4, scale=0.1, mean=1.0, dtype=torch.float16), 1e-5)
    return _matvec64(c["fmt"], n, k, h, seed, 2), None


# ------------------------------------------------------------ decode step

def _cfg(c):
    shape, small = (LLAMA8B, False) if c["model"] == "llama8b" else (QWEN05B, True)
    return DecoderConfig(n_layers=c["layers"], vocab=c["vocab"], ggml_type=FMT[c["fmt"]], max_seq=c["max_seq"],
                         window=c["window"], rope_theta=1e6 if small else 5e5, rms_eps=1e-6 if small else 1e-5,
                         qkv_bias=small, tied=True, **shape)


def _mats(c, cfg):
    """name -> (format, rows, columns, key) of a layer's matrices."""
    qd, kvd, h, f = cfg.q_heads * cfg.head_dim, cfg.kv_heads * cfg.head_dim, cfg.hidden, cfg.ffn
    fmt, vd = c["fmt"], c["v_down"]
    m = {"wo": (fmt, h, qd, 4), "w_gate_up": (fmt, 2 * f, h, 6), "w_down": (vd, h, f, 7)}
    if fmt == vd:
        m["wqkv"] = (fmt, qd + 2 * kvd, h, 5)
    else:
        m.update(wqkv=(fmt, qd, h, 5), wk=(fmt, kvd, h, 8), wv=(vd, kvd, h, 9))
    return m


def _vec(cfg, seed, i, what):
    """Norm weights and biases (f16)."""
    if what == "bqkv":
        return _normal((cfg.q_heads + 2 * cfg.kv_heads) * cfg.head_dim, seed, i, 13, scale=0.1, dtype=torch.float16)
    return _normal(cfg.hidden, seed, i, {"attn_norm": 11, "ffn_norm": 12, "final_norm": 14}[what], scale=0.1,
                   mean=1.0, dtype=torch.float16)


def _kv(c, cfg, seed, i):
    """The layer's caches with positions [0, pos) filled, zeros beyond."""
    out = []
    for j in (21, 22):
        t = torch.zeros((cfg.kv_heads, cfg.max_seq, cfg.head_dim), dtype=torch.float16, device="cuda")
        t[:, :c["pos"]] = _normal((cfg.kv_heads, c["pos"], cfg.head_dim), seed, i, j, dtype=torch.float16)
        out.append(t)
    return out


def _token(c, seed):
    return (seed * 7919 + 17) % c["vocab"]


def _prep_decode(c, seed):
    cfg = _cfg(c)
    host = lambda t: t.cpu().numpy()  # noqa: E731
    types = {p: FMT[c["fmt"]] for p in PROJECTIONS}
    types["v"] = types["down"] = FMT[c["v_down"]]
    model = HostModel(cfg, host(_packed(c["fmt"], cfg.vocab, cfg.hidden, seed, 3)),
                      host(_vec(cfg, seed, 0, "final_norm")))
    for i in range(1, cfg.n_layers + 1):
        L = {name: host(_packed(f, r, k, seed, i, key)) for name, (f, r, k, key) in _mats(c, cfg).items()}
        L.update(attn_norm=host(_vec(cfg, seed, i, "attn_norm")), ffn_norm=host(_vec(cfg, seed, i, "ffn_norm")),
                 bqkv=host(_vec(cfg, seed, i, "bqkv")) if cfg.qkv_bias else None, types=types)
        model.layers.append(L)
    dd = DeviceDecoder(_hip(), model)
    for i, L in enumerate(dd.layers):
        for t, v in zip((L["k_cache"], L["v_cache"]), _kv(c, cfg, seed, i + 1)):
            t.copy_(v)
    return dict(case=c, dd=dd, token=torch.full((1,), _token(c, seed), dtype=torch.int32, device="cuda"),
                pos=torch.full((1,), c["pos"], dtype=torch.int32, device="cuda"))


def _run_decode(s):
    # a serving loop whose sampler sits outside the step writes the token and
    # its position, then steps
    dd = s["dd"]
    dd.ids.copy_(s["token"])
    dd.pos.copy_(s["pos"])
    dd.step()
    return [dd.logits, dd.ids, dd.x] + [L[n] for L in dd.layers for n in ("k_cache", "v_cache")]


def _rope64(x, pos, theta):
    """NeoX rotation of x [..., heads, dim] in f64; pos broadcasts over the leading axes."""
    half = x.shape[-1] // 2
    f = theta ** (-2.0 * torch.arange(half, dtype=torch.float64, device=x.device) / x.shape[-1])
    a = torch.as_tensor(pos, dtype=torch.float64, device=x.device)[..., None, None] * f
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * torch.cos(a) - hi * torch.sin(a), lo * torch.sin(a) + hi * torch.cos(a)], -1)


def _exact_decode(c, seed):
    cfg, pos = _cfg(c), c["pos"]
    qd, kvd, D = cfg.q_heads * cfg.head_dim, cfg.kv_heads * cfg.head_dim, cfg.head_dim
    x = _row64(c["fmt"], cfg.vocab, cfg.hidden, torch.tensor([_token(c, seed)], device="cuda"), seed, 3)[0]
    caches = []
    for i in range(1, cfg.n_layers + 1):
        mats = _mats(c, cfg)
        mv = lambda name, v: _matvec64(*mats[name][:3], v, seed, i, mats[name][3])  # noqa: E731, B023
        h = _rms64(x, _vec(cfg, seed, i, "attn_norm"), cfg.rms_eps)
        qkv = mv("wqkv", h)
        if "wk" in mats:
            qkv = torch.cat([qkv, mv("wk", h), mv("wv", h)])
        if cfg.qkv_bias:
            qkv = qkv + _vec(cfg, seed, i, "bqkv").to(torch.float64)
        q = _rope64(qkv[:qd].reshape(cfg.q_heads, D), pos, cfg.rope_theta)
        kc, vc = (t.to(torch.float64) for t in _kv(c, cfg, seed, i))
        kc[:, pos] = _rope64(qkv[qd:qd + kvd].reshape(cfg.kv_heads, D), pos, cfg.rope_theta)
        vc[:, pos] = qkv[qd + kvd:].reshape(cfg.kv_heads, D)
        lo = max(0, pos + 1 - cfg.window) if cfg.window else 0
        g = cfg.q_heads // cfg.kv_heads
        sc = torch.matmul(q.reshape(cfg.kv_heads, g, D), kc[:, lo:pos + 1].transpose(1, 2).contiguous()) / math.sqrt(D)
        att = torch.matmul(torch.softmax(sc, -1), vc[:, lo:pos + 1].contiguous()).reshape(qd)
        x = x + mv("wo", att)
        gu = mv("w_gate_up", _rms64(x, _vec(cfg, seed, i, "ffn_norm"), cfg.rms_eps))
        x = x + mv("w_down", gu[:cfg.ffn] * torch.sigmoid(gu[:cfg.ffn]) * gu[cfg.ffn:])
        caches += [kc, vc]
    logits = _matvec64(c["fmt"], cfg.vocab, cfg.hidden, _rms64(x, _vec(cfg, seed, 0, "final_norm"), cfg.rms_eps),
                       seed, 3)
    return [logits, None, x] + caches


# ------------------------------------------------- first half of a prefill

def _prep_prefill_in(c, seed):
    h, qd, kvd, D = 4096, 4096, 1024, 128
    m, fmt = c["m"], c["fmt"]
    e = lambda *s: torch.empty(s, dtype=torch.float16, device="cuda")  # noqa: E731
    cache = lambda: torch.zeros((kvd // D, c["max_seq"], D), dtype=torch.float16, device="cuda")  # noqa: E731
    return dict(case=c, ctx=_hip(), table=_packed(fmt, c["vocab"], h, seed, 1), wq=_packed(fmt, qd, h, seed, 2),
                wk=_packed(fmt, kvd, h, seed, 3), wv=_packed(fmt, kvd, h, seed, 4),
                norm=_normal(h, seed, 5, scale=0.1, mean=1.0, dtype=torch.float16), ids=_ids(c, seed),
                x=e(m, h), hn=e(m, h), q=e(m, qd), k=e(m, kvd), v=e(m, kvd), kc=cache(), vc=cache(),
                slab=torch.empty(SLAB_BYTES, dtype=torch.uint8, device="cuda"))


def _ids(c, seed):
    return torch.randint(0, c["vocab"], (c["m"],), generator=_gen(seed, 6), device="cuda", dtype=torch.int32)


def _run_prefill_in(s):
    c, ctx, m, h = s["case"], s["ctx"], s["case"]["m"], 4096
    t = FMT[c["fmt"]]
    ctx.use_torch_stream()
    ctx.gguf_gather(t, s["table"], s["ids"], s["x"], m, h)
    ctx.rmsnorm(s["x"], s["norm"], s["hn"], m, h, 1e-5)
    for w, y in (("wq", "q"), ("wk", "k"), ("wv", "v")):
        ctx.gguf_gemm_slab(t, s["hn"], s[w], s[y], m, s[y].shape[1], h, s["slab"])
    ctx.rope(s["q"], m, 32, 128, c["pos"], 5e5, 64)
    ctx.rope(s["k"], m, 8, 128, c["pos"], 5e5, 64)
    ctx.kv_append(s["k"], s["v"], s["kc"], s["vc"], m, 8, 128, c["pos"], c["max_seq"])
    return s["x"], s["q"], s["kc"], s["vc"]


def _exact_prefill_in(c, seed):
    h, m, fmt, p0 = 4096, c["m"], c["fmt"], c["pos"]
    x = _row64(fmt, c["vocab"], h, _ids(c, seed).long(), seed, 1)
    hn = _rms64(x, _normal(h, seed, 5, scale=0.1, mean=1.0, dtype=torch.float16), 1e-5)

    def proj(n, key):
        return torch.cat([hn @ _f16_values(v).to(torch.float64).T for _, _, v in _chunks(fmt, n, h, seed, key)], 1)
    pos = p0 + torch.arange(m, device="cuda")
    q = _rope64(proj(4096, 2).reshape(m, 32, 128), pos, 5e5).reshape(m, 4096)
    kc, vc = (torch.zeros((8, c["max_seq"], 128), dtype=torch.float64, device="cuda") for _ in range(2))
    kc[:, p0:p0 + m] = _rope64(proj(1024, 3).reshape(m, 8, 128), pos, 5e5).transpose(0, 1)
    vc[:, p0:p0 + m] = proj(1024, 4).reshape(m, 8, 128).transpose(0, 1)
    return x, q, kc, vc


# ----------------------------------------------------------- prefill GEMM

def _prep_gemm(c, seed):
    m, n, k = c["m"], c["n"], c["k"]
    return dict(case=c, ctx=_hip(), x=_normal((m, k), seed, 1, dtype=DTYPES[c["x"]]),
                w=_nf4_weight(n, k, seed) if c["fmt"] == "NF4" else _packed(c["fmt"], n, k, seed, 2),
                y=torch.empty((m, n), dtype=DTYPES[c["y"]], device="cuda"),
                slab=torch.empty(SLAB_BYTES, dtype=torch.uint8, device="cuda") if c["slab"] else None)


def _run_gemm(s):
    c, ctx = s["case"], s["ctx"]
    ctx.use_torch_stream()
    if c["fmt"] == "NF4":
        s["w"].gemm(ctx, s["x"], s["y"], s["slab"])
    elif c["slab"]:
        ctx.gguf_gemm_slab(FMT[c["fmt"]], s["x"], s["w"], s["y"], c["m"], c["n"], c["k"], s["slab"])
    else:
        ctx.gguf_gemm(FMT[c["fmt"]], s["x"], s["w"], s["y"], c["m"], c["n"], c["k"])
    return s["y"]


def _exact_gemm(c, seed):
    return _matmul64(c["fmt"], c["n"], c["k"], _normal((c["m"], c["k"]), seed, 1, dtype=DTYPES[c["x"]]), seed, 2)


# ---------------------------------------------------------------- dequant

def _prep_dequant(c, seed):
    n, k = c["n"], c["k"]
    return dict(case=c, ctx=_hip(), w=_nf4_weight(n, k, seed) if c["fmt"] == "NF4" else _packed(c["fmt"], n, k, seed, 2),
                out=torch.empty(n * k, dtype=torch.float16, device="cuda"))


def _run_dequant(s):
    c, ctx = s["case"], s["ctx"]
    ctx.use_torch_stream()
    if c["fmt"] == "NF4":
        s["w"].dequant(ctx, s["out"])
    else:
        ctx.gguf_dequant(FMT[c["fmt"]], s["w"], s["out"], c["n"] * c["k"] // gguf.block_elems(FMT[c["fmt"]]))
    return s["out"]


def _exact_dequant(c, seed):
    return torch.cat([_f16_values(v).reshape(-1) for _, _, v in _chunks(c["fmt"], c["n"], c["k"], seed, 2)]).to(
        torch.float64)


# ------------------------------------------------------------ the interface

_KINDS = {
    "gemv": (_prep_gemv, _run_gemv, _exact_gemv),
    "head": (_prep_head, _run_head, _exact_head),
    "decode": (_prep_decode, _run_decode, _exact_decode),
    "prefill_in": (_prep_prefill_in, _run_prefill_in, _exact_prefill_in),
    "gemm": (_prep_gemm, _run_gemm, _exact_gemm),
    "dequant": (_prep_dequant, _run_dequant, _exact_dequant),
}


def prepare(case, seed):
    state = _KINDS[case["kind"]][0](case, int(seed))
    state["kind"] = case["kind"]
    return state


def run(state):
    return _KINDS[state["kind"]][1](state)


def exact(case, seed):
    with torch.no_grad():
        return _KINDS[case["kind"]][2](case, int(seed))


def work(case):
    c, kind = case, case["kind"]
    if kind in ("gemv", "head"):
        act = _esz(c.get("act", "f16"))
        rows = 2 * c["n"] if c.get("mode") == 2 else c["n"]
        return {"bytes": _wbytes(c["fmt"], rows, c["k"]) + act * (c["k"] + c["n"] + (rows if kind == "gemv" else c["k"])),
                "flops": 2 * rows * c["k"]}
    if kind == "gemm":
        return {"bytes": _wbytes(c["fmt"], c["n"], c["k"]) + c["m"] * (c["k"] * _esz(c["x"]) + c["n"] * _esz(c["y"])),
                "flops": 2 * c["m"] * c["n"] * c["k"]}
    if kind == "dequant":
        return {"bytes": _wbytes(c["fmt"], c["n"], c["k"]) + 2 * c["n"] * c["k"], "flops": c["n"] * c["k"]}
    if kind == "prefill_in":
        m, n = c["m"], 4096 + 2048
        return {"bytes": m * gguf.row_bytes(FMT[c["fmt"]], 4096) + _wbytes(c["fmt"], n, 4096) + 2 * m * (4096 + n),
                "flops": 2 * m * n * 4096}
    cfg = _cfg(c)
    live = min(c["pos"] + 1, c["window"]) if c["window"] else c["pos"] + 1
    mats = _mats(c, cfg).values()
    kv = 2 * 2 * live * cfg.kv_heads * cfg.head_dim
    bytes_ = cfg.n_layers * (sum(_wbytes(f, r, k) for f, r, k, _ in mats) + kv) + _wbytes(c["fmt"], cfg.vocab, cfg.hidden)
    flops = cfg.n_layers * (sum(2 * r * k for _, r, k, _ in mats) + 4 * live * cfg.q_heads * cfg.head_dim)
    return {"bytes": bytes_ + 2 * cfg.vocab, "flops": flops + 2 * cfg.vocab * cfg.hidden}


def tolerance(case):
    """Four times the error of the outputs against ``exact``, or of what the
    element types give where that is larger."""
    c, kind = case, case["kind"]
    if kind == "dequant":
        return "exact"
    if kind == "decode":
        # f16 activations rounded after every launch, adding in quadrature
        # over the layers (1.6e-3 seen after 4 layers, 2.9e-3 after 24)
        return {"rel": 2.5e-3 * math.sqrt(c["layers"])}
    if kind == "prefill_in":
        return {"rel": 1.5e-3}  # f16 outputs of f16 norms
    if kind == "gemm" and c["y"] == "f32":
        return {"rel": 5e-6}  # fp32 accumulation
    if kind in ("gemv", "head") and c.get("act", "f16") == "f32":
        return {"rel": 1e-4}  # x as 16-bit fixed point per 32 elements, fp32 accumulation
    return {"rel": 1e-3}  # f16 outputs
