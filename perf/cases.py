"""The work whose speed this library is judged by: the calls that a decode
loop, a prompt pass and a key codec make, through the public Python API.

Shapes are those of ``bench.py`` and of the tests: Hq 32 / Hkv 16 / D 256 with
a window of 1024 (sliding layers of a 31B-class model) or without one (the
context sweep), Hq 32 / Hkv 4 / D 512 (global layers), D 128 (the small
configuration and the compressed keys).  Queries and keys are RMS-normed
N(0, 1) per head vector and are scored with scale 1; values are N(0, 1).

Inputs are made here with plain torch, packed caches included, so that
``exact`` can compute each result in float64 from the same words.
"""
import math

import torch

from gemma4metal_amd import polar as pq
from gemma4metal_amd import turboquant as tq

_DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "f16": 2, "bf16": 2}


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one decode call of the reference's own unit test: 33 keys, fp32
        # everywhere; nothing but latency
        dict(name="decode_tiny", kind="decode", Hq=2, Hkv=1, D=128, L=33, window=0, q="f32", sb="f32"),
        # the sliding layers of one decode step (50 of them at 786 tokens of
        # context, window 1024), captured once and replayed per token
        dict(name="decode_step50", kind="step", layers=50, Hq=32, Hkv=16, D=256, L=786, window=1024, q="bf16",
             sb="f16"),
        # one full-attention layer at 32k tokens: the headline benchmark
        dict(name="decode_32k", kind="decode", Hq=32, Hkv=16, D=256, L=32768, window=0, q="bf16", sb="f16"),
        # one global layer (8 query heads per kv head, D 512) at 32k tokens
        dict(name="decode_global", kind="decode", Hq=32, Hkv=4, D=512, L=32768, window=0, q="bf16", sb="f16"),
        # a serving batch: 64 sequences of 512 .. 32768 tokens, every other
        # one under a 1024-token window
        dict(name="ragged_64", kind="ragged", B=64, Hq=32, Hkv=16, D=256, lo=512, hi=32768, window=1024, q="bf16",
             sb="f16"),
        # a 512-token prompt chunk after 3584 cached tokens, sliding layer:
        # its K/V rows are quantized into the cache, then its queries attend
        dict(name="prefill_sliding", kind="prefill", Hq=32, Hkv=16, D=256, prior=3584, new=512, window=1024,
             q="bf16", sb="f16"),
        # the same chunk through a global layer
        dict(name="prefill_global", kind="prefill", Hq=32, Hkv=4, D=512, prior=3584, new=512, window=0, q="bf16",
             sb="f16"),
        # a prompt's K rows through the cache's number format and back (the
        # engine quantizes on arrival and dequantizes on its fallback path)
        dict(name="cache_codec", kind="codec", rows=65536, D=256, x="f32", sb="f16"),
        # one decode layer over 7-level polar keys with a sign sketch and
        # int4 values, at 32k tokens
        dict(name="polar7_decode", kind="polar7", Hq=32, Hkv=16, L=32768, window=0, sb="f16"),
        # a prompt's keys into that format
        dict(name="polar7_prompt", kind="polar7_encode", rows=65536),
        # the reference's packed block codec: rotate and encode, then decode
        # with (cos, sin) tables
        dict(name="polar_codec", kind="polar_codec", rows=32768, D=128),
        # the reference's attention over block-encoded keys, one key set per
        # query head and fp32 values
        dict(name="compressed_sdpa", kind="compressed", op="sdpa", Hq=16, Hkv=16, D=128, N=8192),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "step", "ragged", "prefill", "prefill", "codec", "polar7",
                       "polar7_encode", "polar_codec", "compressed"])
    q = rng.choice(["bf16", "bf16", "f16", "f32"])
    sb = rng.choice(["f16", "f16", "f32"])
    Hq, Hkv, D = rng.choice([(32, 16, 256), (32, 16, 256), (32, 4, 512), (16, 8, 128), (32, 8, 128), (8, 1, 256)])
    if kind == "decode":
        return dict(kind=kind, Hq=Hq, Hkv=Hkv, D=D, L=_log(rng, 33, 262144 if D <= 256 else 65536),
                    window=rng.choice([0, 0, 1024]), q=q, sb=sb)
    if kind == "step":
        return dict(kind=kind, layers=rng.randint(8, 50), Hq=Hq, Hkv=Hkv, D=D, L=_log(rng, 64, 3000), window=1024,
                    q=q, sb=sb)
    if kind == "ragged":
        return dict(kind=kind, B=rng.randint(3, 48), Hq=Hq, Hkv=Hkv, D=D, lo=_log(rng, 33, 512),
                    hi=_log(rng, 1024, 16384), window=rng.choice([0, 1024]), q=q, sb=sb)
    if kind == "prefill":
        prior = rng.choice([0, _log(rng, 16, 3584)])
        return dict(kind=kind, Hq=Hq, Hkv=Hkv, D=D, prior=prior, new=_log(rng, 16, 512),
                    window=rng.choice([0, 1024]), q=q, sb=sb)
    if kind == "codec":
        return dict(kind=kind, rows=_log(rng, 16, 65536), D=rng.choice([128, 256, 512]),
                    x=rng.choice(["f32", "bf16", "f16"]), sb=sb)
    if kind == "polar7":
        return dict(kind=kind, Hq=32, Hkv=rng.choice([16, 8]), L=_log(rng, 512, 32768),
                    window=rng.choice([0, 0, 1024]), sb=sb)
    if kind == "polar7_encode":
        return dict(kind=kind, rows=_log(rng, 16, 65536))
    if kind == "polar_codec":
        return dict(kind=kind, rows=_log(rng, 16, 32768), D=rng.choice([64, 128, 256]))
    Hkv = rng.choice([16, 8])
    D = rng.choice([64, 128, 128, 256])
    return dict(kind=kind, op=rng.choice(["sdpa", "score"]), Hq=16, Hkv=Hkv, D=D,
                N=_log(rng, 200, 8192 * 128 // max(D, 128)))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _rms(x):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6)


def _mlx_rule(x, sb):
    """The cache's number format (MLX affine int4, groups of 64) in fp32:
    nibbles [.., D] as int32, scale and bias [.., D/64]."""
    g = x.float().reshape(*x.shape[:-1], -1, 64)
    mx, mn = g.amax(-1), g.amin(-1)
    scale = ((mx - mn) / 15.0).clamp(min=1e-7)
    side = mn.abs() > mx.abs()
    scale = torch.where(side, scale, -scale)
    edge = torch.where(side, mn, mx)
    q0 = torch.round(edge / scale)
    nz = q0 != 0
    scale = torch.where(nz, edge / q0, scale)
    bias = torch.where(nz, edge, torch.zeros_like(edge))
    n = torch.round((g - bias[..., None]) / scale[..., None]).clamp(0, 15).to(torch.int32)
    return n.reshape(x.shape), scale.to(sb), bias.to(sb)


def _pack(n):
    """Eight nibbles a word, element i at bits 4i; int32 bit patterns."""
    sh = torch.arange(0, 32, 4, device=n.device, dtype=torch.int32)
    return (n.reshape(*n.shape[:-1], -1, 8) << sh).sum(-1, dtype=torch.int32)


def _unpack(w):
    sh = torch.arange(0, 32, 4, device=w.device, dtype=torch.int32)
    return ((w[..., None] >> sh) & 15).reshape(*w.shape[:-1], -1)


def _rows64(w, s, b):
    """Dequantized rows in float64."""
    n = _unpack(w.view(torch.int32)).double()
    return (n.reshape(*s.shape, 64) * s.double()[..., None] + b.double()[..., None]).reshape(n.shape)


def _new_cache(lead, rows, D, sb):
    kq = torch.zeros((*lead, rows, D // 8), dtype=torch.int32, device="cuda")
    ks = torch.zeros((*lead, rows, D // 64), dtype=sb, device="cuda")
    return [kq, ks, ks.clone(), kq.clone(), ks.clone(), ks.clone()]


def _fill(cache, at, g, rows, D, sb):
    """`rows` random rows into cache tensors [at][0:rows]."""
    for j, norm in ((0, True), (3, False)):
        x = _normal(g, rows, D)
        n, s, b = _mlx_rule(_rms(x) if norm else x, sb)
        cache[j][at][:rows] = _pack(n)
        cache[j + 1][at][:rows] = s
        cache[j + 2][at][:rows] = b


def _words(cache):
    """The packed tensors as the uint32 that the API names."""
    return [t.view(torch.uint32) if t.dtype == torch.int32 else t for t in cache]


def _queries(g, dtype, *shape):
    return _rms(_normal(g, *shape)).to(dtype)


def _lens(case, seed):
    g = torch.Generator().manual_seed(int(seed) * 104729 + 5)
    return torch.randint(case["lo"], case["hi"] + 1, (case["B"],), generator=g, dtype=torch.int32)


def _orthogonal(g, D):
    return torch.linalg.qr(_normal(g, D, D).double())[0].float().contiguous()


def _tree(y, levels):
    """Angles of the pairwise polar tree over the last axis, level 1 first,
    and the radius."""
    out, r = [], y
    for _ in range(levels):
        a, b = r[..., 0::2], r[..., 1::2]
        out.append(torch.atan2(b, a) % (2 * math.pi))
        r = torch.sqrt(a * a + b * b)
    return out, r[..., 0]


def _untree(idx, cbs, r):
    """Values of the tree from its indices: the inverse of `_tree`."""
    v = r[..., None]
    for k, cb in zip(reversed(idx), reversed(cbs)):
        th = cb[k.long()]
        v = torch.stack([v * torch.cos(th), v * torch.sin(th)], -1).flatten(-2)
    return v


def _p7_books():
    one = ((torch.arange(16, dtype=torch.float64) + 0.5) * (2 * math.pi / 16)).cuda()
    two = ((torch.arange(4, dtype=torch.float64) + 0.5) * (math.pi / 8)).cuda()
    return [one] + [two] * 6


def _p7_indices(ang):
    return [(ang[0] * (16 / (2 * math.pi))).long().clamp(0, 15)] + [
        (a * (8 / math.pi)).long().clamp(0, 3) for a in ang[1:]]


def _bits(idx, width):
    """Indices [.., n] into int32 words, index j at bits width * j."""
    per = 32 // width
    pad = -idx.shape[-1] % per
    idx = torch.nn.functional.pad(idx, (0, pad)).reshape(*idx.shape[:-1], -1, per).to(torch.int32)
    sh = (torch.arange(per, device=idx.device, dtype=torch.int32) * width)
    return (idx << sh).sum(-1, dtype=torch.int32)


def _p7_keys(g, P, S, Hkv, L):
    """Random keys in the 7-level format: the packed cache, and the rotated
    keys' values and sketch signs in float64 (per head)."""
    angles = torch.zeros((Hkv, L, 12), dtype=torch.int32, device="cuda")
    norms = torch.zeros((Hkv, L), dtype=torch.int32, device="cuda")
    qjl = torch.zeros((Hkv, L, 4), dtype=torch.int32, device="cuda")
    cbs = _p7_books()
    for h in range(Hkv):
        y = _normal(g, L, 128) @ P.t()
        ang, r = _tree(y.double(), 7)
        idx = _p7_indices(ang)
        rad = r.half()
        res = y.double() - _untree(idx, cbs, rad.double())
        w = [_bits(idx[0], 4), _bits(idx[1], 2), _bits(idx[2], 2)]
        last = (_bits(idx[3], 2) | (_bits(idx[4], 2) << 16) | (_bits(idx[5], 2) << 24) | (_bits(idx[6], 2) << 28))
        angles[h] = torch.cat(w + [last], -1)
        rn = res.norm(dim=-1).half()
        norms[h] = (rad.view(torch.int16).int() & 0xFFFF) | (rn.view(torch.int16).int() << 16)
        qjl[h] = _bits((res @ S.double().t() >= 0).int(), 1)
    return angles, norms, qjl


def _block_books():
    """Level 1: 16 angles of the circle; levels 2 to 4: 4 of the quadrant."""
    one = (torch.arange(16, dtype=torch.float64) + 0.5) * (2 * math.pi / 16)
    two = (torch.arange(4, dtype=torch.float64) + 0.5) * (math.pi / 8)
    return [one.float().cuda()] + [two.float().cuda() for _ in range(3)]


def _block_keys(g, rows, D):
    """Random keys as 16-value blocks of 4 levels (u8 per angle)."""
    y = _normal(g, rows * D // 16, 16)
    ang, r = _tree(y, 4)
    return [k.to(torch.uint8).reshape(-1).contiguous() for k in _p7_indices(ang)[:4]] + [r.half()]


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = dict(case)
    if kind == "codec":
        s["rows_"] = _rms(_normal(g, case["rows"], case["D"])).to(_DT[case["x"]])
        return s
    if kind == "polar7_encode":
        s["codec"] = pq.Polar7Codec(_orthogonal(g, 128), _normal(g, 128, 128))
        s["k"] = _normal(g, case["rows"], 128)
        return s
    if kind == "polar_codec":
        s["P"] = _orthogonal(g, case["D"])
        s["k"] = _normal(g, case["rows"], case["D"])
        s["cb"] = _block_books()
        s["cs"] = [pq.cos_sin_table(c) for c in s["cb"]]
        return s
    if kind == "polar7":
        P, S = _orthogonal(g, 128), _normal(g, 128, 128)
        s["codec"] = pq.Polar7Codec(P, S)
        s["keys"] = [t.view(torch.uint32) for t in _p7_keys(g, P, S, case["Hkv"], case["L"])]
        v = _new_cache((case["Hkv"],), case["L"], 128, _DT[case["sb"]])[3:]
        for h in range(case["Hkv"]):
            n, sc, b = _mlx_rule(_normal(g, case["L"], 128), _DT[case["sb"]])
            v[0][h], v[1][h], v[2][h] = _pack(n), sc, b
        s["v"] = _words(v)
        s["q_"] = _normal(g, case["Hq"], 128)
        return s
    if kind == "compressed":
        rows = case["Hkv"] * case["N"]
        s["keys"] = _block_keys(g, rows, case["D"])
        s["cb"] = _block_books()
        s["v"] = _normal(g, rows, case["D"])
        s["q_"] = _normal(g, case["Hq"], case["D"])
        return s
    Hq, Hkv, D, sb, qt = case["Hq"], case["Hkv"], case["D"], _DT[case["sb"]], _DT[case["q"]]
    if kind == "decode":
        cache = _new_cache((Hkv,), case["L"], D, sb)
        for h in range(Hkv):
            _fill(cache, h, g, case["L"], D, sb)
        s["cache"], s["q_"] = _words(cache), _queries(g, qt, Hq, D)
    elif kind == "step":
        cache = _new_cache((case["layers"] * Hkv,), case["L"], D, sb)
        for h in range(case["layers"] * Hkv):
            _fill(cache, h, g, case["L"], D, sb)
        cache = [t.view(case["layers"], Hkv, *t.shape[1:]) for t in cache]
        s["cache"], s["q_"] = _words(cache), _queries(g, qt, case["layers"], Hq, D)
        s["out"] = torch.empty((case["layers"], Hq, D), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        with torch.cuda.stream(stream):
            _layer(s, 0)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            for i in range(case["layers"]):
                _layer(s, i)
        s["graph"] = graph
    elif kind == "ragged":
        lens = _lens(case, seed)
        cache = _new_cache((case["B"], Hkv), int(lens.max()), D, sb)
        for b in range(case["B"]):
            n = int(lens[b])
            part = _new_cache((1,), Hkv * n, D, sb)
            _fill(part, 0, g, Hkv * n, D, sb)
            for t, u in zip(cache, part):
                t[b, :, :n] = u.view(Hkv, n, -1)
        s["cache"], s["q_"] = _words(cache), _queries(g, qt, case["B"], Hq, D)
        s["lens"] = lens.cuda()
        s["windows"] = torch.tensor([case["window"] if b % 2 == 0 else 0 for b in range(case["B"])],
                                    dtype=torch.int32, device="cuda")
    elif kind == "prefill":
        cache, k, v = _prompt(g, case)
        s["cache"], s["k"], s["v"] = _words(cache), k, v
        s["q_"] = _queries(g, qt, case["new"], Hq, D)
        s["at"] = torch.tensor([case["prior"]], dtype=torch.int32, device="cuda")
    return s


def _prompt(g, case):
    """A cache [1, Hkv, prior + new] whose first `prior` rows are filled, and
    the chunk's fp32 K and V rows [1, Hkv, new, D]."""
    Hkv, D, prior, new = case["Hkv"], case["D"], case["prior"], case["new"]
    cache = _new_cache((1, Hkv), prior + new, D, _DT[case["sb"]])
    if prior:
        for h in range(Hkv):
            _fill(cache, (0, h), g, prior, D, _DT[case["sb"]])
    return cache, _rms(_normal(g, 1, Hkv, new, D)), _normal(g, 1, Hkv, new, D)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _layer(s, i):
    tq.sdpa_int4(s["q_"][i], *[t[i] for t in s["cache"]], s["Hq"] // s["Hkv"], 1.0, s["window"], out=s["out"][i])


def run(s):
    kind = s["kind"]
    if kind == "decode":
        return tq.sdpa_int4(s["q_"], *s["cache"], s["Hq"] // s["Hkv"], 1.0, s["window"])
    if kind == "step":
        s["graph"].replay()
        return s["out"]
    if kind == "ragged":
        return tq.sdpa_int4_ragged(s["q_"], *s["cache"], s["lens"], s["Hq"] // s["Hkv"], 1.0, 0,
                                   windows=s["windows"])
    if kind == "prefill":
        tq.kv_append_int4(s["k"], s["v"], *s["cache"], s["at"])
        out = tq.sdpa_int4_prefill(s["q_"], *[t[0] for t in s["cache"]], s["prior"], s["Hq"] // s["Hkv"], 1.0,
                                   s["window"])
        return [out, *s["cache"]]
    if kind == "codec":
        w, sc, b = tq.quantize(s["rows_"], scale_dtype=_DT[s["sb"]])
        return [w, sc, b, tq.dequantize(w, sc, b)]
    if kind == "polar7":
        return s["codec"].sdpa_int4v_q(s["q_"], *s["keys"], *s["v"], 1.0, s["window"])
    if kind == "polar7_encode":
        return list(s["codec"].encode(s["k"]))
    if kind == "polar_codec":
        packed = pq.polar_quantize_packed(s["k"], s["P"], *s["cb"])
        return packed + [pq.polar_dequantize_packed_fast(*packed, *s["cs"], s["D"])]
    scale = 1.0 / math.sqrt(s["D"])
    if s["op"] == "score":
        return pq.compressed_score(s["q_"], *s["keys"], *s["cb"], s["N"], 16, scale, num_kv_heads=s["Hkv"])
    return pq.compressed_sdpa(s["q_"], *s["keys"], *s["cb"], s["v"], 16, scale, num_kv_heads=s["Hkv"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _row(D, sb):
    """Bytes of one token's K and V rows of one kv head."""
    return D + 4 * (D // 64) * _SIZE[sb]


def _seen(prior, new, window):
    """(query, key) pairs of a causal chunk."""
    return sum(min(prior + i + 1, window) if window else prior + i + 1 for i in range(new))


def work(case):
    kind = case["kind"]
    if kind == "codec":
        n = case["rows"] * case["D"]
        packed = n // 2 + n // 64 * 2 * _SIZE[case["sb"]]
        return {"bytes": n * _SIZE[case["x"]] + 2 * packed + 4 * n, "flops": 0}
    if kind == "polar7_encode":
        n = case["rows"]
        return {"bytes": n * (512 + 68) + 2 * 65536, "flops": 2 * 2 * 128 * 128 * n}
    if kind == "polar_codec":
        n, D = case["rows"], case["D"]
        return {"bytes": 2 * n * D * 4 + 2 * n * (D // 16) * 9 + 4 * D * D, "flops": 2 * n * D * D}
    if kind == "polar7":
        n = min(case["L"], case["window"] or case["L"])
        keys = 68 + 64 + 4 * _SIZE[case["sb"]]
        return {"bytes": case["Hkv"] * n * keys + case["Hq"] * 128 * 8, "flops": 6 * 128 * n * case["Hq"]}
    if kind == "compressed":
        rows, D = case["Hkv"] * case["N"], case["D"]
        b = rows * (D // 16) * 17 + case["Hq"] * D * 4
        if case["op"] == "score":
            return {"bytes": b + case["Hq"] * case["N"] * 4, "flops": 2 * D * case["Hq"] * case["N"]}
        return {"bytes": b + rows * D * 4 + case["Hq"] * D * 4, "flops": 4 * D * case["Hq"] * case["N"]}
    Hq, Hkv, D = case["Hq"], case["Hkv"], case["D"]
    io = Hq * D * (_SIZE[case["q"]] + 4)
    if kind == "prefill":
        prior, new, W = case["prior"], case["new"], case["window"]
        first = max(0, prior + 1 - W) if W else 0
        rows = prior + new - first
        b = Hkv * (rows * _row(D, case["sb"]) + new * (8 * D + _row(D, case["sb"]))) + new * io
        return {"bytes": b, "flops": 4 * D * Hq * _seen(prior, new, W)}
    if kind == "ragged":
        lens = _lens(case, 0).tolist()  # the mean over seeds differs little
        keys = sum(min(n, case["window"]) if case["window"] and b % 2 == 0 else n for b, n in enumerate(lens))
        return {"bytes": Hkv * keys * _row(D, case["sb"]) + case["B"] * io, "flops": 4 * D * Hq * keys}
    n = min(case["L"], case["window"] or case["L"])
    k = case.get("layers", 1)
    return {"bytes": k * (Hkv * n * _row(D, case["sb"]) + io), "flops": k * 4 * D * Hq * n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("codec", "polar7_encode"):
        return "exact"
    if kind == "polar_codec":
        # indices and radii are whole decisions; the decoded values are
        # products of four fp32 factors
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    if kind == "polar7":
        return {"rel": 2e-5, "max": 2e-4}
    if kind == "compressed":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 5e-5, "max": 1e-3, "differ": 0.0}


# ---------------------------------------------------------------------------
# results in 64 bits
# ---------------------------------------------------------------------------

def _attend64(q, k, v, keep):
    """q [n, D], k / v [L, D], keep [n, L]: one head's attention."""
    x = (q.double() @ k.t()).masked_fill(~keep, -math.inf)
    return torch.softmax(x, -1) @ v


def _decode64(q, cache, window):
    Hq, Hkv = q.shape[0], cache[0].shape[0]
    n, out = cache[0].shape[1], []
    lo = max(0, n - window) if window else 0
    keep = torch.ones((1, n - lo), dtype=torch.bool, device="cuda")
    for h in range(Hkv):
        k, v = (_rows64(*[t[h, lo:] for t in cache[j:j + 3]]) for j in (0, 3))
        out.append(_attend64(q[h * (Hq // Hkv):(h + 1) * (Hq // Hkv)], k, v, keep))
    return torch.cat(out)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("polar7_encode", "polar_codec"):
        return None
    if kind == "codec":
        g = _gen(seed)
        x = _rms(_normal(g, case["rows"], case["D"])).to(_DT[case["x"]])
        n, sc, b = _mlx_rule(x, _DT[case["sb"]])
        y = n.double().reshape(*sc.shape, 64) * sc.double()[..., None] + b.double()[..., None]
        return [None, sc.double(), b.double(), y.reshape(n.shape)]
    if kind == "prefill":
        g = _gen(seed)
        cache, k, v = _prompt(g, case)
        q = _queries(g, _DT[case["q"]], case["new"], case["Hq"], case["D"])
        for j, x in ((0, k), (3, v)):
            n, sc, b = _mlx_rule(x, _DT[case["sb"]])
            for t, u in zip(cache[j:j + 3], (_pack(n), sc, b)):
                t[:, :, case["prior"]:] = u
        gqa, new, prior, W = case["Hq"] // case["Hkv"], case["new"], case["prior"], case["window"]
        pos = torch.arange(prior, prior + new, device="cuda")[:, None]
        key = torch.arange(prior + new, device="cuda")[None]
        keep = key <= pos
        if W:
            keep &= pos - key < W
        out = torch.empty((new, case["Hq"], case["D"]), dtype=torch.float64, device="cuda")
        for h in range(case["Hkv"]):
            k64, v64 = (_rows64(*[t[0, h] for t in cache[j:j + 3]]) for j in (0, 3))
            for i in range(gqa):
                out[:, h * gqa + i] = _attend64(q[:, h * gqa + i], k64, v64, keep)
        return [out, None, cache[1].double(), cache[2].double(), None, cache[4].double(), cache[5].double()]
    s = prepare(case, seed)
    if kind == "decode":
        return _decode64(s["q_"], s["cache"], case["window"])
    if kind == "step":
        return torch.stack([_decode64(s["q_"][i], [t[i] for t in s["cache"]], case["window"])
                            for i in range(case["layers"])])
    if kind == "ragged":
        return torch.stack([_decode64(s["q_"][b], [t[b, :, :int(n)] for t in s["cache"]], int(w)) for b, (n, w) in
                            enumerate(zip(s["lens"].tolist(), s["windows"].tolist()))])
    if kind == "compressed":
        cb = [c.double() for c in s["cb"]]
        nb, N, G = case["D"] // 16, case["N"], case["Hq"] // case["Hkv"]
        out = []
        for h in range(case["Hkv"]):
            part = slice(h * N * nb, (h + 1) * N * nb)
            idx = [k.view(-1, w)[part] for k, w in zip(s["keys"][:4], (8, 4, 2, 1))]
            k = _untree(idx, cb, s["keys"][4][part].double()).reshape(N, case["D"])
            x = s["q_"][h * G:(h + 1) * G].double() @ k.t() / math.sqrt(case["D"])
            out.append(x if case["op"] == "score" else torch.softmax(x, -1) @ s["v"][h * N:(h + 1) * N].double())
        return torch.cat(out)
    # polar7
    P, S, L, G = s["codec"].P.double(), s["codec"].S.double(), case["L"], case["Hq"] // case["Hkv"]
    cbs, out = [c.float().double() for c in _p7_books()], []
    lo = max(0, L - case["window"]) if case["window"] else 0
    for h in range(case["Hkv"]):
        a, nm, sg = (t[h, lo:].view(torch.int32) for t in s["keys"])
        take = lambda w, width, n: ((w[..., None] >> (torch.arange(32 // width, device="cuda", dtype=torch.int32) *  # noqa: E731
                                                      width)) & ((1 << width) - 1)).flatten(-2)[..., :n]
        last = take(a[:, 11:12], 2, 16)
        idx = [take(a[:, :8], 4, 64), take(a[:, 8:10], 2, 32), take(a[:, 10:11], 2, 16), last[:, :8], last[:, 8:12],
               last[:, 12:14], last[:, 14:15]]
        rad, rn = ((nm >> sh).to(torch.int16).view(torch.float16).double() for sh in (0, 16))
        k = _untree(idx, cbs, rad)
        signs = take(sg, 1, 128).double() * 2 - 1
        q = s["q_"][h * G:(h + 1) * G].double() @ P.t()
        x = q @ k.t() + math.sqrt(math.pi / 2) / 128 * rn[None] * ((q @ S.t()) @ signs.t())
        out.append(torch.softmax(x, -1) @ _rows64(*[t[h, lo:] for t in s["v"]]))
    return torch.cat(out)
