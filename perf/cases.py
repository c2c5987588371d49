"""The work that a user of this framework has it do, as measurable cases.

Each case goes through the public entry points (``dexter_amd.ops``, ``models.SelfAttention``,
``models.KVCache``, ``runtime.capture``). Shapes are those of the Wan-5B (24 heads x 128, hidden
3072, 30 layers, 83-token chunks) and Wan-14B (40 heads x 128, hidden 5120, 913-token chunks)
paths, GR00T's grouped-query backbone (16 query heads over 8) and the other head dims and types
that the attention op takes. ``draw`` gives more cases of the same kinds over the sizes around
them.

Kinds:

* ``append``  one chunk through the QK-norm + rotary prologue and into the KV cache;
* ``step``    a captured control step: ``layers`` x (adaLN, self-attention, gated residual) over
              a cache whose cursor lives in device memory;
* ``layer``   one eager ``SelfAttention`` call that writes its chunk into the cache;
* ``prefill`` prologue, cache write and attention of a whole sequence in one call;
* ``attn``    the attention op alone: over a cache, block-causal, token-causal, cross or
              grouped-query; ``calls`` > 0 captures that many layers' calls into one graph;
* ``ragged``  the attention op over a batch with a cache length per sequence, captured likewise;
* ``norms``   adaLN modulation and gated residual of one activation.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "dexter-labs_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from dexter_amd import ops  # noqa: E402
from dexter_amd.bench.workloads import rope_table  # noqa: E402
from dexter_amd.models.attention import SelfAttention  # noqa: E402
from dexter_amd.models.kv_cache import KVCache  # noqa: E402
from dexter_amd.runtime.graph import capture  # noqa: E402

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
EPS = 1e-6


def _attn(name, lq, heads, dim, *, lk=0, kv_heads=0, cache=0, batch=1, block=0, causal=False,
          dtype="bf16", calls=0):
    """lk 0: as many new keys as queries; block 0: no block boundaries; calls 0: eager."""
    case = {"kind": "attn", "batch": batch, "lq": lq, "lk": lk or lq, "heads": heads,
            "kv_heads": kv_heads or heads, "dim": dim, "cache": cache, "block": block,
            "causal": causal, "dtype": dtype, "calls": calls}
    return {"name": name, **case} if name else case


def listed():
    return [
        # The smallest call: a layer's 83-token chunk rotated and written to the cache, eagerly.
        {"name": "append_chunk_5b", "kind": "append", "batch": 1, "lq": 83, "heads": 24,
         "dim": 128, "cache": 1245, "dtype": "bf16"},
        # The closed control loop: one captured denoising step, 30 layers, 15 blocks of history.
        {"name": "step_5b", "kind": "step", "layers": 30, "lq": 83, "heads": 24, "dim": 128,
         "cache": 1245, "capacity": 1660, "dtype": "bf16"},
        # The final step of a chunk on the larger model, run eagerly: a layer that writes its K/V.
        {"name": "layer_14b", "kind": "layer", "batch": 1, "lq": 83, "heads": 40, "dim": 128,
         "cache": 1245, "dtype": "bf16"},
        # Priming a cache: eight 1,024-token blocks of the 5B model, block-causal.
        {"name": "prefill_5b", "kind": "prefill", "batch": 1, "lq": 8192, "heads": 24,
         "dim": 128, "block": 1024, "dtype": "bf16"},
        # A long chunk of the 14B model over eight cached chunks (odd sizes throughout).
        _attn("chunk_14b", 913, 40, 128, cache=7304),
        # A short chunk late in a long episode: the cache read is the whole cost.
        _attn("decode_long", 83, 24, 128, cache=32768),
        # Four sequences at different points of their episodes, frame + action block, 8 layers.
        {"name": "ragged_batch", "kind": "ragged", "lq": 99, "heads": 24, "dim": 128,
         "cache0": 0, "cache1": 332, "cache2": 1245, "cache3": 3237, "block": 83,
         "dtype": "bf16", "calls": 8},
        # Text conditioning of the 83-token chunk, each of 30 layers onto its own 512 keys.
        _attn("cross_text_5b", 83, 24, 128, lk=512, calls=30),
        # The vision-language backbone's prompt: token-causal, grouped-query, 16 layers.
        _attn("gqa_causal", 300, 16, 128, kv_heads=8, causal=True, calls=16),
        # fp32 runs of the op (the type that results are checked in): four 83-token blocks.
        _attn("fp32_blocks", 332, 24, 128, cache=996, block=83, dtype="f32"),
        # The widest heads the op takes, a 2,048-token sequence.
        _attn("wide_heads", 2048, 16, 256),
        # The element-wise work around attention in every block, over the whole prefill.
        {"name": "norms_prefill", "kind": "norms", "batch": 1, "lq": 8192, "hidden": 3072,
         "dtype": "bf16"},
    ]


# ---------------------------------------------------------------------------
# Drawn cases: the same kinds, sizes log-uniform over the range in use.
# ---------------------------------------------------------------------------
def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _capped(rng, make):
    """A case of `make` that costs no more than the 8K prefill (fp32 products run at a
    sixteenth of the 16-bit rate, and the general head dims at about half of it)."""
    while True:
        case = make(rng)
        w = work(case)
        rate = {"f32": 1 / 12}.get(case["dtype"], 1.0)
        if case.get("dim") in (16, 32, 256):
            rate *= 0.3
        if w["flops"] / rate <= 3.0e11 and w["bytes"] <= 1.2e9:
            return case


def _draw_attn(rng):
    form = rng.choice(["chunk", "chunk", "decode", "causal", "blocks", "cross"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
    if dtype == "f32":
        dim = rng.choice([32, 64, 128, 256])
    else:
        dim = rng.choice([128, 128, 128, 64, 64, 256, 32])
    heads, kv = rng.choice([(24, 24), (40, 40), (16, 8), (12, 12), (16, 16), (16, 4)])
    kw = dict(kv_heads=kv, dtype=dtype)
    if form == "decode":
        return _attn("", _log(rng, 8, 128), heads, dim, cache=_log(rng, 500, 32768),
                     calls=rng.choice([0, 8]), **kw)
    if form == "chunk":
        lq = _log(rng, 64, 1024)
        return _attn("", lq, heads, dim, cache=_log(rng, 200, 8192), calls=rng.choice([0, 4]),
                     block=rng.choice([0, 83]), **kw)
    if form == "causal":
        return _attn("", _log(rng, 100, 4096), heads, dim, causal=True,
                     batch=rng.choice([1, 1, 2, 4]), calls=rng.choice([0, 4]), **kw)
    if form == "blocks":
        lq = _log(rng, 200, 6000)
        return _attn("", lq, heads, dim, block=_log(rng, 64, lq), **kw)
    return _attn("", _log(rng, 32, 4096), heads, dim, lk=_log(rng, 64, 1024),
                 calls=rng.choice([0, 8]), **kw)


def _draw_other(rng):
    kind = rng.choice(["append", "step", "layer", "layer", "prefill", "ragged", "ragged", "norms"])
    heads, dim = rng.choice([(12, 128), (24, 128), (40, 128), (24, 64)])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if kind == "append":
        return {"kind": kind, "batch": rng.choice([1, 1, 2]), "lq": _log(rng, 16, 1024),
                "heads": heads, "dim": dim, "cache": _log(rng, 100, 4000), "dtype": dtype}
    if kind == "step":
        heads = rng.choice([12, 24])
        cache = _log(rng, 83, 3320)
        return {"kind": kind, "layers": rng.randint(4, 12), "lq": _log(rng, 24, 128),
                "heads": heads, "dim": 128, "cache": cache, "capacity": cache + 415,
                "dtype": dtype}
    if kind == "layer":
        return {"kind": kind, "batch": 1, "lq": _log(rng, 16, 512), "heads": heads, "dim": 128,
                "cache": _log(rng, 83, 4000), "dtype": dtype}
    if kind == "prefill":
        lq = _log(rng, 300, 6000)
        return {"kind": kind, "batch": 1, "lq": lq, "heads": heads, "dim": dim,
                "block": _log(rng, 83, lq), "dtype": dtype}
    if kind == "ragged":
        lens = {f"cache{i}": _log(rng, 83, 4000) for i in range(4)}
        return {"kind": kind, "lq": _log(rng, 32, 128), "heads": heads, "dim": dim, **lens,
                "block": rng.choice([0, 83]), "dtype": dtype, "calls": rng.choice([4, 8])}
    return {"kind": kind, "batch": rng.choice([1, 2, 4]), "lq": _log(rng, 83, 8192),
            "hidden": rng.choice([1536, 3072, 5120, 3000]), "dtype": rng.choice(["bf16", "f16", "f32"])}


def draw(rng):
    return _capped(rng, rng.choice([_draw_attn, _draw_other]))


# ---------------------------------------------------------------------------
# Inputs: made on the GPU from the seed alone, shared by prepare() and exact().
# ---------------------------------------------------------------------------
class _Rand:
    def __init__(self, seed, dtype):
        self.g = torch.Generator(device=DEVICE).manual_seed(int(seed))
        self.dtype = dtype

    def __call__(self, *shape, scale=1.0, mean=0.0):
        t = torch.randn(*shape, generator=self.g, device=DEVICE)
        return (t * scale + mean).to(self.dtype)


def _starts(case):
    if not case["block"]:
        return None
    return torch.arange(0, case["lq"], case["block"], dtype=torch.int32, device=DEVICE)


def _tables(first, count, dim):
    cos, sin = rope_table(torch.arange(first, first + count), dim)
    return cos.to(DEVICE), sin.to(DEVICE)


def _cache_lens(case):
    return [case[f"cache{i}"] for i in range(4)]


def _inputs(case, seed):
    kind, dt = case["kind"], DTYPES[case["dtype"]]
    rand = _Rand(seed, dt)
    if kind == "norms":
        b, lq, c = case["batch"], case["lq"], case["hidden"]
        # A Wan block's modulation: [B, 6, 1, C], each row read in place.
        return {"x": rand(b, lq, c), "y": rand(b, lq, c), "mod": rand(b, 6, 1, c, scale=0.3)}
    heads, dim, lq = case["heads"], case["dim"], case["lq"]
    hid = heads * dim
    if kind in ("append", "prefill"):
        b = case["batch"]
        first = case.get("cache", 0)
        cos, sin = _tables(first, lq, dim)
        return {"q": rand(b, lq, heads, dim), "k": rand(b, lq, heads, dim),
                "v": rand(b, lq, heads, dim), "qw": rand(hid, scale=0.1, mean=1.0),
                "kw": rand(hid, scale=0.1, mean=1.0), "cos": cos, "sin": sin, "first": first,
                "starts": _starts(case) if kind == "prefill" else None}
    if kind in ("step", "layer"):
        n = case.get("layers", 1)
        b = case.get("batch", 1)
        cos, sin = _tables(case["cache"], lq, dim)
        layers = []
        for _ in range(n):
            p = {name: (rand(hid, hid, scale=hid ** -0.5), rand(hid, scale=0.02)) for name in "qkvo"}
            p["qn"], p["kn"] = rand(hid, scale=0.1, mean=1.0), rand(hid, scale=0.1, mean=1.0)
            p["hist"] = rand(2, b, case["cache"], heads, dim)
            if kind == "step":
                p["mod"] = rand(b, 3, 1, hid, scale=0.3)
            layers.append(p)
        return {"x": rand(b, lq, hid), "cos": cos, "sin": sin, "layers": layers}
    if kind == "attn":
        b, lk, kv = case["batch"], case["lk"], case["kv_heads"]
        calls = []
        for _ in range(max(case["calls"], 1)):
            calls.append({"q": rand(b, lq, heads, dim), "k": rand(b, lk, kv, dim),
                          "v": rand(b, lk, kv, dim),
                          "cache": rand(2, b, case["cache"], kv, dim) if case["cache"] else None})
        return {"calls": calls, "starts": _starts(case)}
    lens = _cache_lens(case)
    calls = [{"q": rand(4, lq, heads, dim), "k": rand(4, lq, heads, dim),
              "v": rand(4, lq, heads, dim), "cache": rand(2, 4, max(lens), heads, dim)}
             for _ in range(case["calls"])]
    return {"calls": calls, "starts": _starts(case), "lens": lens}


def _module(case, p):
    hid = case["heads"] * case["dim"]
    m = SelfAttention(hid, case["heads"], EPS, dtype=DTYPES[case["dtype"]], device=DEVICE)
    with torch.no_grad():
        for name in "qkvo":
            lin = getattr(m, name)
            lin.weight.copy_(p[name][0])
            lin.bias.copy_(p[name][1])
        m.q_norm.copy_(p["qn"])
        m.k_norm.copy_(p["kn"])
    return m


def prepare(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    s["case"] = case
    dt = DTYPES[case["dtype"]]
    if kind in ("append", "prefill"):
        rows = s["first"] + case["lq"]
        s["cache"] = torch.zeros(2, case["batch"], rows, case["heads"], case["dim"],
                                 device=DEVICE, dtype=dt)
        return s
    if kind in ("step", "layer"):
        n = len(s["layers"])
        cap = case.get("capacity", case["cache"] + case["lq"])
        kv = KVCache(n, case.get("batch", 1), cap, case["heads"], case["dim"], DEVICE, dt,
                     device_cursor=kind == "step")
        modules, mods = [], []
        for i, p in enumerate(s.pop("layers")):
            kv.cache[i][:, :, :case["cache"]].copy_(p["hist"])
            modules.append(_module(case, p))
            mods.append(p.get("mod"))
        kv.commit(case["cache"])
        s.update(kv=kv, modules=modules)
        if kind == "step":
            cos, sin = s["cos"], s["sin"]

            @torch.no_grad()
            def step(x):
                for i, (m, mod) in enumerate(zip(modules, mods)):
                    shift, scale, gate = mod[:, 0], mod[:, 1], mod[:, 2]
                    y = m(ops.adaln_modulate(x, scale, shift), cos, sin, kv, i)
                    x = ops.gated_residual(x, y, gate)
                return x

            s["runner"] = capture(step, (s["x"],))
        return s
    if kind == "attn" and case["calls"]:
        s["runner"] = capture(lambda: tuple(_attend(case, c, s["starts"]) for c in s["calls"]), ())
    if kind == "ragged":
        s["runner"] = capture(lambda: tuple(
            ops.blockwise_causal_attention_varlen(
                c["q"], c["k"], c["v"], kv_cache=c["cache"], cache_lens=s["lens"],
                block_boundaries=s["starts"]) for c in s["calls"]), ())
    return s


def _attend(case, c, starts):
    return ops.blockwise_causal_attention(
        c["q"], c["k"], c["v"], kv_cache=c["cache"], cache_len=case["cache"],
        block_boundaries=starts, causal=case["causal"])


def run(state):
    case = state["case"]
    kind = case["kind"]
    s = state
    if kind == "append":
        q, k = ops.qk_norm_rope_append(s["q"], s["k"], s["v"], s["qw"], s["kw"], s["cos"],
                                       s["sin"], s["cache"], s["first"], EPS)
        return {"q": q, "k": k, "rows": s["cache"][:, :, s["first"]:]}
    if kind == "prefill":
        out = ops.qk_norm_rope_attention(
            s["q"], s["k"], s["v"], s["qw"], s["kw"], s["cos"], s["sin"], kv_cache=s["cache"],
            cache_len=0, append=True, block_boundaries=s["starts"], eps=EPS)
        return {"out": out, "cache": s["cache"]}
    if kind == "step":
        return s["runner"](s["x"])[0]
    if kind == "layer":
        out = s["modules"][0](s["x"], s["cos"], s["sin"], s["kv"], 0, write=True)
        return {"out": out, "rows": s["kv"].cache[0][:, :, case["cache"]:]}
    if kind == "norms":
        mod = s["mod"]
        h = ops.adaln_modulate(s["x"], mod[:, 1], mod[:, 0], EPS)
        return {"h": h, "x": ops.gated_residual(s["x"], s["y"], mod[:, 2])}
    if "runner" in s:
        return list(s["runner"]())
    return [_attend(case, s["calls"][0], s["starts"])]


# ---------------------------------------------------------------------------
# What one pass cannot do without.
# ---------------------------------------------------------------------------
def _pairs(lq, lk, cache, block, causal):
    if causal:
        return lq * cache + lq * (lq + 1) // 2
    if block:
        return sum((min(lo + block, lq) - lo) * (cache + min(lo + block, lq))
                   for lo in range(0, lq, block))
    return lq * (cache + lk)


def work(case):
    kind = case["kind"]
    es = 4 if case["dtype"] == "f32" else 2
    if kind == "norms":
        n = case["batch"] * case["lq"] * case["hidden"]
        return {"bytes": 5 * n * es, "flops": 12 * n}
    heads, dim, lq = case["heads"], case["dim"], case["lq"]
    hid = heads * dim
    b = case.get("batch", 1)
    if kind == "append":
        n = b * lq * hid
        return {"bytes": (3 + 4) * n * es, "flops": 20 * n}
    if kind == "prefill":
        return {"bytes": (3 + 1 + 2) * b * lq * hid * es,
                "flops": 4 * dim * heads * b * _pairs(lq, lq, 0, case["block"], False)}
    if kind in ("step", "layer"):
        rows = b * lq
        per = {"bytes": 4 * hid * hid * es + 2 * b * case["cache"] * hid * es
               + (2 if kind == "layer" else 0) * rows * hid * es,
               "flops": 2 * rows * hid * 4 * hid
               + 4 * dim * heads * b * lq * (case["cache"] + lq)}
        n = case.get("layers", 1)
        return {"bytes": n * per["bytes"] + 2 * rows * hid * es, "flops": n * per["flops"]}
    if kind == "attn":
        kv = 2 * (case["cache"] + case["lk"]) * case["kv_heads"] * dim
        n = max(case["calls"], 1) * b
        return {"bytes": n * (2 * lq * hid + kv) * es,
                "flops": n * 4 * dim * heads * _pairs(lq, case["lk"], case["cache"],
                                                      case["block"], case["causal"])}
    lens = _cache_lens(case)
    return {"bytes": case["calls"] * es * hid * sum(2 * lq + 2 * (c + lq) for c in lens),
            "flops": case["calls"] * 4 * dim * heads
            * sum(_pairs(lq, lq, c, case["block"], False) for c in lens)}


def tolerance(case):
    """Relative errors that another correct implementation at the same precision shows."""
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 2e-4}
    if case["kind"] == "step":
        return {"rel": 3e-2, "max": 2e-1}
    return {"rel": 1e-2, "max": 1e-1}


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch.
# ---------------------------------------------------------------------------
def _attend64(q, k, v, cache, cache_len, starts, causal):
    """softmax(q k^T / sqrt(D)) v over [cache[:cache_len] | k], [B, L, H, D] in, out in fp64."""
    b, lq, heads, dim = q.shape
    lk, group = k.shape[1], heads // k.shape[2]
    ends = torch.full((lq,), lk, device=q.device)
    if causal:
        ends = torch.arange(1, lq + 1, device=q.device)
    elif starts is not None:
        bounds = starts.tolist() + [lq]
        for lo, hi in zip(bounds[:-1], bounds[1:]):
            ends[lo:hi] = hi
    cols = torch.arange(cache_len + lk, device=q.device)
    hidden = cols[None, :] >= (cache_len + ends)[:, None]
    out = torch.empty(b, lq, heads, dim, dtype=torch.float64, device=q.device)
    for i in range(b):
        for h in range(heads):
            kh, vh = k[i, :, h // group], v[i, :, h // group]
            if cache_len:
                kh = torch.cat((cache[0, i, :cache_len, h // group], kh))
                vh = torch.cat((cache[1, i, :cache_len, h // group], vh))
            s = q[i, :, h].double() @ kh.double().t().contiguous() / math.sqrt(dim)
            s.masked_fill_(hidden, -math.inf)
            out[i, :, h] = torch.softmax(s, -1) @ vh.double()
    return out


def _norm_rope64(x, w, cos, sin):
    """RMS norm over the whole H*D plane, then rotation of the pairs (2j, 2j+1)."""
    b, lq, heads, dim = x.shape
    x = x.double()
    x = x * torch.rsqrt(x.square().mean((2, 3), keepdim=True) + EPS) * w.double().view(heads, dim)
    c, s = cos.double()[None, :, None], sin.double()[None, :, None]
    even, odd = x[..., 0::2], x[..., 1::2]
    return torch.stack((even * c - odd * s, even * s + odd * c), -1).flatten(-2)


def _adaln64(x, scale, shift):
    x = x.double()
    d = x - x.mean(-1, keepdim=True)
    n = d * torch.rsqrt(d.square().mean(-1, keepdim=True) + EPS)
    return n * (1 + scale.double()) + shift.double()


def _layer64(case, x, p, cos, sin):
    b, lq, hid = x.shape
    shape = (b, lq, case["heads"], case["dim"])
    rows = x.double().reshape(-1, hid)
    q, k, v = ((rows @ p[n][0].double().t().contiguous() + p[n][1].double()).view(shape)
               for n in "qkv")
    q, k = _norm_rope64(q, p["qn"], cos, sin), _norm_rope64(k, p["kn"], cos, sin)
    out = _attend64(q, k, v, p["hist"].double(), case["cache"], None, False)
    out = out.reshape(-1, hid) @ p["o"][0].double().t().contiguous() + p["o"][1].double()
    return out.view(b, lq, hid), k, v


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    if kind == "norms":
        mod = s["mod"]
        return {"h": _adaln64(s["x"], mod[:, 1], mod[:, 0]),
                "x": s["x"].double() + s["y"].double() * mod[:, 2].double()}
    if kind in ("append", "prefill"):
        q = _norm_rope64(s["q"], s["qw"], s["cos"], s["sin"])
        k = _norm_rope64(s["k"], s["kw"], s["cos"], s["sin"])
        rows = torch.stack((k, s["v"].double()))
        if kind == "append":
            return {"q": q, "k": k, "rows": rows}
        return {"out": _attend64(q, k, s["v"], None, 0, s["starts"], False), "cache": rows}
    if kind == "layer":
        out, k, v = _layer64(case, s["x"], s["layers"][0], s["cos"], s["sin"])
        return {"out": out, "rows": torch.stack((k, v))}
    if kind == "step":
        x = s["x"].double()
        for p in s["layers"]:
            shift, scale, gate = (p["mod"][:, i].double() for i in range(3))
            y, _, _ = _layer64(case, _adaln64(x, scale, shift), p, s["cos"], s["sin"])
            x = x + y * gate
        return x
    if kind == "attn":
        return [_attend64(c["q"], c["k"], c["v"], c["cache"], case["cache"], s["starts"],
                          case["causal"]) for c in s["calls"]]
    outs = []
    for c in s["calls"]:
        outs.append(torch.cat([
            _attend64(c["q"][i:i + 1], c["k"][i:i + 1], c["v"][i:i + 1], c["cache"][:, i:i + 1],
                      n, s["starts"], False) for i, n in enumerate(s["lens"])]))
    return outs
