"""The work that programs have this KV-cache engine do, one layer's call at a time.

Six kinds of call, each through the package's public entry points:

  decode    one new token over a per-layer cache (attention_with_cache_update)
  chunk     a chunk of a prompt over a per-layer cache (attention_with_cache_update)
  paged     a continuous-batching step over a block pool: the append of the step's
            tokens, the decode of every sequence, and the attention of one
            sequence's prefill chunk
  mla       a latent-cache decode step: the append and the absorbed decode
  compress  a float cache turned into a TurboQuant cache (encode and decode)
  quantize  a float cache turned into an affine 4- / 8-bit cache

The listed sizes are those of the repository's benchmark and tests; draw() takes
others of the same ranges.  Run from the repository's root.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "vmlx-swift_amd"))
import vkv  # noqa: E402

GROUP = 64          # affine group size
BLOCK = 32          # tokens per pool block
MLA_BLOCK = 64      # tokens per latent page
LATENT, ROPE = 512, 64
DECODE_RUN = 64     # decode tokens before a decode case's cache is trimmed back

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
CODES = {"f16": vkv.F16, "bf16": vkv.BF16}


def listed():
    return [
        # A short chat's decode step on one layer, batch 1: launch latency.
        dict(name="decode_f16_b1_512", kind="decode", cache="simple", dtype="f16", B=1, Hq=32,
             Hkv=8, D=128, T=512, bits=0, window=0),
        # Eight long conversations decoded together over float caches of an
        # odd length: bandwidth.
        dict(name="decode_bf16_b8_6001", kind="decode", cache="simple", dtype="bf16", B=8, Hq=32,
             Hkv=8, D=128, T=6001, bits=0, window=0),
        # A sliding-window layer (ring of 1024) in steady-state decode.
        dict(name="decode_window_b4_1024", kind="decode", cache="rotating", dtype="bf16", B=4,
             Hq=16, Hkv=8, D=256, T=1123, bits=0, window=1024),
        # A layer of an 8B model's 4-bit cache, batch 8 at 4096 tokens.
        dict(name="decode_q4_b8_4096", kind="decode", cache="quantized", dtype="bf16", B=8, Hq=32,
             Hkv=8, D=128, T=4096, bits=4, window=0),
        # The global layer of a sliding-window model: 8-bit, 32768 tokens.
        dict(name="decode_q8_b4_32768", kind="decode", cache="quantized", dtype="bf16", B=4, Hq=16,
             Hkv=8, D=256, T=32768, bits=8, window=0),
        # Continuous batching: 64 sequences of 128-8192 tokens, half of them
        # behind a shared 2048-token prefix, and a 512-token prefill chunk.
        dict(name="paged_q4_64x8192", kind="paged", dtype="bf16", n=64, lo=128, hi=8192, share=2048,
             chunk=512, bits=4, Hq=32, Hkv=8, D=128),
        # The same engine over unquantized blocks, 16 sequences, no chunk.
        dict(name="paged_bf16_16x4096", kind="paged", dtype="bf16", n=16, lo=128, hi=4096, share=0,
             chunk=0, bits=0, Hq=32, Hkv=8, D=128),
        # A 512-token prompt chunk behind 4096 tokens of a 4-bit cache.
        dict(name="chunk_q4_512_4096", kind="chunk", cache="quantized", dtype="bf16", B=1, Hq=32,
             Hkv=8, D=128, T=4096, L=512, bits=4, window=0, mask="causal"),
        # A 512-token prompt chunk on a sliding-window layer, under the array
        # mask that the layer's cache makes for it.
        dict(name="chunk_window_512_1024", kind="chunk", cache="rotating", dtype="bf16", B=1, Hq=16,
             Hkv=8, D=256, T=1500, L=512, bits=0, window=1024, mask="cache"),
        # Latent-cache decode, 32 sequences of 16384 tokens, 128 heads.
        dict(name="mla_32x16384", kind="mla", n=32, lo=16384, hi=16384, H=128),
        # A layer's cache of 8 prompts of 4096 tokens compressed with the
        # codec's default bits.
        dict(name="compress_bf16_b8_4096", kind="compress", dtype="bf16", B=8, Hkv=8, D=128, T=4096,
             key_bits=3, value_bits=3),
        # A layer's float cache quantized in mid-generation.
        dict(name="quantize_bf16_b8_4096", kind="quantize", dtype="bf16", B=8, Hkv=8, D=128, T=4096,
             bits=4),
    ]


# (query heads, kv heads, head dim) of the tests' and benchmark's layers
HEADS = [(32, 8, 128), (32, 8, 128), (16, 8, 256), (32, 8, 64), (8, 8, 128), (24, 8, 128),
         (64, 8, 128)]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "chunk", "chunk", "paged", "paged", "mla",
                       "compress", "quantize"])
    Hq, Hkv, D = rng.choice(HEADS)
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if kind in ("decode", "chunk"):
        cache = rng.choice(["simple", "rotating", "quantized", "quantized"])
        c = dict(kind=kind, cache=cache, dtype=dtype, B=_log(rng, 1, 8), Hq=Hq, Hkv=Hkv, D=D,
                 T=_log(rng, 100, 32768), bits=rng.choice([4, 8]) if cache == "quantized" else 0,
                 window=rng.choice([512, 1024, 2048, 4096]) if cache == "rotating" else 0)
        if cache == "rotating":
            c["T"] = _log(rng, c["window"] + 1, 3 * c["window"])
        if kind == "chunk":
            # models pass the causal mode, or the mask their cache makes
            # (an array behind earlier tokens, or for a window)
            c["L"] = _log(rng, 16, 1024)
            c["mask"] = "cache" if cache == "rotating" else rng.choice(["causal", "cache"])
        return c
    if kind == "paged":
        hi = _log(rng, 256, 8192)
        bits = rng.choice([0, 4, 4, 8])
        return dict(kind=kind, dtype="bf16", n=_log(rng, 1, 64), lo=rng.randint(1, 128), hi=hi,
                    share=rng.choice([0, BLOCK * (hi // 4 // BLOCK)]),
                    chunk=rng.choice([0, _log(rng, 16, 512)]) if bits else 0, bits=bits, Hq=Hq,
                    Hkv=Hkv, D=D)
    if kind == "mla":
        hi = _log(rng, 512, 16384)
        return dict(kind=kind, n=_log(rng, 1, 32), lo=rng.randint(hi // 8, hi), hi=hi,
                    H=rng.choice([16, 64, 128, 128]))
    T = _log(rng, 256, 4096)
    if kind == "compress":
        return dict(kind=kind, dtype=dtype, B=_log(rng, 1, 8), Hkv=8, D=rng.choice([64, 128, 128, 256]),
                    T=T, key_bits=rng.choice([3, 4]), value_bits=rng.choice([3, 4]))
    return dict(kind=kind, dtype=dtype, B=_log(rng, 1, 8), Hkv=8, D=D, T=T, bits=rng.choice([4, 8]))


def draw(rng):
    most = {}
    for c in listed():
        w = work(c)
        b, f = most.get(c["kind"], (0.0, 0.0))
        most[c["kind"]] = (max(b, w["bytes"]), max(f, w["flops"]))
    while True:
        c = _draw(rng)
        w = work(c)
        b, f = most[c["kind"]]
        if w["bytes"] <= b and w["flops"] <= f:
            return c


# ------------------------------------------------------------------ work

def _seq_lens(c):
    """The sequences' lengths before the step (fixed by the case) and which
    of them share the prefix (half of those longer than it)."""
    r = random.Random(c["n"] * 100003 + c["lo"] * 31 + c["hi"])
    lens = [r.randint(min(c["lo"], c["hi"]), c["hi"]) for _ in range(c["n"])]
    share = c.get("share", 0)
    sharers = [i for i in range(c["n"]) if share and lens[i] > share][:c["n"] // 2]
    return lens, sharers if len(sharers) > 1 else []


def _token_bytes(c):
    """Stored bytes of one token's K and V of one kv head."""
    if c["bits"]:
        return 2 * (c["D"] * c["bits"] // 8 + c["D"] // GROUP * 4)
    return 2 * c["D"] * 2


def work(c):
    kind = c["kind"]
    if kind in ("decode", "chunk"):
        L = c.get("L", 1)
        T, W = c["T"], c["window"]
        keys = min(T + L, W - 1 + L) if W else T + L       # keys the call attends
        if W:
            seen = sum(min(W, T + l + 1) for l in range(L))
        else:
            seen = L * T + L * (L + 1) // 2
        row = c["B"] * c["D"] * L * 2
        return {"bytes": c["B"] * c["Hkv"] * keys * _token_bytes(c) + row * 2 * c["Hq"]
                + row * 2 * c["Hkv"],
                "flops": 4.0 * c["B"] * c["Hq"] * c["D"] * seen}
    if kind == "paged":
        lens, sharers = _seq_lens(c)
        total = sum(lens) + c["n"]
        unique = total - c["share"] * max(0, len(sharers) - 1)
        L = c["chunk"]
        new = (c["n"] + L) * c["D"] * 2
        return {"bytes": c["Hkv"] * (unique + L) * _token_bytes(c) + new * 2 * c["Hkv"]
                + new * 2 * c["Hq"],
                "flops": 4.0 * c["Hq"] * c["D"] * (total + L * (L + 1) // 2)}
    if kind == "mla":
        lens, _ = _seq_lens(c)
        total = sum(lens) + c["n"]
        ent = LATENT + ROPE
        return {"bytes": total * (ent + ent // GROUP * 4) + c["n"] * ent * 2
                + c["n"] * c["H"] * (ent + LATENT) * 2,
                "flops": 2.0 * c["H"] * total * (ent + LATENT)}
    rows = c["B"] * c["Hkv"] * c["T"]
    if kind == "compress":
        # read K and V, write the records and the decoded f16 / f32 rows; a
        # key's two D x D products and the rotations of both, each way
        D = c["D"]
        out = 4 if c["dtype"] == "bf16" else 2
        records = D * (c["key_bits"] + c["value_bits"]) / 8 + 6
        return {"bytes": rows * (2 * D * 2 + records + 2 * D * out),
                "flops": rows * (4.0 * D * D + 4 * D * math.log2(D))}
    return {"bytes": rows * (2 * c["D"] * 2 + _token_bytes(c)), "flops": 10.0 * rows * c["D"]}


# ------------------------------------------------------------------ inputs

def _inputs(c, seed):
    """The case's tensors, from the seed alone (standard normal rows; the
    quantized decode caches have 4 value and key channels a head at 20 times
    that, as real caches have outliers)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, dtype=torch.bfloat16):
        return torch.randn(shape, generator=g, device="cuda", dtype=dtype)

    kind = c["kind"]
    if kind in ("decode", "chunk"):
        dt, L = DTYPES[c["dtype"]], c.get("L", 1)
        kv = (c["B"], c["Hkv"])
        x = dict(k0=normal(*kv, c["T"], c["D"], dtype=dt), v0=normal(*kv, c["T"], c["D"], dtype=dt),
                 q=normal(c["B"], c["Hq"], L, c["D"], dtype=dt), k=normal(*kv, L, c["D"], dtype=dt),
                 v=normal(*kv, L, c["D"], dtype=dt))
        if kind == "decode" and c["bits"]:
            m = torch.ones((*kv, 1, c["D"]), device="cuda", dtype=dt)
            ch = torch.rand((*kv, 1, c["D"]), device="cuda", generator=g).argsort(-1)[..., :4]
            m.scatter_(-1, ch, 20.0)
            x["k0"] *= m
            x["v0"] *= m
        return x
    if kind == "paged":
        dt = DTYPES[c["dtype"]]
        lens, sharers = _seq_lens(c)
        own = [n - (c["share"] if i in sharers[1:] else 0) for i, n in enumerate(lens)]
        x = dict(k0=normal(sum(own), c["Hkv"], c["D"], dtype=dt),
                 v0=normal(sum(own), c["Hkv"], c["D"], dtype=dt),
                 q=normal(c["n"], c["Hq"], c["D"], dtype=dt),
                 k=normal(c["n"] + c["chunk"], c["Hkv"], c["D"], dtype=dt),
                 v=normal(c["n"] + c["chunk"], c["Hkv"], c["D"], dtype=dt), order=None)
        if c["chunk"]:
            x["cq"] = normal(1, c["Hq"], c["chunk"], c["D"], dtype=dt)
        blocks = sum((n + 1 + BLOCK - 1) // BLOCK + 1 for n in lens) + c["chunk"] // BLOCK + 2
        x["order"] = torch.randperm(blocks, device="cuda", generator=g).int()
        return x
    if kind == "mla":
        lens, _ = _seq_lens(c)
        blocks = sum((n + MLA_BLOCK) // MLA_BLOCK for n in lens)
        ent = LATENT + ROPE
        return dict(x0=normal(sum(lens), 1, ent) * 0.5, x=normal(c["n"], 1, ent) * 0.5,
                    q=normal(c["n"], c["H"], ent),
                    order=torch.randperm(blocks, device="cuda", generator=g).int())
    dt = DTYPES[c["dtype"]]
    shape = (c["B"], c["Hkv"], c["T"], c["D"])
    return dict(k0=normal(*shape, dtype=dt), v0=normal(*shape, dtype=dt))


def _slots(table, pos, size):
    """Pool slots of positions `pos` of a sequence with this block table."""
    return table[pos // size] * size + (pos % size).int()


def _paged_layout(c, order):
    """Block tables, the slots of the stored tokens in the inputs' order,
    of the decode tokens and of the chunk."""
    lens, sharers = _seq_lens(c)
    at, tables, shared = 0, [], None
    dev = order.device
    for i, n in enumerate(lens):
        nb = (n + 1 + BLOCK - 1) // BLOCK
        keep = c["share"] // BLOCK if i in sharers[1:] else 0
        own = order[at:at + nb - keep]
        at += nb - keep
        tables.append(torch.cat([shared[:keep], own]) if keep else own)
        if sharers and i == sharers[0]:
            shared = tables[-1]
    fill, dec = [], []
    for i, n in enumerate(lens):
        first = c["share"] if i in sharers[1:] else 0
        fill.append(_slots(tables[i], torch.arange(first, n, device=dev), BLOCK))
        dec.append(_slots(tables[i], torch.arange(n, n + 1, device=dev), BLOCK))
    nb = (c["chunk"] + BLOCK - 1) // BLOCK
    ctable = order[at:at + nb]
    if c["chunk"]:
        dec.append(_slots(ctable, torch.arange(c["chunk"], device=dev), BLOCK))
    width = max(len(t) for t in tables)
    table = torch.zeros((c["n"], width), dtype=torch.int32, device=dev)
    for i, t in enumerate(tables):
        table[i, :len(t)] = t
    return lens, table, ctable, torch.cat(fill).int(), torch.cat(dec).int()


def _make_cache(c):
    if c["cache"] == "simple":
        return vkv.KVCacheSimple()
    if c["cache"] == "rotating":
        return vkv.RotatingKVCache(c["window"])
    return vkv.QuantizedKVCache(group_size=GROUP, bits=c["bits"])


def prepare(c, seed):
    x = _inputs(c, seed)
    kind = c["kind"]
    if kind in ("decode", "chunk"):
        cache = _make_cache(c)
        fill = cache.update_quantized if c["bits"] else cache.update
        fill(x["k0"], x["v0"])
        s = dict(case=c, cache=cache, q=x["q"], k=x["k"], v=x["v"], scale=c["D"] ** -0.5, steps=0)
        if kind == "chunk":
            # the mask a model makes once for all layers of a kind
            s["mask"] = c["mask"] if c["mask"] == "causal" else cache.make_mask(
                c["L"], window_size=c["window"] or None)
        return s
    if kind == "paged":
        lens, table, ctable, fill, new = _paged_layout(c, x["order"])
        pool = vkv.PagedPool(len(x["order"]), BLOCK, 1, c["Hkv"], c["D"], dtype=CODES[c["dtype"]],
                             bits=c["bits"])
        pool.append(0, x["k0"], x["v0"], fill)
        dev = dict(dtype=torch.int32, device="cuda")
        view = pool.view(0, table, torch.tensor([n + 1 for n in lens], **dev), max(lens) + 1)
        s = dict(case=c, pool=pool, view=view, new=new, q=x["q"], k=x["k"], v=x["v"],
                 scale=c["D"] ** -0.5)
        if c["chunk"]:
            s["cq"] = x["cq"]
            s["cview"] = pool.view(0, ctable.view(1, -1).contiguous(),
                                   torch.tensor([c["chunk"]], **dev), c["chunk"])
        return s
    if kind == "mla":
        lens, _ = _seq_lens(c)
        pool = vkv.PagedPool(len(x["order"]), MLA_BLOCK, 1, 1, LATENT + ROPE, dtype=vkv.BF16, bits=8,
                             group_size=GROUP, v_head_dim=LATENT, flags=vkv.VIEW_KEYS_ONLY)
        width = max((n + MLA_BLOCK) // MLA_BLOCK for n in lens)
        table = torch.zeros((c["n"], width), dtype=torch.int32, device="cuda")
        fill, new, at = [], [], 0
        for i, n in enumerate(lens):
            nb = (n + MLA_BLOCK) // MLA_BLOCK
            t = x["order"][at:at + nb]
            at += nb
            table[i, :nb] = t
            fill.append(_slots(t, torch.arange(n, device="cuda"), MLA_BLOCK))
            new.append(_slots(t, torch.arange(n, n + 1, device="cuda"), MLA_BLOCK))
        pool.append(0, x["x0"], None, torch.cat(fill).int())
        view = pool.view(0, table, torch.tensor([n + 1 for n in lens], dtype=torch.int32,
                                                device="cuda"), max(lens) + 1)
        return dict(case=c, pool=pool, view=view, new=torch.cat(new).int(), q=x["q"], x=x["x"],
                    scale=192 ** -0.5)
    cache = vkv.KVCacheSimple()
    cache.update(x["k0"], x["v0"])
    return dict(case=c, cache=cache)


# ------------------------------------------------------------------ one pass

def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "decode":
        out = vkv.attention_with_cache_update(s["q"], s["k"], s["v"], s["cache"], s["scale"])
        if not c["window"]:
            s["steps"] += 1
            if s["steps"] == DECODE_RUN:
                s["cache"].trim(DECODE_RUN)
                s["steps"] = 0
        return out
    if kind == "chunk":
        out = vkv.attention_with_cache_update(s["q"], s["k"], s["v"], s["cache"], s["scale"],
                                              mask=s["mask"])
        if not c["window"]:
            s["cache"].trim(c["L"])
        return out
    if kind == "paged":
        s["pool"].append(0, s["k"], s["v"], s["new"])
        out = vkv.paged_attention(s["q"], s["view"], s["scale"])
        if not c["chunk"]:
            return out
        return out, vkv.quantized_paged_attention(s["cq"], s["cview"], s["scale"], mask="causal")
    if kind == "mla":
        s["pool"].append(0, s["x"], None, s["new"])
        return vkv.mla_decode(s["q"], s["view"], s["scale"])
    if kind == "compress":
        tq = vkv.TurboQuantKVCache.from_simple_cache(s["cache"], c["key_bits"], c["value_bits"])
        k, v = tq.encoded()
        keep = ("indices", "qjl", "res_norms", "vec_norms", "sink", "tail")
        return {"keys": [k[n] for n in keep], "values": [v[n] for n in keep], "state": tq.state}
    return s["cache"].to_quantized(GROUP, c["bits"]).state


# ------------------------------------------------------------------ 64 bits

def _affine(x, bits):
    """Codes, scales and biases (rounded to x's type) of groups of 64.  In 32
    bits, operation for operation: the formula rounds edge / scale to a whole
    number, which 16-bit inputs often leave half way between two, and the
    codes are defined by the 32-bit arithmetic."""
    n = 2 ** bits - 1
    w = x.float().unflatten(-1, (-1, GROUP))
    lo, hi = w.amin(-1, keepdim=True), w.amax(-1, keepdim=True).clamp_min(0)
    # (a division by a number would become a product with its reciprocal)
    scale = ((hi - lo) / torch.full_like(hi, n)).clamp_min(1e-7)
    side = lo.abs() > hi.abs()
    scale = torch.where(side, scale, -scale)
    edge = torch.where(side, lo, hi)
    half_up = lambda t: torch.sign(t) * torch.floor(t.abs() + 0.5)  # noqa: E731
    q0 = half_up(edge / scale)
    zero = q0 == 0
    scale = torch.where(zero, scale, edge / torch.where(zero, torch.ones_like(q0), q0))
    bias = torch.where(zero, torch.zeros_like(edge), edge)
    code = half_up((w - bias) / scale).clamp(0, n)
    return code.double(), scale.to(x.dtype).double(), bias.to(x.dtype).double()


def _stored(x, bits, rounded):
    """What a cache of `bits` holds of x, in 64 bits (rounded: dequantized to
    x's type, as a chunk's attention reads it)."""
    if not bits:
        return x.double()
    code, scale, bias = _affine(x, bits)
    y = (scale * code + bias).flatten(-2)
    return y.to(x.dtype).double() if rounded else y


def _attend(q, k, v, scale, quantized, seen=None):
    """Attention of q [Hq, L, D] over k, v [Hkv, T, D] in 64 bits.  Over a
    quantized cache the scaled queries and the scores are stored in q's type
    (the reference's quantizedScaledDotProductAttention); seen [L, T]."""
    Hq, L, D = q.shape
    Hkv = k.shape[0]
    if quantized:
        st = torch.tensor(scale).to(q.dtype).float().to(q.device)
        q = (q.float() * st).to(q.dtype)
        scale = 1.0
    s = torch.matmul(q.double().reshape(Hkv, -1, D), k.transpose(1, 2).contiguous()) * scale
    if quantized:
        s = s.to(q.dtype).double()
    if seen is not None:
        s = s.view(Hkv, -1, L, k.shape[1]).masked_fill(~seen, -math.inf).view(Hkv, -1, k.shape[1])
    return torch.matmul(torch.softmax(s, -1), v).reshape(Hq, L, v.shape[2])


def exact(c, seed):
    kind = c["kind"]
    if kind == "compress":
        return None  # the codec's own tables define its values; its outputs are compared bit by bit
    x = _inputs(c, seed)
    if kind in ("decode", "chunk"):
        L, W, quant = c.get("L", 1), c["window"], c["bits"] > 0
        k, v = (torch.cat([x[n + "0"], x[n]], 2) for n in "kv")
        if W:
            k, v = (t[:, :, -(W - 1 + L):] for t in (k, v))
        T = k.shape[2]
        seen = None
        if L > 1 or W:
            pos = torch.arange(T - L, T, device="cuda")[:, None]
            key = torch.arange(T, device="cuda")[None]
            seen = key <= pos
            if W:
                seen &= key > pos - W
        scale, rounded = c["D"] ** -0.5, L > 1
        return torch.stack([_attend(x["q"][b], _stored(k[b], c["bits"], rounded),
                                    _stored(v[b], c["bits"], rounded), scale, quant, seen)
                            for b in range(c["B"])])
    if kind == "paged":
        lens, sharers = _seq_lens(c)
        scale, quant, out, at, prefix = c["D"] ** -0.5, c["bits"] > 0, [], 0, None
        for i, n in enumerate(lens):
            first = c["share"] if i in sharers[1:] else 0
            k, v = (x[m + "0"][at:at + n - first] for m in "kv")
            at += n - first
            if first:
                k, v = torch.cat([prefix[0], k]), torch.cat([prefix[1], v])
            if sharers and i == sharers[0]:
                prefix = k[:c["share"]], v[:c["share"]]
            k, v = (torch.cat([t, x[m][i:i + 1]]).transpose(0, 1) for m, t in (("k", k), ("v", v)))
            out.append(_attend(x["q"][i][:, None], _stored(k, c["bits"], False),
                               _stored(v, c["bits"], False), scale, quant)[:, 0])
        out = torch.stack(out)
        if not c["chunk"]:
            return out
        k, v = (_stored(x[m][c["n"]:].transpose(0, 1), c["bits"], True) for m in "kv")
        seen = torch.ones((c["chunk"],) * 2, dtype=torch.bool, device="cuda").tril()
        return out, _attend(x["cq"][0], k, v, scale, quant, seen)[None]
    if kind == "mla":
        lens, _ = _seq_lens(c)
        out, at = [], 0
        for i, n in enumerate(lens):
            e = torch.cat([x["x0"][at:at + n], x["x"][i:i + 1]])[:, 0]
            at += n
            e = _stored(e, 8, True)[None]
            out.append(_attend(x["q"][i][:, None], e, e[..., :LATENT], 192 ** -0.5, False)[:, 0])
        return torch.stack(out)
    out = []
    for t in (x["k0"], x["v0"]):
        _, scale, bias = _affine(t, c["bits"])
        out += [None, scale.squeeze(-1), bias.squeeze(-1)]
    return out


def tolerance(c):
    # whole numbers and stored bits: the codec's records and decoded rows, an
    # affine cache's codes, scales and biases
    if c["kind"] in ("compress", "quantize"):
        return "exact"
    # four times what the calls show against exact(): the rounding of the
    # outputs (1.7e-3 in bf16, 2.1e-4 to 4.3e-4 in f16) and of probabilities
    return {"rel": 2e-3 if c.get("dtype") == "f16" else 8e-3}
