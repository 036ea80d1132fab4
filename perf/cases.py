"""The calls whose speed matters to a user of this package, with the sizes they are made at.

Six kinds of call, each through the entry point that a serving program uses:

``step``        one decode step of a few layers through the paged cache, as an engine
                makes it: ``PagedPackedCache`` over the pool's leases, then per layer
                ``update`` (append) and ``winnow_packed_attention`` (decode).
``decode``      ``packed_decode_attention``: one query token per sequence over packed pages.
``append``      ``append_kv``: quantize, pack and scatter new K and V into pool pages.
``prefill``     ``winnow_packed_attention`` with Q > 1 query tokens over packed pages.
``dequant``     ``tq_dequant``: a packed history back to bf16.
``contiguous``  ``TQPackedLayer``: reset, a prompt, one decoded token; both histories returned.

Inputs are K and V ~ N(0, 1) with one channel in a hundred scaled by ten (the outlier
channels that the random rotation is there for), quantized here in plain torch with the
package's own constants (rotation, codebook), so that the pages a decode reads do not
depend on the package's append. Page tables are shuffled unless a case says otherwise.
"""
import math
import random

import torch

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ESIZE = {"bf16": 2, "fp16": 2, "fp32": 4}


# ------------------------------------------------------------------------------ cases

def _decode(name, B, Hq, Hkv, Lmin, Lmax, bwk, bwv, D=128, S=16, dtype="bf16", tf32=False, shuffled=True, lens_seed=3):
    return dict(name=name, kind="decode", B=B, Hq=Hq, Hkv=Hkv, D=D, Lmin=Lmin, Lmax=Lmax, lens_seed=lens_seed, S=S,
                bwk=bwk, bwv=bwv, dtype=dtype, tf32=tf32, shuffled=shuffled)


def listed():
    return [
        # a small serving batch in mid-conversation: latency and launches count, 8-bit
        # (the width that leaves a model's outputs unchanged), seven query heads per kv head
        dict(name="step_small", kind="step", B=3, Hq=28, Hkv=4, D=128, Lmin=5, Lmax=300, lens_seed=1, S=16, bwk=8, bwv=8,
             dtype="bf16", layers=4),
        # the headline: a full batch at 32k context, 4-bit, pages in order
        _decode("decode_4bit_32k", 16, 32, 8, 32768, 32768, 4, 4, shuffled=False),
        # continuous batching: many sequences of very different lengths, pages scattered
        _decode("decode_ragged", 64, 32, 8, 512, 65536, 4, 4),
        # few very long contexts, K and V at different widths
        _decode("decode_long_k4v6", 4, 64, 8, 131072, 131072, 4, 6, shuffled=False),
        # a 32-sequence batch at 8 bits, lengths up to 4k, seven query heads per kv head
        _decode("decode_8bit", 32, 28, 4, 1000, 4096, 8, 8),
        # a model with 64-wide heads, medium contexts
        _decode("decode_hd64", 16, 32, 8, 3000, 12000, 4, 4, D=64, S=32),
        # one decode step's worth of new tokens (16 per sequence), 6-bit
        dict(name="append_step", kind="append", B=16, Hkv=8, n=16, D=128, S=16, bwk=6, bwv=6, dtype="bf16", start=4001),
        # a prompt of some thousand tokens stored at once
        dict(name="append_prompt", kind="append", B=1, Hkv=8, n=8191, D=128, S=16, bwk=4, bwv=4, dtype="bf16", start=0),
        # chunked prefill of two long prompts, 4-bit
        dict(name="prefill_chunk", kind="prefill", B=2, Hq=32, Hkv=8, Q=512, D=128, Lmin=32768, Lmax=32768, lens_seed=1, S=16,
             bwk=4, bwv=4, dtype="bf16"),
        # follow-up turns over an 8-bit cache
        dict(name="prefill_8bit", kind="prefill", B=4, Hq=28, Hkv=4, Q=64, D=128, Lmin=1000, Lmax=4096, lens_seed=5, S=16,
             bwk=8, bwv=8, dtype="bf16"),
        # a packed history of a million vectors handed to dense attention
        dict(name="dequant_1m", kind="dequant", B=16, H=8, L=8192, maxlen=8200, D=128, bw=4, fast=False),
        # the contiguous cache with outlier channels at a higher width: prompt, then a token
        dict(name="contiguous_outliers", kind="contiguous", B=2, H=8, n=2048, D=128, bw=4, n_out=8, out_bits=8, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# pairs of widths for K and V: what models are served at, most used first
WIDTHS = [(4, 4)] * 4 + [(8, 8)] * 3 + [(6, 6), (4, 6), (6, 4), (3, 3), (2, 2), (4, 8)]
HEADS = [(32, 8), (28, 4), (64, 8), (8, 8), (8, 2), (16, 2)]


def draw(rng):
    kind = rng.choice(["step", "decode", "decode", "decode", "append", "append", "prefill", "prefill", "dequant", "contiguous"])
    Hq, Hkv = rng.choice(HEADS)
    bwk, bwv = rng.choice(WIDTHS)
    D = rng.choice([128, 128, 128, 64])
    S = rng.choice([16, 16, 32, 64])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    seed = rng.randrange(1 << 30)
    if kind == "step":
        Lmin = _log(rng, 1, 500)
        return dict(kind=kind, B=_log(rng, 1, 16), Hq=Hq, Hkv=Hkv, D=D, Lmin=Lmin, Lmax=Lmin + _log(rng, 1, 1500), lens_seed=seed,
                    S=S, bwk=bwk, bwv=bwv, dtype=dtype, layers=rng.randint(1, 4))
    if kind == "decode":
        B = _log(rng, 1, 64)
        most = (1 << 21) // (B * Hkv)          # at most a quarter of the largest listed batch's (token, kv head) pairs
        Lmax = _log(rng, 40, min(131072, most))
        Lmin = rng.choice([Lmax, max(1, Lmax // rng.randint(2, 30))])
        return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, D=D, Lmin=Lmin, Lmax=Lmax, lens_seed=seed, S=S, bwk=bwk, bwv=bwv,
                    dtype=rng.choice([dtype, dtype, "fp32"]), tf32=rng.random() < 0.2, shuffled=rng.random() < 0.7)
    if kind == "append":
        B = rng.choice([1, 1, 2, 4, 8, 16, 32])
        return dict(kind=kind, B=B, Hkv=Hkv, n=_log(rng, 1, 16384 // B), D=D, S=S, bwk=bwk, bwv=bwv, dtype=dtype,
                    start=rng.choice([0, _log(rng, 1, 5000)]))
    if kind == "prefill":
        B, Q = _log(rng, 1, 8), _log(rng, 2, 512)
        most = (1 << 19) // (B * Hkv)
        Lmax = _log(rng, Q, max(Q + 1, min(32768, most, (1 << 24) // (Q * B))))
        return dict(kind=kind, B=B, Hq=Hq, Hkv=Hkv, Q=Q, D=D, Lmin=rng.choice([Lmax, max(Q, Lmax // 3)]), Lmax=Lmax, lens_seed=seed,
                    S=S, bwk=bwk, bwv=bwv, dtype=dtype)
    if kind == "dequant":
        B, H = rng.choice([1, 2, 4, 8]), rng.choice([2, 4, 8])
        L = _log(rng, 100, 16384)
        return dict(kind=kind, B=B, H=H, L=L, maxlen=L + rng.choice([0, 1, 33]), D=128, bw=rng.choice([2, 3, 4, 4, 6, 8]),
                    fast=rng.random() < 0.5)
    n_out, out_bits = rng.choice([(0, 0), (8, 8), (16, 6)])
    return dict(kind=kind, B=rng.choice([1, 2, 3]), H=rng.choice([2, 4, 8]), n=_log(rng, 60, 2000), D=D, bw=rng.choice([2, 3, 4]),
                n_out=n_out, out_bits=out_bits, dtype=dtype)


def _lens(c):
    """The lengths of the batch's sequences (for prefill and step they count the new tokens)."""
    r = random.Random(c["lens_seed"])
    return [r.randint(c["Lmin"], c["Lmax"]) if c["Lmin"] < c["Lmax"] else c["Lmax"] for _ in range(c["B"])]


# ------------------------------------------------------------------------ plain torch

def _pack(codes, bw):
    """(..., D) codes -> (..., D bw / 8) bytes, LSB first: bw bytes per eight codes."""
    at = torch.arange(8, device=codes.device) * bw
    words = (codes.to(torch.int64).unflatten(-1, (-1, 8)) << at).sum(-1) if bw < 8 else None
    if words is None:
        return codes.to(torch.uint8)
    out = (words[..., None] >> (8 * torch.arange(bw, device=codes.device))) & 255
    return out.flatten(-2).to(torch.uint8)


def _unpack(packed, bw):
    if bw == 8:
        return packed.to(torch.int64)
    words = (packed.to(torch.int64).unflatten(-1, (-1, bw)) << (8 * torch.arange(bw, device=packed.device))).sum(-1)
    return ((words[..., None] >> (bw * torch.arange(8, device=packed.device))) & ((1 << bw) - 1)).flatten(-2)


def _quantize(x, tq, f=torch.float32):
    """Packed codes and fp16 norms of x's last axis."""
    x = x.to(f)
    n = x.norm(dim=-1, keepdim=True).clamp_min(1e-10)
    y = (x / n) @ tq.Pi.to(f).T
    return _pack(torch.bucketize(y, tq.boundaries.to(f)), tq.bit_width), n[..., 0].to(torch.float16)


def _dequantize(packed, norms, tq):
    return (tq.centroids.double()[_unpack(packed, tq.bit_width)] @ tq.Pi.double()) * norms.double()[..., None]


def _kv(g, shape, loud):
    x = torch.randn(shape, generator=g, device=DEV)
    return x * (1 + 9 * loud)


def _loud(g, heads, D):
    """(heads, 1, D): 1 on one channel in a hundred of each head, else 0."""
    pick = torch.rand(heads, D, generator=g, device=DEV).topk(max(1, round(0.01 * D)), dim=-1).indices
    return torch.zeros(heads, D, device=DEV).scatter_(1, pick, 1.0)[:, None]


def _quantizers(c):
    from winnow_amd.quantizer import get_quantizer
    return get_quantizer(c["bwk"], c["D"], DEV, seed=42), get_quantizer(c["bwv"], c["D"], DEV, seed=42)


def _table(need, order):
    table = torch.full((len(need), max(need)), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        table[b, :n] = order[at:at + n]
        at += n
    return table


def _store(pages, norms, ids, x, tq):
    """Quantize (Hkv, L, D) into the pages `ids` of (P, Hkv, S, NB)."""
    L, S = x.shape[1], pages.shape[2]
    codes, n = _quantize(x, tq)
    codes = torch.nn.functional.pad(codes, (0, 0, 0, ids.numel() * S - L))
    n = torch.nn.functional.pad(n, (0, ids.numel() * S - L))
    pages[ids] = codes.unflatten(1, (-1, S)).transpose(0, 1)
    norms[ids] = n.unflatten(1, (-1, S)).transpose(0, 1)


def _handle(c, g):
    """A PackedKV over a filled pool, with the host mirrors that the paged cache attaches."""
    from winnow_amd import packed_attention as pa
    lens, S, Hkv, D = _lens(c), c["S"], c["Hkv"], c["D"]
    need = [max(1, -(-L // S)) for L in lens]
    P = sum(need)
    order = torch.randperm(P, generator=torch.Generator().manual_seed(c["lens_seed"])) if c.get("shuffled", True) else torch.arange(P)
    table = _table(need, order.to(torch.int32))
    tqs = _quantizers(c)
    loud = [_loud(g, Hkv, D) for _ in tqs]
    pages = [torch.zeros(P, Hkv, S, D * tq.bit_width // 8, dtype=torch.uint8, device=DEV) for tq in tqs]
    norms = [torch.zeros(P, Hkv, S, dtype=torch.float16, device=DEV) for _ in tqs]
    for b, L in enumerate(lens):
        ids = table[b, :need[b]].long().to(DEV)
        for p, n, tq, ld in zip(pages, norms, tqs, loud):
            _store(p, n, ids, _kv(g, (Hkv, L, D), ld).bfloat16(), tq)
    seq = torch.tensor(lens, dtype=torch.int32)
    return pa.PackedKV(pages[0], norms[0], pages[1], norms[1], table.to(DEV), seq.to(DEV), pa.Quantizer.from_tq(tqs[0]),
                       pa.Quantizer.from_tq(tqs[1]), D, seq_lens_host=seq, page_table_host=table)


# --------------------------------------------------------------------- prepare and run

def prepare(c, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind, D = c["kind"], c["D"]
    dt = DTYPES[c.get("dtype", "bf16")]
    if kind in ("decode", "prefill"):
        s = dict(c=c, kv=_handle(c, g), scale=D ** -0.5)
        s["q"] = torch.randn(c["B"], c["Hq"], c.get("Q", 1), D, generator=g, device=DEV).to(dt)
        return s
    if kind == "step":
        from winnow_amd.page_pool import PagePool
        tqs, lens, S, Hkv = _quantizers(c), _lens(c), c["S"], c["Hkv"]
        need = [-(-L // S) for L in lens]
        pool = PagePool(num_layers=c["layers"], num_pages=sum(need) + 8, num_kv_heads=Hkv, page_size=S,
                        nb_k=D * c["bwk"] // 8, nb_v=D * c["bwv"] // 8, device=DEV)
        owners = ["r%d" % b for b in range(c["B"])]
        loud, news = _loud(g, Hkv, D), []
        for b, L in enumerate(lens):
            ids = torch.tensor([r.page for r in pool.ensure(owners[b], L)], device=DEV)
            for l in range(c["layers"]):
                for p, n, tq in ((pool.k_pages, pool.k_norms, tqs[0]), (pool.v_pages, pool.v_norms, tqs[1])):
                    if L > 1:
                        _store(p[l], n[l], ids, _kv(g, (Hkv, L, D), loud).bfloat16(), tq)
        for _ in range(c["layers"]):
            news.append(tuple(_kv(g, (c["B"], Hkv, 1, D), loud).to(dt) for _ in range(2))
                        + (torch.randn(c["B"], c["Hq"], 1, D, generator=g, device=DEV).to(dt),))
        return dict(c=c, pool=pool, owners=owners, before=[L - 1 for L in lens], tqs=tqs, news=news, scale=D ** -0.5)
    if kind == "append":
        B, Hkv, n, S = c["B"], c["Hkv"], c["n"], c["S"]
        tqs = _quantizers(c)
        loud = _loud(g, Hkv, D)
        need = [-(-(c["start"] + n) // S)] * B
        P = sum(need)
        table = _table(need, torch.randperm(P, generator=torch.Generator().manual_seed(seed)).to(torch.int32))
        start = torch.full((B,), c["start"], dtype=torch.int32)
        # K and V as the projections leave them: (B, n, heads, D) viewed as (B, heads, n, D)
        k, v = (_kv(g, (B, Hkv, n, D), loud).to(dt).transpose(1, 2).contiguous().transpose(1, 2) for _ in range(2))
        pages = [torch.zeros(P, Hkv, S, D * tq.bit_width // 8, dtype=torch.uint8, device=DEV) for tq in tqs]
        norms = [torch.zeros(P, Hkv, S, dtype=torch.float16, device=DEV) for _ in tqs]
        return dict(c=c, k=k, v=v, tqs=tqs, pages=pages, norms=norms, table=table.to(DEV), table_host=table,
                    start=start.to(DEV), start_host=start)
    if kind == "dequant":
        from winnow_amd.quantizer import get_quantizer
        tq = get_quantizer(c["bw"], D, DEV)
        codes = torch.zeros(c["B"], c["H"], c["maxlen"], D * c["bw"] // 8, dtype=torch.uint8, device=DEV)
        norms = torch.zeros(c["B"], c["H"], c["maxlen"], dtype=torch.float16, device=DEV)
        loud = _loud(g, c["H"], D)
        for b in range(c["B"]):
            codes[b], norms[b] = _quantize(_kv(g, (c["H"], c["maxlen"], D), loud).bfloat16(), tq)
        return dict(c=c, codes=codes, norms=norms, tq=tq)
    from winnow_amd.cache import TQPackedLayer
    layer = TQPackedLayer(D, c["bw"], DEV, c["n"] + 8, num_outlier_channels=c["n_out"], outlier_bits=c["out_bits"])
    # the outlier channels: as many loud ones as the cache keeps apart, the same in every head
    loud = torch.zeros(D, device=DEV)
    loud[torch.rand(D, generator=g, device=DEV).topk(max(1, c["n_out"])).indices] = 1.0
    x = [_kv(g, (c["B"], c["H"], n, D), loud).to(dt) for n in (c["n"], c["n"], 1, 1)]
    return dict(c=c, layer=layer, x=x)


def run(s):
    c = s["c"]
    kind = c["kind"]
    if kind == "decode":
        from winnow_amd.packed_attention import packed_decode_attention
        return packed_decode_attention(s["q"], s["kv"], s["scale"], allow_tf32=c["tf32"])
    if kind == "prefill":
        from winnow_amd.packed_backend import winnow_packed_attention
        return winnow_packed_attention(None, s["q"], s["kv"], s["kv"], None, scaling=s["scale"])[0]
    if kind == "step":
        from winnow_amd.packed_backend import PagedPackedCache, winnow_packed_attention
        pool = s["pool"]
        cache = PagedPackedCache(pool, s["owners"], s["before"], k_quant=s["tqs"][0], v_quant=s["tqs"][1], head_dim=c["D"])
        outs = []
        for layer, (k, v, q) in enumerate(s["news"]):
            kk, vv = cache.update(k, v, layer)
            outs.append(winnow_packed_attention(None, q, kk, vv, None, scaling=s["scale"])[0])
        return outs, pool.k_pages, pool.v_pages, pool.k_norms, pool.v_norms
    if kind == "append":
        from winnow_amd.packed_backend import append_kv
        append_kv(s["k"], s["v"], s["tqs"][0], s["tqs"][1], s["pages"][0], s["pages"][1], s["norms"][0], s["norms"][1],
                  s["table"], s["start"], page_table_host=s["table_host"], start_pos_host=s["start_host"])
        return s["pages"], s["norms"]
    if kind == "dequant":
        from winnow_amd.kernel import tq_dequant
        L = c["L"]
        return tq_dequant(s["codes"][:, :, :L], s["norms"][:, :, :L], s["tq"].centroids, s["tq"].Pi, c["bw"], c["D"],
                          allow_tf32=c["fast"])
    s["layer"].reset()
    s["layer"].update(s["x"][0], s["x"][1])
    return s["layer"].update(s["x"][2], s["x"][3])


# ------------------------------------------------------------------- work and precision

def work(c):
    kind, D = c["kind"], c["D"]
    es = ESIZE[c.get("dtype", "bf16")]
    if kind in ("decode", "prefill", "step"):
        lens, Q = _lens(c), c.get("Q", 1)
        row = D * (c["bwk"] + c["bwv"]) / 8 + 4
        pairs = sum(Q * L - Q * (Q - 1) // 2 for L in lens)
        layers = c.get("layers", 1)
        new = 0 if kind != "step" else c["B"] * c["Hkv"] * (2 * D * es + row)
        return {"bytes": layers * (sum(lens) * c["Hkv"] * row + 2 * c["B"] * c["Hq"] * Q * D * es + new),
                "flops": layers * 4.0 * c["Hq"] * D * pairs}
    if kind == "append":
        vectors = c["B"] * c["Hkv"] * c["n"]
        return {"bytes": vectors * (2 * D * es + D * (c["bwk"] + c["bwv"]) / 8 + 4), "flops": 2 * 2.0 * D * D * vectors}
    if kind == "dequant":
        vectors = c["B"] * c["H"] * c["L"]
        return {"bytes": vectors * (D * c["bw"] / 8 + 2 + 2 * D), "flops": 2.0 * D * D * vectors}
    vectors, n_out = 2 * c["B"] * c["H"] * c["n"], c["n_out"]
    packed = ((D - n_out) * c["bw"] + n_out * c["out_bits"]) / 8 + 4
    # the prompt in, its codes out, and two histories read and handed back
    return {"bytes": vectors * (D * es + 3 * packed + 2 * D * es),
            "flops": 3 * 2.0 * ((D - n_out) ** 2 + n_out ** 2) * vectors}


def tolerance(c):
    kind = c["kind"]
    if kind == "append":
        return "exact"           # codes and fp16 norms are the quantizer's, bit for bit
    if c.get("tf32"):
        return {"rel": 4e-3, "max": 4e-2}       # products of 11-bit operands
    if kind == "decode" and c["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 2e-4}
    # 16-bit results: half a unit in the last place of bf16 is 2e-3 of a value
    if kind == "prefill":
        return {"rel": 1e-2, "max": 1e-1}       # 16-bit operands as well
    return {"rel": 4e-3, "max": 4e-2}


def _attend(q, k, v, scale):
    """Offset-causal attention of q (r, Q, D) over one kv head's k and v (L, D), in 64 bits."""
    Q, L = q.shape[1], k.shape[0]
    s = scale * (q.reshape(-1, q.shape[-1]) @ k.T).unflatten(0, (-1, Q))
    if Q > 1:
        at = torch.arange(L, device=s.device)
        s.masked_fill_(at[None, :] > (L - Q + torch.arange(Q, device=s.device))[:, None], -math.inf)
    return (torch.softmax(s, -1).flatten(0, 1) @ v).unflatten(0, (-1, Q))


def exact(c, seed):
    kind, D = c["kind"], c["D"]
    s = prepare(c, seed)
    if kind in ("decode", "prefill"):
        kv, tqs = s["kv"], _quantizers(c)
        rep = c["Hq"] // c["Hkv"]
        out = torch.zeros(s["q"].shape, dtype=torch.float64, device=DEV)
        for b, L in enumerate(_lens(c)):
            ids = kv.page_table[b, :-(-L // c["S"])].long()
            for h in range(c["Hkv"]):
                k, v = (_dequantize(p[ids, h].flatten(0, 1)[:L], n[ids, h].flatten()[:L], tq)
                        for p, n, tq in ((kv.k_pages, kv.k_norms, tqs[0]), (kv.v_pages, kv.v_norms, tqs[1])))
                out[b, h * rep:(h + 1) * rep] = _attend(s["q"][b, h * rep:(h + 1) * rep].double(), k, v, s["scale"])
        return out if kind == "decode" else out.transpose(1, 2).contiguous()
    if kind == "step":
        pool, rep, outs = s["pool"], c["Hq"] // c["Hkv"], []
        for l, (k, v, q) in enumerate(s["news"]):
            out = torch.zeros(c["B"], 1, c["Hq"], D, dtype=torch.float64, device=DEV)
            new = [_quantize(x, tq, torch.float64) for x, tq in zip((k, v), s["tqs"])]
            for b, L in enumerate(_lens(c)):
                ids = torch.tensor([r.page for r in pool.held(s["owners"][b])], device=DEV)
                for h in range(c["Hkv"]):
                    sides = []
                    for p, n, tq, (codes, norm) in ((pool.k_pages, pool.k_norms, s["tqs"][0], new[0]),
                                                    (pool.v_pages, pool.v_norms, s["tqs"][1], new[1])):
                        rows = torch.cat([p[l][ids, h].flatten(0, 1)[:L - 1], codes[b, h]])
                        sides.append(_dequantize(rows, torch.cat([n[l][ids, h].flatten()[:L - 1], norm[b, h]]), tq))
                    out[b, 0, h * rep:(h + 1) * rep] = _attend(q[b, h * rep:(h + 1) * rep].double(), *sides, s["scale"])[:, 0]
            outs.append(out)
        return outs, None, None, None, None
    if kind == "append":
        norms = []
        for x in (s["k"], s["v"]):
            full = torch.zeros(s["norms"][0].shape, dtype=torch.float64, device=DEV)
            pos = c["start"] + torch.arange(c["n"], device=DEV)
            for b in range(c["B"]):
                full[s["table"][b].long()[pos // c["S"]], :, pos % c["S"]] = x[b].double().norm(dim=-1).T
            norms.append(full)
        return [None, None], norms
    if kind == "dequant":
        L = c["L"]
        return torch.stack([_dequantize(s["codes"][b, :, :L], s["norms"][b, :, :L], s["tq"]) for b in range(c["B"])])
    from winnow_amd.quantizer import get_quantizer
    x = [torch.cat([s["x"][0], s["x"][2]], 2), torch.cat([s["x"][1], s["x"][3]], 2)]
    apart = torch.zeros(D, dtype=torch.bool, device=DEV)
    if c["n_out"]:
        apart[s["x"][0].double().pow(2).mean(dim=(0, 1, 2)).topk(c["n_out"]).indices] = True
    outs = []
    for y in x:
        out = torch.zeros(y.shape, dtype=torch.float64, device=DEV)
        for mask, bw, qseed in ((~apart, c["bw"], 42), (apart, c["out_bits"], 43)):
            if int(mask.sum()):
                tq = get_quantizer(bw, int(mask.sum()), DEV, seed=qseed)
                out[..., mask] = _dequantize(*_quantize(y[..., mask], tq, torch.float64), tq)
        outs.append(out)
    return outs[0], outs[1]
