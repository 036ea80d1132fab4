"""The decode row scan on the 16-bit matrix cores at the widths and sizes where a chunk,
a page or a split ends, against the same attention in float64.

The scan multiplies fp16 pairs (H + L carries a value to 2^-22 of itself) and accumulates
in fp32, so a score is off by at most 2^-19 sum|q k| (both factors, 128 products' sums), a weight by twice that relative to itself with the exponential's own
error, and an output by that share of the largest value; the values' own split and the
rotation back add 2^-17 of the largest value. The bound below is that, from the case's data.
"""
from __future__ import annotations

import pytest
import torch

from cases import build, to_device
from oracle import attention as oa

pytestmark = pytest.mark.gpu


def _float64(q, kv, scale):
    """(attention in float64 over the rotated codes, the bound above)."""
    B, Hq, _, D = q.shape
    rep = Hq // kv.num_kv_heads
    out = torch.zeros(B, Hq, 1, D, dtype=torch.float64)
    qr = q.double() @ kv.k_quant.Pi.double().T
    smax = vmax = 0.0
    for b in range(B):
        if int(kv.seq_lens[b]) == 0:
            continue
        kc, kn = oa._gather_history(kv.k_pages, kv.k_norms, kv, b)
        vc, vn = oa._gather_history(kv.v_pages, kv.v_norms, kv, b)
        k = oa._centroids(kc, kv.k_quant, D).double() * kn.double()[..., None]
        v = oa._centroids(vc, kv.v_quant, D).double() * vn.double()[..., None]
        k, v = (x.repeat_interleave(rep, 0) for x in (k, v))
        p = torch.softmax((k @ qr[b].transpose(-1, -2)).squeeze(-1) * scale, -1)
        out[b, :, 0] = (p[:, None] @ v).squeeze(1) @ kv.v_quant.Pi.double()
        smax = max(smax, float((k.abs() @ qr[b].abs().transpose(-1, -2)).max()) * scale)
        vmax = max(vmax, float(v.norm(dim=-1).max()))
    return out, (2 * 2.0 ** -19 * smax + 2.0 ** -17) * vmax


@pytest.mark.parametrize("D,S,Hq,Hkv,bwk,bwv", [(128, 16, 28, 4, 8, 8), (128, 64, 8, 8, 8, 8), (128, 32, 64, 8, 8, 8),
                                                (128, 16, 12, 2, 4, 8), (128, 128, 4, 2, 4, 8), (128, 16, 28, 4, 4, 4),
                                                # head_dim 64: two tokens to a row, up to four heads of a kv head
                                                (64, 16, 8, 2, 4, 4), (64, 32, 12, 4, 4, 4), (64, 128, 3, 3, 8, 8),
                                                (64, 16, 4, 2, 5, 5), (64, 64, 8, 2, 6, 4), (64, 16, 6, 2, 3, 3)])
def test_scan_edges(D, S, Hq, Hkv, bwk, bwv):
    lens = (0, 1, 2, 63, 64, 65, 127, 128, 129, 130, 257, 2049)
    q, kv = build(700 + S + bwk + D, len(lens), Hq, Hkv, D, lens, S, bwk, bw_v=bwv)
    scale = oa.default_scale(D)
    ref, tol = _float64(q, kv, scale)
    from winnow_amd import packed_attention as pa
    for splits in (None, 1, 7):
        print(f"S={S} {Hq}/{Hkv} heads {bwk}/{bwv} bits D={D} splits={splits}", flush=True)
        got = pa.packed_decode_attention(q.cuda(), to_device(kv, "cuda"), scale, num_splits=splits,
                                         out_dtype=torch.float32).cpu().double()
        assert torch.isfinite(got).all()
        err = float((got - ref).abs().max())
        assert err <= tol, (err, tol)
        assert (got[0] == 0).all()


def test_norms_off_the_word(Hq=8, Hkv=2, D=64, S=16):
    """head_dim 64 reads the norms of two tokens in one word: norms that begin on an odd
    element, and plans asked for by number, give the same attention."""
    from winnow_amd import packed_attention as pa
    lens = (5, 300, 64)
    q, kv = build(41, len(lens), Hq, Hkv, D, lens, S, 4)
    scale = oa.default_scale(D)
    ref, tol = _float64(q, kv, scale)
    dev = to_device(kv, "cuda")
    for name in ("k_norms", "v_norms"):
        n = getattr(dev, name)
        room = torch.zeros(n.numel() + 1, dtype=n.dtype, device=n.device)
        room[1:] = n.flatten()
        setattr(dev, name, room[1:].view(n.shape))
    for splits in (None, 3):
        got = pa.packed_decode_attention(q.cuda(), dev, scale, num_splits=splits, out_dtype=torch.float32).cpu().double()
        assert float((got - ref).abs().max()) <= tol


def _room(dev, tokens=3 << 18):
    """The handle with a page table that has room for ``tokens`` (token, query head) pairs at
    three heads and more: the size from which head_dim 64 runs two tokens to a row."""
    B, width = dev.page_table.shape
    pad = torch.full((B, -(-tokens // (3 * B * dev.page_size)) + 1 - width), -1, dtype=torch.int32)
    dev.page_table_host = torch.cat([dev.page_table_host, pad], 1)
    dev.page_table = dev.page_table_host.cuda()
    return dev


@pytest.mark.parametrize("S,Hq,Hkv,bwk,bwv", [(16, 8, 2, 4, 4), (32, 12, 4, 4, 4), (128, 3, 3, 8, 8), (16, 4, 2, 5, 5), (64, 8, 2, 6, 4),
                                              (16, 6, 2, 3, 3), (16, 8, 4, 2, 2), (32, 8, 2, 6, 6), (16, 4, 1, 4, 6), (64, 6, 2, 4, 8),
                                              (16, 8, 2, 8, 8)])
@pytest.mark.parametrize("apart", [False, True])
def test_two_tokens_to_a_row(S, Hq, Hkv, bwk, bwv, apart):
    """head_dim 64 in a table large enough for the row scan, at the lengths where a row, a
    chunk, a page or a split ends, and with a head's pages and norms apart from the next
    one's (strides larger than a block)."""
    from winnow_amd import packed_attention as pa
    D = 64
    lens = (0, 1, 2, 3, 63, 64, 65, 127, 128, 129, 130, 255, 257, 2049)
    q, kv = build(900 + S + bwk + bwv, len(lens), Hq, Hkv, D, lens, S, bwk, bw_v=bwv)
    scale = oa.default_scale(D)
    ref, tol = _float64(q, kv, scale)
    dev = _room(to_device(kv, "cuda"))
    if apart:
        for name in ("k_pages", "v_pages", "k_norms", "v_norms"):
            x = getattr(dev, name)
            wide = torch.full((x.shape[0], 2 * Hkv, *x.shape[2:]), 0x55, dtype=torch.uint8, device="cuda").to(x.dtype)
            wide[:, 1::2] = x
            setattr(dev, name, wide[:, 1::2])
    plan = pa.plan_for(q.cuda(), dev)
    assert plan[1] <= 256 and plan[0] * dev.page_size >= 128
    for splits in (None, 1, 7, 2000):
        got = pa.packed_decode_attention(q.cuda(), dev, scale, num_splits=splits, out_dtype=torch.float32).cpu().double()
        assert torch.isfinite(got).all()
        err = float((got - ref).abs().max())
        assert err <= tol, (err, tol)
        assert (got[0] == 0).all()


@pytest.mark.parametrize("D,S,Hq,Hkv,bwk,bwv,tf32", [(128, 16, 28, 4, 8, 8, False), (128, 16, 8, 8, 4, 8, False),
                                                     (128, 32, 16, 4, 4, 4, False), (128, 16, 16, 2, 6, 6, False),
                                                     (128, 16, 8, 8, 4, 6, True), (64, 16, 8, 2, 4, 4, False),
                                                     (64, 32, 12, 4, 8, 8, False), (64, 16, 3, 3, 2, 2, False)])
def test_value_norms_of_any_size(D, S, Hq, Hkv, bwk, bwv, tf32):
    """V norms times a power of two (exact in fp16 here) give the same attention times that
    power, bit for bit: the scan scales its 16-bit weights by the norms' own exponent,
    so small norms lose nothing. Norms of a head_dim of 64 or 128 lie within 4 and 20."""
    from winnow_amd import packed_attention as pa
    lens = (1, 70, 300, 1500)
    q, kv = build(800 + S + bwv + D, len(lens), Hq, Hkv, D, lens, S, bwk, bw_v=bwv)
    scale = oa.default_scale(D)
    dev = to_device(kv, "cuda")
    if D == 64:
        _room(dev)
    norms, outs = dev.v_norms.clone(), {}
    for e in (0, -15, 11):
        dev.v_norms.copy_((norms.float() * 2.0 ** e).half())
        assert torch.equal(dev.v_norms.float(), norms.float() * 2.0 ** e)
        outs[e] = pa.packed_decode_attention(q.cuda(), dev, scale, out_dtype=torch.float32, allow_tf32=tf32) * 2.0 ** -e
    assert float(outs[0].abs().max()) > 0
    for e in (-15, 11):
        assert torch.equal(outs[e], outs[0])
    # the scale is the magnitude's: negative norms give the attention negated, up to the sums'
    # rounding, which is not the same for both signs (some thousand sums of 2^-24 each)
    dev.v_norms.copy_(-norms)
    out = pa.packed_decode_attention(q.cuda(), dev, scale, out_dtype=torch.float32, allow_tf32=tf32)
    assert float((out + outs[0]).abs().max()) <= 2.0 ** -16 * float(outs[0].abs().max())
    dev.v_norms.zero_()
    out = pa.packed_decode_attention(q.cuda(), dev, scale, out_dtype=torch.float32, allow_tf32=tf32)
    assert (out == 0).all()
