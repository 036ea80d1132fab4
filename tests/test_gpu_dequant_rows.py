"""GPU parity of the fp32-accurate rows kernels of the contiguous cache: the outlier-channel
append (``wn_append_split``) against ``wn_quantize`` + ``wn_pack`` per channel group, bit
for bit, and the dequantization (``wn_dequantize_rows``, ``wn_dequantize_pages``,
``wn_dequantize``) against float64 closed forms. A float32 sum of D products of values
below 1 has an error below D 2^-24 of the row's norm; 2e-6 of the largest value is
asked at D <= 256 (measured: 3e-7).
"""
from __future__ import annotations

import pytest
import torch

from cases import build, to_device

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _layer(D, bw, n_out, out_bits, cap, **kw):
    from winnow_amd.cache import TQPackedLayer
    return TQPackedLayer(D, bw, DEV, cap, num_outlier_channels=n_out, outlier_bits=out_bits, **kw)


def _kv(B, H, n, D, loud, dtype, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(2, B, H, n, D, generator=g, device=DEV)
    x[..., loud] *= 12
    x[0, 0, 0, 0] = 0                        # a zero vector
    x[1, 0, 0, min(1, n - 1)] *= 1e-6
    return x[0].to(dtype), x[1].to(dtype)


# group widths that fill eights of codes and ones that do not (122 x 4 bits = 61 bytes),
# one outlier eight, several, most of the channels
SPLITS = [(128, 4, 8, 8), (128, 3, 16, 6), (128, 4, 6, 8), (128, 2, 32, 3), (64, 3, 8, 8), (64, 4, 14, 8), (64, 2, 40, 5)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("D,bw,n_out,out_bits", SPLITS)
def test_split_append_equals_the_group_kernels(D, bw, n_out, out_bits, dtype):
    """A prompt whose vectors do not fill the last pass, then single tokens; K and V as a
    projection leaves them (heads next to tokens). The rows past the end stay untouched."""
    B, H, cap = 2, 3, 61
    loud = torch.randperm(D, generator=torch.Generator().manual_seed(D + n_out))[:n_out].to(DEV)
    layers = [_layer(D, bw, n_out, out_bits, cap) for _ in range(2)]
    pos = 0
    for step, n in enumerate((37, 1, 5)):
        k, v = _kv(B, H, n, D, loud, dtype, step)
        k, v = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (k, v))
        for i, layer in enumerate(layers):
            if not layer.is_initialized:
                layer.lazy_initialization(k, v)
                for grp in layer._k_groups + layer._v_groups:
                    grp.codes.fill_(0xA5)
                    grp.norms.fill_(-1)
            if i == 0:
                assert layer._split_append_ok(k, v)
                layer._append_split(k, v, pos)
            else:
                layer._append_groups(k, layer._k_groups, pos)
                layer._append_groups(v, layer._v_groups, pos)
        pos += n
    assert torch.equal(layers[0]._outlier_channels, layers[1]._outlier_channels)
    for a, b in zip(layers[0]._k_groups + layers[0]._v_groups, layers[1]._k_groups + layers[1]._v_groups):
        assert torch.equal(a.codes, b.codes) and torch.equal(a.norms, b.norms)


def test_split_append_of_vectors_a_fast_path_could_get_wrong():
    """Infinite, NaN and huge values in one group leave the other group's codes alone."""
    D, bw, n_out, out_bits = 128, 4, 8, 8
    loud = torch.arange(0, D, D // n_out, device=DEV)
    k, v = _kv(1, 2, 50, D, loud, torch.float32, 9)
    for x in (k, v):
        x[0, 0, 3, 1] = float("inf")
        x[0, 0, 4, int(loud[2])] = float("nan")
        x[0, 0, 5, int(loud[1])] = 3e38
        x[0, 1, 6, 7] = -3e38
        x[0, 1, 7] = 1e-35
    layers = [_layer(D, bw, n_out, out_bits, 50) for _ in range(2)]
    for layer in layers:
        layer.lazy_initialization(*(torch.nan_to_num(x, posinf=1.0).clamp(-50, 50) for x in (k, v)))
    layers[0]._append_split(k, v, 0)
    layers[1]._append_groups(k, layers[1]._k_groups, 0)
    layers[1]._append_groups(v, layers[1]._v_groups, 0)
    for a, b in zip(layers[0]._k_groups + layers[0]._v_groups, layers[1]._k_groups + layers[1]._v_groups):
        assert torch.equal(a.codes, b.codes) and torch.equal(a.norms.view(torch.int16), b.norms.view(torch.int16))


def _closed(codes, norms, tq):
    return (tq.centroids.double()[codes.long()] @ tq.Pi.double()) * norms.double()[..., None]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,bw,n_out,out_bits", SPLITS + [(128, 4, 0, 0), (64, 5, 0, 0), (256, 3, 0, 0), (256, 4, 16, 8),
                                                         (32, 8, 0, 0), (48, 2, 8, 4)])
def test_histories(D, bw, n_out, out_bits, dtype):
    """Read in place from a longer buffer, K and V in one launch, channels in their places."""
    from winnow_amd.packing import unpack
    B, H, n = 2, 3, 77
    loud = torch.randperm(D, generator=torch.Generator().manual_seed(D))[:max(n_out, 1)].to(DEV)
    layer = _layer(D, bw, n_out, out_bits, n + 6, kernel_backend="torch_fp32")
    k, v = _kv(B, H, n, D, loud, dtype, 5)
    for got, groups in zip(layer.update(k, v), (layer._k_groups, layer._v_groups)):
        want = torch.zeros(B, H, n, D, dtype=torch.float64, device=DEV)
        quants = [(layer._quant, bw, D - n_out)] + ([(layer._quant_outlier, out_bits, n_out)] if n_out else [])
        masks = [~layer._outlier_channels, layer._outlier_channels] if n_out else [torch.ones(D, dtype=torch.bool, device=DEV)]
        for grp, (tq, w, dim), mask in zip(groups, quants, masks):
            want[..., mask] = _closed(unpack(grp.codes[:, :, :n].contiguous(), w, dim), grp.norms[:, :, :n], tq)
        assert got.shape == want.shape and got.dtype == dtype
        step = 0.0 if dtype == torch.float32 else 2.0 ** -8   # half a unit of bf16's last place
        assert ((got.double() - want).abs() <= step * want.abs() + 2e-6 * want.abs().max()).all()
    assert layer.last_dispatch_decision.backend == "chunked"


@pytest.mark.parametrize("D,rows", [(16, 1), (64, 65), (100, 33), (120, 31), (128, 100000), (256, 40), (7, 9)])
def test_byte_codes(D, rows):
    """``dequantize_into`` at odd and even head dims (an infinite norm gives infinities of
    the sums' signs), into an output that four-element stores cannot address."""
    from winnow_amd.quantizer import TurboQuantMSE
    tq = TurboQuantMSE(4, D, DEV)
    g = torch.Generator(device=DEV).manual_seed(D)
    codes = torch.randint(0, 16, (rows, D), generator=g, device=DEV, dtype=torch.uint8)
    norms = torch.rand(rows, generator=g, device=DEV).half() * 20
    want = _closed(codes, norms, tq)
    out = torch.empty(rows * D + 1, device=DEV)[1:].view(rows, D)
    tq.dequantize_into(codes, norms, out)
    assert ((out.double() - want).abs() <= 2e-6 * want.abs().max()).all()
    again = torch.empty(rows, D, device=DEV)
    tq.dequantize_into(codes, norms, again)
    assert torch.equal(again, out)
    norms[0] = float("inf")
    tq.dequantize_into(codes, norms, again)
    sure = want[0].abs() > 1e-5 * want[0].abs().max()
    assert torch.equal(again[0][sure].double(), (want[0].sign() * float("inf"))[sure])


@pytest.mark.parametrize("D,bw", [(64, 4), (64, 3), (16, 8), (32, 5), (256, 6)])
def test_pages(D, bw):
    """Batched and single histories at the head dims without the fused dequant."""
    from winnow_amd import packed_backend as pb
    from winnow_amd.packing import unpack
    lens = (0, 1, 77, 160, 33)
    _, kv = build(500 + D + bw, len(lens), 4, 2, D, lens, 16, bw)
    dkv = to_device(kv, DEV)
    batch = pb._histories(dkv, dkv.v_pages, dkv.v_norms, dkv.v_quant, torch.tensor(lens), 163, torch.float32)
    for b, L in enumerate(lens):
        one = pb.dequantize_history(dkv, dkv.v_pages, dkv.v_norms, dkv.v_quant, b, torch.float32)[0]
        assert torch.equal(batch[b, :, :L], one)
        if L:
            rows = dkv.v_pages[dkv.page_table[b, :-(-L // 16)].long()].transpose(0, 1).reshape(2, -1, D * bw // 8)[:, :L]
            nrm = dkv.v_norms[dkv.page_table[b, :-(-L // 16)].long()].transpose(0, 1).reshape(2, -1)[:, :L]
            want = _closed(unpack(rows.contiguous(), bw, D), nrm, dkv.v_quant)
            assert ((one.double() - want).abs() <= 2e-6 * want.abs().max()).all()


@pytest.mark.parametrize("D,bw", [(64, 4), (32, 5)])
def test_pages_of_whole_sequences(D, bw):
    """Without lengths every sequence has Lpad rows, each through its own table row."""
    from winnow_amd import packed_backend as pb
    B, L = 3, 50
    _, kv = build(600 + D, B, 4, 2, D, (L,) * B, 16, bw)
    dkv = to_device(kv, DEV)
    side = (dkv.k_pages, dkv.k_norms, dkv.k_quant)
    got = torch.empty(B, 2, L, D, device=DEV)
    pb._dequantize_pages(dkv, *side, dkv.page_table, None, L, got)
    for b in range(B):
        assert torch.equal(got[b], pb.dequantize_history(dkv, *side, b, torch.float32)[0])


@pytest.mark.parametrize("D,n_out,span", [(320, 64, 1024), (288, 40, 10), (512, 256, 1024)])
def test_heads_wider_than_the_rows_kernel(D, n_out, span):
    """Outlier channels beside at most 256 regular ones: group by group, by chunks."""
    from winnow_amd.packing import unpack
    B, H, n = 2, 2, 37
    loud = torch.randperm(D, generator=torch.Generator().manual_seed(D))[:n_out].to(DEV)
    layer = _layer(D, 4, n_out, 8, n + 3, chunk=span)
    for step, m in enumerate((n - 1, 1)):
        got = layer.update(*_kv(B, H, m, D, loud, torch.float32, step))
    for x, groups in zip(got, (layer._k_groups, layer._v_groups)):
        want = torch.zeros(B, H, n, D, dtype=torch.float64, device=DEV)
        for grp, tq, w, dim, mask in ((groups[0], layer._quant, 4, D - n_out, ~layer._outlier_channels),
                                      (groups[1], layer._quant_outlier, 8, n_out, layer._outlier_channels)):
            want[..., mask] = _closed(unpack(grp.codes[:, :, :n].contiguous(), w, dim), grp.norms[:, :, :n], tq)
        assert ((x.double() - want).abs() <= 2e-6 * want.abs().max()).all()


def test_histories_past_the_row_limit_go_group_by_group(monkeypatch):
    """The rows kernel counts rows in 31 bits: with the limit lowered, the same values."""
    from winnow_amd import cache as wc
    D, n = 64, 50
    loud = torch.arange(8, device=DEV)
    k, v = _kv(2, 3, n, D, loud, torch.float32, 3)
    whole = _layer(D, 4, 8, 8, n).update(k, v)
    monkeypatch.setattr(wc, "_ROWS_LIMIT", 2 * 3 * n)
    for a, b in zip(_layer(D, 4, 8, 8, n, chunk=16).update(k, v), whole):
        assert torch.allclose(a, b, rtol=0, atol=2e-6 * b.abs().max().item())


def test_split_append_of_mixed_dtypes():
    """K and V of different types, and rows that 16-byte loads cannot read, take the
    per-group kernels: the same codes as the values alike."""
    D, n = 128, 21
    loud = torch.arange(0, D, 16, device=DEV)
    k, v = _kv(2, 3, n, D, loud, torch.bfloat16, 4)
    shifted = torch.empty(k.numel() + 1, dtype=k.dtype, device=DEV)[1:].view(k.shape)
    shifted.copy_(k)
    layers = []
    for kk, vv in ((k, v), (k, v.float()), (shifted, v)):
        layers.append(_layer(D, 4, 8, 8, n))
        layers[-1].update(kk, vv)
    for other in layers[1:]:
        assert not other._split_append_ok(k, v.float()) and not other._split_append_ok(shifted, v)
        for a, b in zip(layers[0]._k_groups + layers[0]._v_groups, other._k_groups + other._v_groups):
            assert torch.equal(a.codes, b.codes) and torch.equal(a.norms, b.norms)


@pytest.mark.parametrize("bw,off", [(4, 2), (8, 4), (4, 1), (6, 3)])
def test_sides_at_different_alignments(bw, off):
    """One side's codes a few bytes off the width that whole eights are read by: both sides
    byte by byte, the same values."""
    from winnow_amd import _lib
    from winnow_amd.quantizer import TurboQuantMSE
    D, rows = 64, 70
    tq = TurboQuantMSE(bw, D, DEV)
    nb = D * bw // 8
    g = torch.Generator(device=DEV).manual_seed(bw)
    sides = torch.randint(0, 256, (2, rows, nb), generator=g, device=DEV, dtype=torch.uint8)
    norms = torch.rand(2, rows, generator=g, device=DEV).half()
    room = torch.empty(rows * nb + off, dtype=torch.uint8, device=DEV)[off:].view(rows, nb)
    room.copy_(sides[1])

    def run(k, v):
        out = torch.empty(2, rows, D, device=DEV)
        _lib.call("wn_dequantize_rows", _lib.ptr(k), _lib.ptr(v), _lib.ptr(norms[0]), _lib.ptr(norms[1]), bw, _lib.ptr(tq.centroids),
                  None, None, None, None, 0, None, 0, _lib.ptr(tq.Pi), None, 1, rows, rows, D, _lib.ptr(out[0]), _lib.ptr(out[1]),
                  _lib.WN_F32, _lib.stream_of(out.device))
        return out
    want = run(sides[0], sides[1])
    assert torch.equal(run(sides[0], room), want)
    norms = norms.flip(0).contiguous()
    assert torch.equal(run(room, sides[0]), want.flip(0))
