"""The many-vector quantize kernel (``csrc/quant_tile.hip``) against the general one.

Both promise the same codes and norms, bit for bit. Rows that 16-byte loads cannot read
(a tensor one element into its storage) always take the general kernel, so the same
values at an aligned and at a shifted address go through both. Sizes sit at the rule's
lines and at the edges of a wave's sixteen vectors; inputs hold what a fast path could
get wrong: zero, one-hot, tiny, huge, infinite and NaN vectors, and values on bucket
boundaries.
"""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _shifted(x):
    """The same values and strides, one element further into a new storage."""
    flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)
    y = flat[1:].view(x.shape)
    y.copy_(x)
    assert x.data_ptr() % 16 == 0 and y.data_ptr() % 16 != 0
    return y


def _vectors(rows, D, dtype, tq, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(rows, D, generator=g, device=DEV)
    x *= torch.exp2(torch.randint(-20, 10, (rows, 1), generator=g, device=DEV).float())
    x[:, 3] *= 30
    # rows of Pi scaled so that one rotated coordinate sits on a boundary
    b = tq.boundaries
    for i in range(32):
        x[100 + i] = tq.Pi[i % D] * b[i % b.numel()] + tq.Pi[(i + 1) % D] * (1 - b[i % b.numel()] ** 2) ** 0.5
    x[0] = 0
    x[1] = 0
    x[1, 5] = 3.0
    x[2] *= 1e-30
    x[3, 7] = float("inf")
    x[4, 9] = float("nan")
    x[5] = float("-inf")
    x = x.to(dtype)
    x[6] = 0
    x[6, 1] = torch.finfo(dtype).max
    x[7] = torch.finfo(dtype).max / 16
    x[8] = torch.finfo(dtype).tiny
    x[-1] = x[1]
    return x


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("D,bw,rows", [(128, 4, 12288), (128, 2, 16383), (128, 3, 16385), (128, 5, 20001), (128, 6, 12289),
                                       (128, 8, 16384), (64, 4, 16384), (64, 8, 16399), (64, 3, 70001)])
def test_codes_and_norms_equal_the_general_kernel(D, bw, rows, dtype):
    from winnow_amd.quantizer import get_quantizer
    tq = get_quantizer(bw, D, DEV, 42)
    x = _vectors(rows, D, dtype, tq, rows + bw)
    codes, norms = tq.quantize(x)
    want, wnorms = tq.quantize(_shifted(x))
    assert torch.equal(codes, want)
    assert torch.equal(norms, wnorms)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,n,D,S,bwk,bwv", [(3, 2, 1025, 128, 16, 4, 6), (1, 8, 2047, 64, 32, 3, 2), (17, 4, 121, 128, 64, 8, 5)])
def test_append_equals_the_general_kernel(B, H, n, D, S, bwk, bwv, dtype):
    """Scattered over shuffled pages from a start inside a page, K and V as a projection
    leaves them (heads next to tokens), some positions beyond the table and some pages
    outside the pool: those are skipped."""
    from winnow_amd.packed_backend import append_kv
    from winnow_amd.quantizer import get_quantizer
    kq, vq = get_quantizer(bwk, D, DEV, 42), get_quantizer(bwv, D, DEV, 43)
    rows = B * H * n
    # (B, n, H, D) viewed as (B, H, n, D)
    k = _vectors(rows, D, dtype, kq, 1).view(B, n, H, D)
    v = _vectors(rows, D, dtype, vq, 2).view(B, n, H, D)
    width = -(-(n + 5) // S)
    g = torch.Generator().manual_seed(B)
    P = B * width
    table = torch.randperm(P, generator=g).to(torch.int32).view(B, width)
    table[0, 1] = -1
    table[B - 1, 0] = P + 3
    start = torch.full((B,), 5, dtype=torch.int32)
    start[B // 2] = width * S - 7
    got = []
    for shift in (lambda t: t, _shifted):
        pages = [torch.full((P, H, S, D * bw // 8), 0xA5, dtype=torch.uint8, device=DEV) for bw in (bwk, bwv)]
        norms = [torch.full((P, H, S), -1.0, dtype=torch.float16, device=DEV) for _ in range(2)]
        append_kv(shift(k).transpose(1, 2), shift(v).transpose(1, 2), kq, vq, *pages, *norms, table.to(DEV), start.to(DEV),
                  check_ranges=False)
        got.append(pages + norms)
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_a_rotation_outside_the_operands_range():
    """Rows of Pi of norm 1000: the fp16 operands cannot hold them, every code is the
    float64 path's."""
    from winnow_amd.quantizer import TurboQuantMSE
    tq = TurboQuantMSE(4, 128, DEV)
    tq.Pi = (tq.Pi * 1000).contiguous()
    x = torch.randn(12288, 128, device=DEV, generator=torch.Generator(device=DEV).manual_seed(3)) * 1e-3
    codes, norms = tq.quantize(x)
    want, wnorms = tq.quantize(_shifted(x))
    assert torch.equal(codes, want) and torch.equal(norms, wnorms)
