"""GPU parity of the reconstruct route's HIP operators: the batched history dequantization
(``wn_dequantize_histories``) against the single-sequence one, and the attention over
16-bit histories (``wn_history_attention``) against float64 attention over the same
16-bit K and V.

The attention's operands are exact, its scores and softmax fp32 and its probabilities pairs
of 16-bit values, so its own error is far below the rounding of its 16-bit output. A
value in [2^e, 2^(e+1)) has a unit in the last place of 2^(e-7) in bf16 (8 significant bits)
and 2^(e-10) in fp16 (11), so half a unit is at most 2^-8 and 2^-11 of the value; a hundredth
of that of the largest value is allowed for the operator's own error beside it.
"""
from __future__ import annotations

import pytest
import torch

from cases import build, to_device

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _f64(q, k, v, lens, scale):
    """Offset-causal float64 attention on the CPU of q (B, Hq, Q, D) over the first lens[b] rows."""
    B, Hq, Q, D = q.shape
    out = torch.zeros(B, Hq, Q, D, dtype=torch.float64)
    rep = Hq // k.shape[1]
    for b, L in enumerate(lens):
        for h in range(Hq):
            kk, vv = k[b, h // rep, :L].double(), v[b, h // rep, :L].double()
            for i in range(Q):
                seen = L - Q + i + 1
                if seen > 0:
                    p = torch.softmax(scale * (kk[:seen] @ q[b, h, i].double()), 0)
                    out[b, h, i] = p @ vv[:seen]
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D,Hq,Hkv,Q", [(128, 28, 4, 9), (128, 8, 8, 1), (128, 8, 2, 70), (128, 12, 1, 33), (64, 8, 2, 16),
                                        (64, 4, 4, 300)])
def test_attention_over_16_bit_histories(D, Hq, Hkv, Q, dtype):
    """Row counts of one partial block up to several work-groups; lengths of none, below Q,
    Q, at and beside a chunk, several chunks (several splits); scores large enough that
    the maximum moves; the buffer past each length holds NaN."""
    from winnow_amd import packed_attention as pa
    from winnow_amd import packed_backend as pb
    lens = [0, max(1, Q - 1), Q, 64, 65, 577]
    B, Lmax = len(lens), max(max(lens), Q) + 3
    g = torch.Generator().manual_seed(D + Hq + Q)
    q = (torch.randn(B, Q, Hq, D, generator=g) * 4).to(dtype).transpose(1, 2)
    k, v = (torch.randn(B, Hkv, Lmax, D, generator=g).to(dtype) for _ in range(2))
    lens = [min(L, Lmax) for L in lens]
    for b, L in enumerate(lens):
        k[b, :, L:] = float("nan")
        v[b, :, L:] = float("nan")
    empty = torch.empty(0, Hkv, 16, D, dtype=torch.uint8, device=DEV)
    kv = pa.PackedKV(empty, None, empty, None, None, torch.tensor(lens, dtype=torch.int32, device=DEV), None, None, D)
    scale = D ** -0.5
    ref = _f64(q, k, v, lens, scale)
    got = pb._history_attention(q.to(DEV), kv, k.to(DEV), v.to(DEV), Lmax, scale)
    assert got.shape == (B, Hq, Q, D) and got.dtype == dtype
    got = got.cpu().double()
    half = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert torch.isfinite(got).all()
    worst = ((got - ref).abs() / (half * (ref.abs() + 0.01 * ref.abs().max()))).max().item()
    assert worst <= 1, f"{worst:.2f} of the bound"
    for b, L in enumerate(lens):
        assert (got[b, :, :max(0, min(Q, Q - L))] == 0).all()
    # the queries' tokens next to each other per head, and rows that 16-byte loads cannot read
    shifted = torch.empty(q.numel() + 1, dtype=dtype, device=DEV)[1:].view(q.shape)
    shifted.copy_(q)
    assert torch.equal(pb._history_attention(shifted, kv, k.to(DEV), v.to(DEV), Lmax, scale).cpu().double(), got)


@pytest.mark.parametrize("bw", [2, 3, 4, 5, 6, 8])
def test_batched_histories_equal_single_ones(bw):
    from winnow_amd import packed_backend as pb
    lens = (0, 1, 77, 160, 33)
    _, kv = build(300 + bw, len(lens), 8, 2, 128, lens, 16, bw)
    dkv = to_device(kv, DEV)
    for dtype in (torch.bfloat16, torch.float32):
        all_ = pb._histories(dkv, dkv.k_pages, dkv.k_norms, dkv.k_quant, torch.tensor(lens), 163, dtype)
        for b, L in enumerate(lens):
            one = pb.dequantize_history(dkv, dkv.k_pages, dkv.k_norms, dkv.k_quant, b, dtype)[0]
            assert torch.equal(all_[b, :, :L], one)


@pytest.mark.parametrize("D,bw", [(128, 8), (64, 4)])
def test_reconstruct_route_with_and_without_the_operator(D, bw):
    """The route's 16-bit steps agree with the library's operator to 16-bit rounding; a
    query whose gradient is wanted keeps the library's."""
    from winnow_amd import packed_backend as pb
    lens, Q = (100, 3, 250), 5
    _, kv = build(400 + D, len(lens), 8, 2, D, lens, 16, bw)
    dkv = to_device(kv, DEV)
    q = torch.randn(3, 8, Q, D, generator=torch.Generator().manual_seed(1)).to(DEV, torch.bfloat16)
    got = pb._reconstruct_sdpa(q, dkv, 0.1)
    wanted = q.clone().requires_grad_()
    want = pb._reconstruct_sdpa(wanted, dkv, 0.1)
    assert torch.allclose(got.float(), want.float(), atol=2e-2 * want.abs().max().item(), rtol=2e-2)
    want.float().sum().backward()
    assert torch.isfinite(wanted.grad).all()


def test_a_trace_is_refused():
    """The histories come through the C ABI, which no trace records: a traced step raises
    where the library's operator is reached, it does not leave a graph without the attention."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from winnow_amd import packed_backend as pb
    lens = (100, 3, 250)
    _, kv = build(500, len(lens), 8, 2, 64, lens, 16, 4)
    dkv = to_device(kv, DEV)
    q = torch.randn(3, 8, 5, 64, generator=torch.Generator().manual_seed(2)).to(DEV, torch.bfloat16)

    def step(x):
        return pb._reconstruct_sdpa(x, dkv, 0.1)
    with pytest.raises((TypeError, RuntimeError)):
        torch.jit.trace(step, q, check_trace=False)
    with pytest.raises((TypeError, RuntimeError)):
        make_fx(step)(q)


def test_transforms_and_autocast_keep_the_library_operator():
    """vmap over queries, forward-mode tangents, and autocast to the other 16-bit type."""
    import torch.autograd.forward_ad as fwd
    from winnow_amd import packed_backend as pb
    lens, Q = (100, 3, 250), 5
    _, kv = build(501, len(lens), 8, 2, 64, lens, 16, 4)
    dkv = to_device(kv, DEV)
    g = torch.Generator().manual_seed(3)
    many = torch.randn(2, 3, 8, Q, 64, generator=g).to(DEV, torch.bfloat16)
    want = torch.stack([pb._reconstruct_sdpa(x, dkv, 0.1) for x in many]).float()
    got = torch.vmap(lambda x: pb._reconstruct_sdpa(x, dkv, 0.1))(many).float()
    assert torch.allclose(got, want, atol=2e-2 * want.abs().max().item(), rtol=2e-2)
    with fwd.dual_level():
        out, tangent = fwd.unpack_dual(pb._reconstruct_sdpa(fwd.make_dual(many[0], many[1]), dkv, 0.1))
    assert torch.allclose(out.float(), want[0], atol=2e-2 * want.abs().max().item(), rtol=2e-2)
    h = 0.125
    along = (pb._reconstruct_sdpa((many[0] + h * many[1]).float(), dkv, 0.1)
             - pb._reconstruct_sdpa((many[0] - h * many[1]).float(), dkv, 0.1)) / (2 * h)
    assert torch.allclose(tangent.float(), along, atol=5e-2 * along.abs().max().item())
    with torch.autocast("cuda", dtype=torch.float16):
        cast = pb._reconstruct_sdpa(many[0], dkv, 0.1)
    assert cast.dtype == torch.float16   # as the library's operator gives it
    assert torch.allclose(cast.float(), want[0], atol=2e-2 * want.abs().max().item(), rtol=2e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [64, 128])
def test_probabilities_keep_fp32_precision(D, dtype):
    """Values of both signs whose weighted sum nearly cancels show the weights' own errors
    beside the output's rounding. fp32 weights are off by about 2^-22 of themselves (the scores here
    are exact in fp32, so that leaves their scaling and the exponential), the result by at
    most 2^-20 of the weighted sum of magnitudes; a single token of large score and no
    value makes the other weights small."""
    from winnow_amd import packed_attention as pa
    from winnow_amd import packed_backend as pb
    B, Hq, Hkv, Q, L = 16, 8, 2, 4, 24
    g = torch.Generator().manual_seed(D)
    q = torch.randint(-8, 9, (B, Hq, Q, D), generator=g).to(dtype) / 8
    k = torch.zeros(B, Hkv, L, D)
    k[..., :6] = torch.randint(-8, 9, (B, Hkv, L, 6), generator=g) / 4
    k[:, :, 0, 6] = 24                       # the token of no value; q's channel 6 is 1
    q[..., 6] = 1
    v = torch.randint(0, 2, (B, Hkv, L, D), generator=g) * 128.0 - 64
    v[:, :, 0] = 0
    k, v = k.to(dtype), v.to(dtype)
    kv = pa.PackedKV(torch.empty(0, Hkv, 16, D, dtype=torch.uint8, device=DEV), None, None, None, None,
                     torch.full((B,), L, dtype=torch.int32, device=DEV), None, None, D)
    scale = 0.25
    got = pb._history_attention(q.to(DEV), kv, k.to(DEV), v.to(DEV), L, scale).cpu().double()
    kk, vv = (x.double().repeat_interleave(Hq // Hkv, 1) for x in (k, v))
    s = scale * (q.double() @ kk.transpose(-1, -2))
    s.masked_fill_(torch.arange(L) > (L - Q + torch.arange(Q))[:, None], -float("inf"))
    p = torch.softmax(s, -1)
    ref, size = p @ vv, p @ vv.abs()
    half = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    worst = ((got - ref).abs() / (half * ref.abs() + 2.0 ** -20 * size)).max().item()
    assert worst <= 1, f"{worst:.2f} of the bound"


def test_a_length_past_the_histories():
    """Device lengths beyond the rows of K and V (ahead of the host's, from which the rows
    were counted) count as that many rows."""
    from winnow_amd import packed_attention as pa
    from winnow_amd import packed_backend as pb
    B, Hq, Hkv, Q, D, Lmax = 2, 4, 2, 3, 64, 70
    g = torch.Generator().manual_seed(7)
    q = torch.randn(B, Hq, Q, D, generator=g).to(DEV, torch.bfloat16)
    k, v = (torch.randn(B, Hkv, Lmax, D, generator=g).to(DEV, torch.bfloat16) for _ in range(2))

    def run(lens):
        kv = pa.PackedKV(torch.empty(0, Hkv, 16, D, dtype=torch.uint8, device=DEV), None, None, None, None,
                         torch.tensor(lens, dtype=torch.int32, device=DEV), None, None, D)
        return pb._history_attention(q, kv, k, v, Lmax, 0.1)
    assert torch.equal(run((Lmax + 1, Lmax + 100)), run((Lmax, Lmax)))
