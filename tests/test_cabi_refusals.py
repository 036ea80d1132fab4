"""The entry points of the outlier append, the rows dequantization and the attention over
histories refuse what their kernels do not serve before any launch (no GPU here: the
pointers are fake, aligned and never read)."""
from __future__ import annotations

import pytest

from winnow_amd import _lib

P = 1 << 20


def _split(D=128, count2=8, bw=4, bw2=8, n=3, cap=10, pos=0, k=P, dtype=2, stride=128):
    return ("wn_append_split", k, stride, stride, stride, P, stride, stride, stride, dtype, P, P, count2, P, bw, P, bw2,
            P, P, P, P, P, P, P, P, 1, 2, n, D, cap, pos, None)


def _rows(D=128, bw=4, count2=0, bw2=0, planes=1, L=4, plane_rows=4, dtype=0, v_norms=P, second=P):
    two = (second, second, second, second, bw2, second) if count2 else (None, None, None, None, 0, None)
    return ("wn_dequantize_rows", P, P, P, v_norms, bw, P, *two, count2, P, P, planes, L, plane_rows, D, P, P, dtype, None)


def _pages(D=64, bw=4, S=16, Lpad=8, B=1, dtype=0, out=P):
    return ("wn_dequantize_pages", P, 0, 0, P, 0, 0, P, 1, P, B, Lpad, 2, S, P, P, bw, D, out, dtype, None)


def _histories(D=128, S=16, dtype=2, pages=P, stride=1024):
    return ("wn_dequantize_histories", pages, stride, 512, P, 16, 8, P, 1, P, 1, 8, 2, S, P, P, 4, D, P, dtype, 0, None)


def _attention(D=128, dtype=2, q=P, stride=128, splits=1, ws=1 << 30, Hq=4, Hkv=2, Q=3, Lpad=64):
    return ("wn_history_attention", q, dtype, stride, stride, stride, P, P, P, P, P, ws, 1, Hq, Hkv, Q, D, Lpad, 1.0, splits, None)


@pytest.mark.parametrize("args,says", [
    (_split(D=96), "head_dim 96"), (_split(n=11), "bad sizes"), (_split(pos=8), "bad sizes"), (_split(dtype=3), "dtype"),
    (_split(count2=0), "outlier channels"), (_split(count2=128), "outlier channels"), (_split(bw=3, count2=9), "outlier channels"),
    (_split(k=None), "null operand"), (_split(k=P + 2), "16-byte aligned"), (_split(stride=129), "16-byte aligned"),
    (_rows(D=257), "head_dim 257"), (_rows(D=0), "head_dim 0"), (_rows(bw=7), "bit widths"), (_rows(D=31, bw=3), "whole bytes"),
    (_rows(L=5), "bad sizes"), (_rows(dtype=4), "dtype"), (_rows(planes=1 << 20, L=1 << 12, plane_rows=1 << 12), "too many rows"),
    (_rows(v_norms=None), "null operand"), (_rows(count2=8, bw2=8, second=None), "null outlier operand"),
    (_pages(S=12), "S=12"), (_pages(D=300), "head_dim 300"), (_pages(bw=7), "7 bits"), (_pages(dtype=9), "dtype"),
    (_pages(out=None), "null operand"), (_pages(B=1 << 16, Lpad=1 << 16), "too many rows"),
    (_histories(D=64), "head_dim 64"), (_histories(S=12), "S=12"), (_histories(pages=P + 8), "16-byte aligned"),
    (_histories(stride=1000), "16-byte aligned"), (_histories(dtype=5), "dtype"),
    (_attention(D=32), "head_dim 32"), (_attention(dtype=0), "dtype"), (_attention(q=P + 8), "16-byte aligned"),
    (_attention(stride=132), "multiples of 8"), (_attention(splits=0), "num_splits"), (_attention(splits=5000), "num_splits"),
    (_attention(ws=10), "workspace"), (_attention(Hq=5), "bad sizes"), (_attention(Q=1 << 24), "too large"),
    (_attention(Lpad=-1), "bad sizes"),
])
def test_refused(args, says):
    with pytest.raises(_lib.WinnowHipError, match=says):
        _lib.call(*args)


@pytest.mark.parametrize("args", [_split(n=0), _rows(L=0), _rows(planes=0), _pages(Lpad=0), _pages(B=0)])
def test_nothing_to_do(args):
    _lib.call(*args)
