"""The contiguous cache refuses K and V that its buffers do not hold, before any launch.

The append kernels address the buffers by the sizes of K, so a step of another batch,
head count or head_dim than the first one's, or a V that is shorter than K, would reach
past an allocation. The C calls are stubbed: a step that gets as far as one is recorded.
"""
from __future__ import annotations

import contextlib

import pytest
import torch

from winnow_amd import cache as wc


@pytest.fixture
def calls(monkeypatch):
    names = []
    monkeypatch.setattr(wc._lib, "call", lambda name, *a: names.append(name))
    monkeypatch.setattr(wc._lib, "stream_of", lambda device: None)
    monkeypatch.setattr(torch.cuda, "device", lambda device: contextlib.nullcontext())
    monkeypatch.setattr(wc, "tq_dequant", lambda *a, **k: names.append("tq_dequant"))
    return names


def _step(B, H, n, D, device="cpu", dtype=torch.bfloat16):
    return torch.zeros(B, H, n, D, dtype=dtype, device=device)


def _layer(n_out, D=128):
    return wc.TQPackedLayer(D, 4, "cpu", 60, num_outlier_channels=n_out, outlier_bits=8 if n_out else 0)


@pytest.mark.parametrize("n_out", [8, 0])
@pytest.mark.parametrize("k,v", [((4, 2, 5, 128), None), ((1, 2, 5, 128), None),      # another batch
                                 ((2, 3, 5, 128), None), ((2, 1, 5, 128), None),      # other heads
                                 ((2, 2, 5, 64), None),                               # another head_dim
                                 ((2, 2, 5, 128), (2, 2, 3, 128)), ((2, 2, 5, 128), (1, 2, 5, 128)),
                                 ((2, 2, 5, 128), (2, 2, 5, 64))])
@pytest.mark.parametrize("reset", [True, False])
def test_a_step_that_the_buffers_do_not_hold(calls, n_out, k, v, reset):
    layer = _layer(n_out)
    layer.update(_step(2, 2, 7, 128), _step(2, 2, 7, 128))
    assert calls
    calls.clear()
    if reset:
        layer.reset()
    before = layer.get_seq_length()
    with pytest.raises(ValueError):
        layer.update(_step(*k), _step(*(v or k)))
    assert calls == [] and layer.get_seq_length() == before
    layer.update(_step(2, 2, 5, 128), _step(2, 2, 5, 128))
    assert calls and layer.get_seq_length() == before + 5


@pytest.mark.parametrize("n_out", [8, 0])
def test_operands_off_the_cache_device(calls, n_out):
    layer = _layer(n_out)
    with pytest.raises(ValueError):
        layer.update(_step(2, 2, 7, 128), _step(2, 2, 3, 128))   # nothing is set up for a V that differs
    assert not layer.is_initialized
    layer.update(_step(2, 2, 7, 128), _step(2, 2, 7, 128))
    calls.clear()
    for k, v in (("meta", "meta"), ("cpu", "meta"), ("meta", "cpu")):
        with pytest.raises(ValueError):
            layer.update(_step(2, 2, 1, 128, k), _step(2, 2, 1, 128, v))
    assert calls == []
