"""The reconstruct route refuses lengths and page ids out of range before any launch, as the
decode does: its kernels read pages by the table's ids, unchecked."""
from __future__ import annotations

import pytest
import torch

from winnow_amd import packed_attention as pa
from winnow_amd import packed_backend as pb


def _handle(D, table, lens, mirrors):
    P, Hkv, S = 4, 2, 16
    quant = pa.Quantizer(torch.eye(D), torch.zeros(16), 4)
    pages, norms = torch.zeros(P, Hkv, S, D // 2, dtype=torch.uint8), torch.zeros(P, Hkv, S, dtype=torch.float16)
    table, lens = torch.tensor(table, dtype=torch.int32), torch.tensor(lens, dtype=torch.int32)
    return pa.PackedKV(pages, norms, pages, norms, table, lens, quant, quant, D,
                       seq_lens_host=lens if mirrors else None, page_table_host=table if mirrors else None)


@pytest.mark.parametrize("wide", [0, 300])   # table entries past every length: small and large tables
@pytest.mark.parametrize("mirrors", [True, False])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("table,lens,bad", [([[0, 1], [2, 4]], [32, 20], 1),      # a page past the pool
                                            ([[0, -1], [2, 3]], [17, 20], 0),     # an unused entry in use
                                            ([[0, 1], [2, 3]], [5, 33], 1)])      # more tokens than the table holds
def test_out_of_range(monkeypatch, D, table, lens, bad, mirrors, wide):
    if wide and lens[1] == 33:
        lens = [5, 33 + 16 * wide]
    table = [row + [-1] * wide for row in table]
    calls = []
    monkeypatch.setattr(pb._lib, "call", lambda name, *a: calls.append(name))
    kv = _handle(D, table, lens, mirrors)
    with pytest.raises(pa.UnsupportedLayout):
        pb._reconstruct_sdpa(torch.zeros(2, 4, 3, D, dtype=torch.bfloat16), kv, 0.1)
    with pytest.raises(pa.UnsupportedLayout):
        pb.dequantize_history(kv, kv.k_pages, kv.k_norms, kv.k_quant, bad, torch.float32)
    assert calls == []


def test_entries_past_a_length_are_not_looked_at(monkeypatch):
    monkeypatch.setattr(pb._lib, "call", lambda name, *a: None)
    monkeypatch.setattr(pb._lib, "stream_of", lambda device: None)
    monkeypatch.setattr(torch.cuda, "device", lambda device: torch.no_grad())
    kv = _handle(64, [[0, -1], [2, 9]], [16, 3], True)
    for b, L in enumerate((16, 3)):
        assert pb.dequantize_history(kv, kv.k_pages, kv.k_norms, kv.k_quant, b, torch.float32).shape == (1, 2, L, 64)


def test_the_short_look_agrees_with_the_long_one():
    """Random tables, small and large, with odd ids and lengths here and there."""
    import random
    r = random.Random(1)
    refused = 0
    for _ in range(1500):
        B, W, S, P = r.randint(1, 6), r.choice([1, 2, 5, 30, 60]), r.choice([1, 16, 12]), r.choice([1, 5, 100])
        odd = [-1, P, 2 ** 31 - 1, -2 ** 31]
        table = torch.tensor([[r.choice(odd) if r.random() < 0.03 else r.randrange(P) for _ in range(W)] for _ in range(B)],
                             dtype=torch.int32)
        lens = torch.tensor([r.choice([0, 1, W * S, W * S + 1, -1]) if r.random() < 0.2 else r.randint(0, W * S) for _ in range(B)],
                            dtype=torch.int32)
        said = []
        for check in (pa.check_page_ranges, pb._check_histories):
            try:
                said.append(check(lens, table, P, S))
            except pa.UnsupportedLayout as e:
                said.append(str(e))
        assert said[0] == said[1], (lens, table, P, S)
        refused += said[0] is not None
    assert 300 < refused < 1200
