"""Decoded rows of the masked attention whose heads a block finishes itself (one range of keys a row), against the plain
kernel on the same pages and against the path that cuts a row's keys into ranges: 1 to 16 heads of a kv head, contexts on
both sides of a wave's 64 keys and a block's 256, windows with and without kept first keys, chunks, sinks, head gates,
several softmax maps, odd sizes of keys and values, both output types; slots and pages no row may read hold NaN."""
import numpy as np
import pytest
import torch

from test_seredra_gpu import DEV, make_step, scattered_tables

pytestmark = pytest.mark.gpu


def launch(H, G, dk, dv, P_, lens, mask, size, keep, sinks, gate, parts, f32, blocks, monkeypatch):
    from allpaca_amd.kernels import ops, tuned
    g = torch.Generator().manual_seed(H * dk + dv)
    n_pages, tables = scattered_tables(np.random.default_rng(dk + H), lens, P_)
    cache = torch.full((n_pages + 1, G, P_ * (dk + dv)), float("nan"))
    for L, table in zip(lens, tables):
        pos = L - 1
        first = {"causal": 0, "window": max(0, L - size), "chunk": pos // size * size if size else 0}[mask]
        for t in range(L):
            if t >= first or t < keep:
                page = cache[table[t // P_]]
                page[:, t % P_ * dk:(t % P_ + 1) * dk] = torch.randn(G, dk, generator=g)
                page[:, P_ * dk + t % P_::P_] = torch.randn(G, dv, generator=g)
    n = len(lens)
    cache = cache.bfloat16().to(DEV)
    q = torch.randn(n, H * dk // parts, generator=g).bfloat16().to(DEV)
    step = make_step([(L - 1, 1) for L in lens], tables)
    sink_scores = torch.randn(H, generator=g).to(DEV) if sinks else None
    logits = torch.randn(n, H + 3, generator=g).to(DEV) if gate else None
    how = dict(key_parts=parts, sinks=sink_scores, gate=logits, keep_first=keep, out_scale=0.7)
    want = torch.empty(n, H * dv, device=DEV)
    ops.masked_attention_plain(q, want, H, G, dk, dv, cache, P_, step.block_tables[0], step.positions, step.row_seg,
                               mask, size, sinks, dk ** -0.5, **how)
    got = torch.empty(n, H * dv, device=DEV, dtype=torch.float32 if f32 else torch.bfloat16)
    monkeypatch.setattr(tuned, "MASKED_DECODE_BLOCKS", blocks)
    assert tuned.masked_attention_bf16(q, got, H, G, dk, dv, cache, P_, step.block_tables[0], step, mask, size, sinks,
                                       dk ** -0.5, **how)
    top = float(cache[~cache.isnan()].abs().max())
    return got.float(), want, top


@pytest.mark.parametrize("H, G, dk, dv, P_, lens, mask, size, keep, sinks, gate, parts, f32", [
    (6, 2, 64, 64, 16, [1, 63, 64, 65, 81, 255, 256], "causal", 0, 0, False, False, 1, False),
    (16, 1, 64, 64, 32, [3, 200, 256], "window", 128, 0, True, True, 1, False),
    (15, 3, 24, 40, 8, [9, 71, 150], "window", 9, 4, True, False, 1, True),           # kept first keys, then a gap
    (8, 2, 128, 128, 64, [257, 511, 512, 513], "causal", 0, 0, False, True, 1, True),  # several passes of a block
    (4, 4, 72, 256, 16, [130, 300], "chunk", 100, 0, True, False, 1, False),
    (8, 2, 256, 64, 16, [300, 17, 64], "window", 300, 0, False, False, 2, True),       # a context of one window
    (12, 2, 208, 136, 16, [90, 700], "window", 256, 20, False, True, 2, False),
])
def test_a_block_finishes_its_heads(H, G, dk, dv, P_, lens, mask, size, keep, sinks, gate, parts, f32, monkeypatch):
    case = (H, G, dk, dv, P_, lens, mask, size, keep, sinks, gate, parts, f32)
    one, want, top = launch(*case, 0, monkeypatch)           # no blocks to cut ranges for: one range a row
    cut, _, _ = launch(*case, 1 << 20, monkeypatch)
    # a weight is rounded to 8 bits (2^-9 of itself), so a head is off by at most 2^-9 of the largest value element;
    # the products' and sums' own float32 errors lie below 2^-14 of it, a bfloat16 output adds 2^-9 of the result
    bound = 0.7 * top * (2 ** -9 + 2 ** -14) + (0 if f32 else top * 2 ** -9)
    for got in (one, cut):
        assert float((got - want).abs().max()) <= bound
