"""Decoded rows whose work is dealt out evenly over all waves of the launch, against the plain attention: rows inside one
wave's share, rows in two and in many pieces, shares that end at a row's first and last step, more than 64 rows, groups
wider than a tile of 16 heads, windows, pages of 8, and slots that hold NaN."""
import ctypes

import pytest
import torch

from test_kernels_tuned import run_attention, tuned

RAGGED = [1 + (i * 977) % 2100 for i in range(70)]


@pytest.fixture
def even(monkeypatch):
    monkeypatch.setattr(tuned(), "EVEN_MIN_PAIRS", 1)
    monkeypatch.setattr(tuned(), "EVEN_MIN_SPAN", 0)


@pytest.mark.gpu
@pytest.mark.parametrize("H,Hk,d,P_,lens,rows,window", [
    (32, 8, 128, 16, [2048, 1, 17, 700, 2047], [1] * 5, 0),
    (6, 2, 64, 16, RAGGED, [1] * 70, 0),                          # rows looked at in two goes
    (6, 2, 64, 16, RAGGED, [1] * 70, 300),
    (8, 8, 128, 16, [256] * 32, [1] * 32, 0),                     # shares that end where rows do
    (2, 1, 128, 16, [9000, 31, 32, 33, 1], [1] * 5, 0),           # one row over most of the waves
    (6, 2, 48, 8, [4000, 129, 64, 1], [1] * 4, 0),                # a wave's keys in several pieces (pages of 8)
    (20, 1, 32, 24, [100, 2600, 64], [1] * 3, 0),                 # a group wider than one tile of heads
    (34, 2, 80, 16, [100, 2600], [1] * 2, 0),
    (16, 1, 256, 32, [500, 90], [1] * 2, 0),
    (4, 2, 32, 16, [300, 200, 90, 2500], [1] * 4, 100),
    (4, 4, 16, 16, [300, 200, 90, 1200], [1] * 4, 1000),
    (8, 2, 128, 16, [900, 133, 400], [1, 40, 1], 5),              # decoded rows beside a portion
])
def test_rows_of_any_lengths(even, H, Hk, d, P_, lens, rows, window):
    run_attention(H=H, Hk=Hk, d=d, P_=P_, lens=lens, rows_per_seg=rows, window=window, seed=H + d)
    run_attention(H=H, Hk=Hk, d=d, P_=P_, lens=lens, rows_per_seg=rows, window=window, seed=H + d, stale=float("nan"))


@pytest.mark.parametrize("H,Hk,d", [(20, 1, 32), (24, 1, 64), (34, 2, 80), (48, 2, 128), (71, 1, 256), (32, 8, 128),
                                    (32, 32, 64), (16, 1, 16), (64, 2, 128)])
def test_the_tiles_pieces_lie_apart(H, Hk, d):
    """The places of all kv head tiles, also of a group's last one with fewer than 16 heads, in the workspace and apart."""
    from allpaca_amd.kernels import lib
    L = lib.load("tuned")
    tiles, at = Hk * -(-(H // Hk) // 16), 0
    for tile in range(tiles):
        first, end = ctypes.c_longlong(), ctypes.c_longlong()
        assert L.apc_attention_decode_even_region(H, Hk, d, tile, ctypes.byref(first), ctypes.byref(end)) == 0
        heads = min(16, H // Hk - tile % (tiles // Hk) * 16)
        waves = max(1, 256 // tiles) * 4
        assert first.value >= at and end.value - first.value == waves * 2 * heads * (d + 4)
        at = end.value
    assert at <= L.apc_attention_decode_even_workspace(H, Hk, d)
    assert L.apc_attention_decode_even_region(H, Hk, d, tiles, ctypes.byref(first), ctypes.byref(end)) < 0


@pytest.mark.gpu
@pytest.mark.parametrize("H,Hk,d,n", [(20, 1, 32, 128), (34, 2, 64, 64), (24, 1, 128, 128)])
def test_wide_groups_with_work_for_nearly_all_waves(H, Hk, d, n):
    """Groups of several tiles of heads, the last one short, in the rule's own range: pieces of every tile in most places."""
    t = tuned()
    lens = [1100 + (i * 977) % 400 for i in range(n)]
    assert t._decode_even(n * Hk * -(-(H // Hk) // 16), max(lens))
    waves, steps = 4 * (256 // (Hk * -(-(H // Hk) // 16))), sum(-(-x // 32) + 2 for x in lens)
    assert steps / max(8, -(-steps // waves)) > 0.9 * waves          # (a wave's share, 8 at least)
    run_attention(H=H, Hk=Hk, d=d, P_=16, lens=lens, rows_per_seg=[1] * n, seed=n)


@pytest.mark.gpu
def test_chosen_by_itself_and_the_counters_are_zero_again():
    t = tuned()
    run_attention(H=16, Hk=8, d=64, P_=16, lens=RAGGED[:40], rows_per_seg=[1] * 40, seed=3)
    used = [c for have in t._counters.values() for c in have]
    assert used and all(int(c.abs().sum()) == 0 for c in used)


def test_the_executors_rule_is_the_wrappers_rule():
    from allpaca_amd.kernels import host, tuned as t
    L = host.load()
    for pairs in (1, 64, 255, 256, 512, 4096):
        for span in (1, 1024, 1025, 2048, 131072):
            assert bool(L.apc_host_rule_decode_even(pairs, span, t.EVEN_MIN_PAIRS, t.EVEN_MIN_SPAN)) == t._decode_even(pairs, span)


def test_recordings_share_counters_within_an_engine_only(monkeypatch):
    """Graphs of two engines may be replayed side by side on two streams, and calls outside of graphs on a third.  A buffer
    that a recording allocates is cleared by that graph's replays alone: it must not be kept for others."""
    from allpaca_amd.kernels import tuned as t
    stream, recording = [1], [False]
    monkeypatch.setattr(t, "_counters", {})
    monkeypatch.setattr(t._ops, "_stream", lambda: stream[0])
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: recording[0])
    cpu = torch.device("cpu")
    one, two = [], []
    recording[0] = True
    assert t._pair_counters(cpu, 8, one).numel() >= 8 and not one        # nothing was made before: the recording's own
    assert t._pair_counters(cpu, 8).numel() >= 8 and not t._counters
    recording[0] = False
    first, other = t._pair_counters(cpu, 8, one), t._pair_counters(cpu, 8, two)
    eager = t._pair_counters(cpu, 8)
    stream[0] = 2
    places = [x.data_ptr() for x in (first, other, eager, t._pair_counters(cpu, 8))]
    assert len(set(places)) == 4 and t._pair_counters(cpu, 8, one) is first
    recording[0], stream[0] = True, 3
    assert t._pair_counters(cpu, 8, one) is first and t._pair_counters(cpu, 8, two) is other
    alone = t._pair_counters(cpu, 8)                                     # a caller's own graph
    assert alone.data_ptr() not in places and (cpu.type, 0, 3) not in t._counters
    assert t._pair_counters(cpu, 5000, one).numel() >= 5000 and len(one) == 1
    recording[0] = False
    assert t._pair_counters(cpu, 5000, one).numel() >= 5000 and one[0] is first


def test_a_step_that_does_not_say_where_its_prompts_start_is_not_cut():
    from allpaca_amd.kernels import tuned as t
    assert t._prompt_passes(None, None) == 0
    assert t._key_splits_by_time(12, 1500, 32, 64, 0, 0) == 1
