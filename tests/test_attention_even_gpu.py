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
    monkeypatch.setattr(tuned(), "EVEN_ALONE_MIN_PAIRS", 1)
    monkeypatch.setattr(tuned(), "_even_pays", lambda *a: True)


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
    for stale in (0.0, float("nan")):
        run_attention(H=H, Hk=Hk, d=d, P_=P_, lens=lens, rows_per_seg=rows, window=window, seed=H + d, stale=stale,
                      entry="apc_attention_decode_even_bf16")


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
def test_wide_groups_with_work_for_nearly_all_waves(even, H, Hk, d, n):
    """Groups of several tiles of heads, the last one short: pieces of every tile in most of its places."""
    lens = [1100 + (i * 977) % 400 for i in range(n)]
    waves, steps = 4 * (256 // (Hk * -(-(H // Hk) // 16))), sum(-(-x // 32) + 2 for x in lens)
    assert steps / max(8, -(-steps // waves)) > 0.9 * waves          # (a wave's share, 8 at least)
    run_attention(H=H, Hk=Hk, d=d, P_=16, lens=lens, rows_per_seg=[1] * n, seed=n, entry="apc_attention_decode_even_bf16")


@pytest.mark.gpu
@pytest.mark.parametrize("lens,chosen", [(RAGGED[:40], True), ([1100] * 32, False)])
def test_chosen_by_itself_and_the_counters_are_zero_again(monkeypatch, lens, chosen):
    t = tuned()
    monkeypatch.setattr(t, "_counters", {})
    run_attention(H=16, Hk=8, d=64, P_=16, lens=lens, rows_per_seg=[1] * len(lens), seed=3,
                  entry="apc_attention_decode_even_bf16" if chosen else "apc_attention_decode_bf16")
    used = [c for have in t._counters.values() for c in have]
    assert bool(used) == chosen and all(int(c.abs().sum()) == 0 for c in used)


def small_runner(model, **kw):
    from allpaca_amd.engine.runner import ModelRunner
    return ModelRunner(model, 16, 6000, 48, **kw)


@pytest.mark.gpu
@pytest.mark.parametrize("walk", [False, True])
def test_graphs_replayed_while_the_rows_lengths_change(monkeypatch, walk):
    """Steps of 32 requests on 8 kv heads whose lengths move from very different to equal and back,
    with eager steps and synchronisations between the replays, through the compiled executor and walked in Python: each
    against the same step on a block a (row, kv head) pair, outside of a graph."""
    from allpaca_amd.engine.batch import Entry, decode_work
    from allpaca_amd.models import DecoderModel, describe_model
    from allpaca_amd.config import preset
    from allpaca_amd.parts import Runtime
    t = tuned()
    if walk:
        monkeypatch.setenv("ALLPACA_AMD_PYTHON_WALK", "1")
    cfg = dict(preset("llama-3.2-1b"), hidden_size=256, intermediate_size=512, num_attention_heads=16, num_key_value_heads=8,
               head_dim=64, num_hidden_layers=2, vocab_size=1000)
    _, _, spec = describe_model(cfg)
    model = DecoderModel(spec)
    g = torch.Generator(device="cuda").manual_seed(1)
    model.bind({n: torch.randn(ps.shape, generator=g, device="cuda", dtype=torch.bfloat16).mul_(0.06).to(
        torch.float32 if ps.store == "float32" else torch.bfloat16) for n, ps in model.param_specs().items()},
        Runtime(torch.device("cuda:0"), torch.bfloat16, 4096))
    toks = [torch.randint(0, 1000, (2300,), generator=torch.Generator().manual_seed(i)).tolist() for i in range(32)]
    ragged, equal = [1 + (i * 977) % 2100 for i in range(32)], [1100] * 32
    # the lengths of the requests in every step; requests are cut back or given a portion of prompt in between
    plan = [ragged, ragged, [n + 100 for n in ragged], equal, equal, ragged[::-1], ragged, [2100] + [33] * 31]
    assert all(t._decode_shares(32, 2048, decode_work(lens), (8, True, 0)) == (lens is not equal) for lens in plan)

    def run(graphs):
        runner, out, at = small_runner(model, use_graphs=graphs), [], [0] * 32
        for i in range(32):
            runner.admit(i)
        for lens in plan:
            for i, n in enumerate(lens):                     # n tokens in the cache, then one step for all
                if at[i] > n:
                    runner.cache.truncate(i, n)
                elif at[i] < n:
                    runner.step([Entry(i, toks[i][at[i]:n], [])])
            for more in range(3):
                lg = runner.step([Entry(i, [toks[i][n + more]], [0]) for i, n in enumerate(lens)])
                out.append(lg.float().clone())
            at = [n + 3 for n in lens]
        torch.cuda.synchronize()
        return runner, out

    shared, got = run(True)
    assert {k[2:] for k in shared.graphs} == {(True,), (False,)} and shared.graph_replays == 3 * len(plan)
    counters = shared.pair_counters if walk else [shared.native.counters]
    assert (shared.native is None) == walk and counters and all(int(c.abs().sum()) == 0 for c in counters)
    monkeypatch.setattr(t, "EVEN_MIN_PAIRS", 1 << 30)
    _, want = run(False)
    for step, (a, b) in enumerate(zip(got, want)):
        # the same kernels but for where keys are cut: weights of 8 bits, twice over two layers
        assert float((a - b).abs().max()) <= 2.0 ** -6 * float(b.abs().max()), step


@pytest.mark.gpu
def test_the_executor_shares_out_rows_of_different_lengths():
    from allpaca_amd.engine.batch import Entry
    from allpaca_amd.models import DecoderModel, describe_model
    from allpaca_amd.config import preset
    from allpaca_amd.parts import Runtime
    cfg = dict(preset("llama-3.2-1b"), hidden_size=256, intermediate_size=512, num_attention_heads=16, num_key_value_heads=8,
               head_dim=64, num_hidden_layers=1, vocab_size=1000)
    _, _, spec = describe_model(cfg)
    model = DecoderModel(spec)
    model.bind({n: torch.zeros(ps.shape, device="cuda", dtype=torch.float32 if ps.store == "float32" else torch.bfloat16)
                for n, ps in model.param_specs().items()}, Runtime(torch.device("cuda:0"), torch.bfloat16, 4096))
    for lens, want in ((RAGGED[:32], "even shares"), ([1100] * 32, "whole")):
        runner = small_runner(model)
        for i, n in enumerate(lens):
            runner.admit(i)
            runner.step([Entry(i, [1] * n, [])])
        runner.native.timing(True)
        runner.step([Entry(i, [1], [0]) for i in range(32)])
        names = [name for name, _ in runner.native.timing_report()]
        assert [n for n in names if "attention" in n] == [f"attention_decode_bf16 ({want})"], names


def test_the_executors_rule_is_the_wrappers_rule():
    from allpaca_amd.kernels import host, tuned as t
    L = host.load()
    for pairs in (1, 64, 255, 256, 512, 1023, 1024, 4096, 4097, 8192):
        for span in (1, 1024, 1025, 2048, 131072):
            for fits in (False, True):
                got = L.apc_host_rule_decode_even(pairs, span, fits, t.EVEN_MIN_PAIRS, t.EVEN_MIN_SPAN)
                assert bool(got) == t._decode_even(pairs, span, fits), (pairs, span, fits)
    for rows in (8, 12, 32, 40, 64, 96, 256, 512):
        for longest in (1, 33, 40, 50, 64, 129, 4000):
            for part in (0, 1, 3, 5, 8, 10):
                steps = longest + (rows - 1) * max(1, longest * part // 10)
                for tiles in (1, 2, 8, 12, 32, 300):
                    for window in (0, 1500, 4096):
                        got = L.apc_host_rule_even_pays(steps, longest, rows, tiles, window)
                        assert bool(got) == t._even_pays(steps, longest, rows, tiles, window), (rows, longest, steps, tiles, window)


def test_rows_of_one_length_keep_a_block_a_pair():
    """32 and 64 rows on 8 kv heads: shares from where the lengths differ much, whatever the longest row is."""
    from allpaca_amd.engine.batch import decode_work
    from allpaca_amd.kernels import tuned as t
    spread = lambda n, lo, hi: [int(lo * (hi / lo) ** (i * 0.618 % 1.0)) for i in range(n)]  # noqa: E731
    for n in (32, 64):
        pays = lambda lens, window=0: t._even_pays(*decode_work(lens), n, 8, window)  # noqa: E731
        assert not pays([1100] * n) and not pays([2048] * n) and not pays([4096] * n)
        assert pays(spread(n, 90, 2100)) and pays([8000] + [100] * (n - 1))
        assert not pays([8000] + [2000] * (n - 1), window=1500)      # all rows see as many keys
    assert decode_work([]) == (0, 0) and decode_work([1, 32, 33]) == (4, 2)
    assert not t._even_pays(0, 0, 64, 8, 0)                          # a step that does not say


def test_graphs_of_a_bucket_are_told_apart_by_the_rows_lengths():
    from allpaca_amd.engine.batch import decode_work
    from allpaca_amd.kernels import tuned as t
    shapes = {(8, True, 0), (8, True, 1200)}
    assert t.decode_routes_differ(64, 2048, shapes) and not t.decode_routes_differ(64, 1024, shapes)
    assert not t.decode_routes_differ(16, 2048, shapes) and not t.decode_routes_differ(64, 2048, {(8, False, 0)})
    assert t.decode_routes(64, 2048, decode_work([2048] * 64), shapes) == (False, False)
    assert t.decode_routes(64, 8192, decode_work([8000] + [1] * 63), shapes) == (True, True)
    assert t.decode_routes(64, 8192, decode_work([8000] + [1200] * 63), shapes) == (True, False)


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
