"""Ranges of keys of a prompt's tiles by the time they are expected to take: what is chosen, the executor's rule beside the
wrapper's, and the attention with every number of ranges."""
import numpy as np
import pytest
import torch


def test_chosen_ranges():
    from allpaca_amd.kernels import tuned as t

    def chosen(rows, before, heads, d, window=0):
        tiles = -(-rows // 128)
        return t._key_splits_by_time(tiles, rows, heads, d, t._prompt_passes([before, 9], [rows, 1]), window)

    assert [chosen(1500, n, 32, 64) for n in (24001, 4000, 1000, 0)] == [4, 1, 1, 1]
    assert (chosen(700, 8000, 32, 64), chosen(300, 16000, 32, 64), chosen(1024, 16384, 32, 64)) == (4, 5, 2)
    assert [chosen(1500, n, 24, 128) for n in (16000, 3000, 0)] == [3, 1, 1]
    # whole rounds of blocks stay whole; a window is what a tile sees
    assert chosen(2048, 16384, 32, 64) == 1 and chosen(2048, 30720, 32, 128) == 1
    assert chosen(1500, 24001, 32, 64, window=1000) == 1
    assert t._prompt_passes([0, 100, 5], [129, 1, 2]) == 2 + 3 + 1


def test_partial_results_are_bounded():
    """Steps of more rows than the default: their ranges' partial results would take up to 8 times the rows' outputs."""
    from allpaca_amd.kernels import tuned as t
    most = 0
    for rows in range(1000, 40000, 371):
        for heads, d in ((32, 64), (24, 128), (64, 128)):
            s = t._key_splits_by_time(-(-rows // 128), rows, heads, d, t._prompt_passes([900000], [rows]), 0)
            if s > 1:
                most = max(most, s * rows * heads * (d + 2) * 4)
    assert 0 < most <= t.KEY_PARTS_MAX


def test_the_executors_rule_is_the_wrappers_rule(monkeypatch):
    from allpaca_amd.kernels import host, tuned as t
    L = host.load()
    for most in (8, 3, 0):
        monkeypatch.setattr(t, "KEY_SPLITS_MAX", most)
        for rows in (64, 300, 700, 1024, 1500, 2048, 4000, 9000, 33000):
            for before in (0, 900, 4000, 24001, 130000):
                for heads, d in ((32, 64), (24, 128), (64, 128), (4, 64)):
                    for window in (0, 1000):
                        tiles, passes = -(-rows // 128), t._prompt_passes([before], [rows])
                        want = t._key_splits_by_time(tiles, rows, heads, d, passes, window)
                        assert L.apc_host_rule_key_splits_by_time(tiles, rows, heads, d, passes, window, most) == want


@pytest.mark.gpu
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("window", [0, 200])
def test_every_number_of_ranges(monkeypatch, d, window):
    """Portions whose tiles see very different numbers of keys, some fewer than there are ranges."""
    from test_kernels_tuned import run_attention, tuned
    for s in range(1, 9):
        monkeypatch.setattr(tuned(), "_prompt_ranges", lambda *a, s=s: s)
        run_attention(H=4, Hk=2, d=d, P_=16, lens=[1500, 130, 77], rows_per_seg=[300, 129, 1], window=window, seed=s, ranges=s)
        run_attention(H=4, Hk=2, d=d, P_=16, lens=[1500, 130, 77], rows_per_seg=[300, 129, 1], window=window, seed=s, ranges=s,
                      stale=float("nan"))
        run_attention(H=4, Hk=2, d=d, P_=16, lens=[1500], rows_per_seg=[256], window=window, seed=s, ranges=s, loud=(0, 1460, 40.0))


@pytest.mark.gpu
@pytest.mark.parametrize("H,d,off,pad", [(4, 64, 4, 4), (4, 128, 0, 4), (6, 64, 8, 8), (40, 64, 4, 12)])
@pytest.mark.parametrize("ranges", [2, 5])
def test_ranges_added_into_rows_off_16_bytes(monkeypatch, H, d, off, pad, ranges):
    """The adding kernel stores 16 bytes where the output's place and its rows allow it, else 8: the same numbers."""
    from allpaca_amd.engine.batch import Entry, pack_step
    from test_kernels_tuned import DEV, tuned
    t, Hk, P_, rows, before = tuned(), H // 2, 16, 200, 900
    blocks = -(-(before + rows) // P_)
    step = pack_step([Entry(0, [0] * rows)], [before], [0], [[list(range(1, blocks + 1))]], torch.device(DEV), [0])
    gen = torch.Generator(device=DEV).manual_seed(H + d)
    q = torch.randn(rows, H * d, generator=gen, device=DEV).bfloat16()
    cache = torch.randn(blocks + 1, 2, Hk, P_, d, generator=gen, device=DEV).bfloat16()
    monkeypatch.setattr(t, "_prompt_ranges", lambda *a: ranges)
    want = torch.empty(rows, H * d, dtype=torch.bfloat16, device=DEV)
    wide = torch.full((rows, off + H * d + pad), 9.0, dtype=torch.bfloat16, device=DEV)
    for out in (want, wide[:, off:off + H * d]):
        assert t.attention_bf16(q, 0, out, H, Hk, d, cache, P_, step.block_tables[0], step)
    assert torch.equal(wide[:, off:off + H * d], want)
    assert (wide[:, :off] == 9.0).all() and (wide[:, off + H * d:] == 9.0).all()
