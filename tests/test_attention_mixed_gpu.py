"""Prompt rows and decoded rows of a step in one launch: the bits that the two launches leave, whatever the split."""
import numpy as np
import pytest
import torch

from test_kernels_tuned import BF, DEV, gen, make_cache, tuned

pytestmark = pytest.mark.gpu


# d, H, Hk, page, contexts, rows of the step, window, ranges of the decoded rows' keys (0: a block a pair), ranges of the prompt's
@pytest.mark.parametrize("d,H,Hk,P_,lens,rows,window,n_parts,splits", [
    (128, 32, 8, 16, [1300, 2047, 1, 700], [504, 1, 1, 1], 0, 16, 1),          # few tiles beside four blocks a pair
    (128, 4, 2, 16, [128, 33, 257], [128, 1, 1], 0, 0, 1),                      # one tile; a block a pair
    (64, 8, 2, 32, [65, 900, 64, 31], [65, 1, 1, 1], 0, 5, 1),                  # a tile just large enough; a last block with one range
    (64, 40, 2, 16, [200, 500, 77], [129, 1, 1], 0, 48, 2),                     # two tiles of heads a group; twelve blocks a pair
    (128, 6, 6, 64, [400, 300, 1000], [190, 1, 1], 100, 8, 2),                  # a window; groups of one head
    (64, 16, 8, 16, [2000, 70] + [9 + 61 * i for i in range(33)], [1500, 1] + [1] * 33, 37, 0, 3),
    (128, 16, 16, 16, [700, 300] + [9 + 61 * i for i in range(17)], [600, 270] + [1] * 17, 0, 4, 1),
])
def test_one_launch_leaves_what_two_leave(monkeypatch, d, H, Hk, P_, lens, rows, window, n_parts, splits):
    from allpaca_amd.engine.batch import Entry, pack_step
    from allpaca_amd.kernels import lib, ops
    t, L = tuned(), lib.load("tuned")
    cache, bt, _, _ = make_cache(lens, Hk, d, P_, BF, seed=d + H, stale=300.0)
    pos0 = [n - r for n, r in zip(lens, rows)]
    tables = [[list(bt[i, : -(-n // P_)].cpu().numpy()) for i, n in enumerate(lens)]]
    used = {int(p) for tb in tables[0] for p in tb}
    spare = next(p for p in range(cache.shape[0]) if p not in used)
    step = pack_step([Entry(i, [0] * r, []) for i, r in enumerate(rows)], pos0, [0] * len(lens), tables, torch.device(DEV), [spare],
                     tile_rows=ops.attention_tile_rows(BF))
    T, n, G, nz = sum(rows), step.n_decode_rows, H // Hk, -(-n_parts // 4)
    assert n == sum(r == 1 for r in rows) and step.decode_rows is not None
    q = gen(T, H * d + 16, seed=7, scale=2.5, dtype=BF).to(DEV)
    table, stream = step.block_tables[0], ops._stream()
    counters = torch.zeros(n * Hk * -(-G // 16), dtype=torch.int32, device=DEV)

    def room():
        return (torch.full((max(1, n * H * nz * (d + 2)),), float("nan"), device=DEV),
                torch.full((splits * T * H * (d + 2),), float("nan"), device=DEV))

    def prompt_args(out, parts):
        return (q.data_ptr(), q.stride(0), 16, out.data_ptr(), out.stride(0), H, Hk, d, cache.data_ptr(), P_, table.data_ptr(), table.shape[1],
                step.positions.data_ptr(), step.row_seg.data_ptr(), step.tile_row0.data_ptr(), step.tile_rows.data_ptr(), step.n_tiles,
                T - n, window, d ** -0.5, splits, T, parts.data_ptr() if splits > 1 else 0)

    want = torch.full((T, H * d), 3.0, dtype=BF, device=DEV)
    ws, parts = room()
    lib.check(L.apc_attention_prefill_bf16(*prompt_args(want, parts), stream), "prompt rows")
    lib.check(L.apc_attention_decode_bf16(
        q.data_ptr(), q.stride(0), 16, want.data_ptr(), want.stride(0), n, H, Hk, d, cache.data_ptr(), P_, table.data_ptr(), table.shape[1],
        step.positions.data_ptr(), step.row_seg.data_ptr(), step.decode_rows.data_ptr(), window, d ** -0.5, 0, n_parts,
        ws.data_ptr() if n_parts else 0, counters.data_ptr() if n_parts else 0, stream), "decoded rows")
    assert L.apc_attention_mixed_takes(H, Hk, d, P_, step.n_tiles, T - n, n, n_parts, int(n_parts > 0))
    for _ in range(3):
        out = torch.full((T, H * d), 5.0, dtype=BF, device=DEV)
        ws, parts = room()
        lib.check(L.apc_attention_mixed_bf16(
            *prompt_args(out, parts), step.decode_rows.data_ptr(), n, n_parts, ws.data_ptr() if n_parts else 0,
            counters.data_ptr() if n_parts else 0, stream), "all rows")
        assert torch.equal(out, want)
        assert not counters.any()


def test_sizes_that_take_two_launches():
    from allpaca_amd.kernels import lib
    L = lib.load("tuned")
    assert L.apc_attention_mixed_takes(32, 8, 128, 16, 4, 504, 8, 16, 1)
    assert not L.apc_attention_mixed_takes(32, 8, 96, 16, 4, 504, 8, 16, 1)         # heads of 96
    assert not L.apc_attention_mixed_takes(32, 8, 128, 24, 4, 504, 8, 16, 1)        # pages of 24
    assert not L.apc_attention_mixed_takes(32, 8, 128, 16, 4, 255, 8, 16, 1)        # tiles mostly empty
    assert not L.apc_attention_mixed_takes(32, 8, 128, 16, 0, 0, 8, 16, 1)          # no prompt
    assert not L.apc_attention_mixed_takes(32, 8, 128, 16, 4, 504, 0, 16, 1)        # nothing decoded


# rows of the prompt's portion, decoded rows and their contexts; heads and their size, window; which launches the executor issues
@pytest.mark.parametrize("portion,contexts,H,Hk,d,window,launches", [
    (200, [300, 20, 700], 8, 2, 128, None, ["attention_mixed_bf16"]),                        # ranges of keys, the last block adds
    (200, [300, 20, 700], 8, 2, 64, None, ["attention_mixed_bf16"]),
    (130, [33, 100, 250], 8, 2, 64, None, ["attention_mixed_bf16"]),                          # a block a pair
    (65, [500, 90], 8, 4, 128, 100, ["attention_mixed_bf16"]),                                # a window
    (300, [500, 90, 610], 16, 2, 64, 70, ["attention_mixed_bf16"]),
    (40, [300, 700], 8, 2, 128, None, ["attention_prefill_bf16", "attention_decode_bf16 (last block merges)"]),   # no tile half full
    (1024, [40 + i for i in range(33)], 32, 8, 128, None, ["attention_prefill_bf16", "attention_decode_bf16 (whole)"]),   # whole rounds of tiles
    (800, [40 + i for i in range(33)], 32, 8, 128, None, ["attention_mixed_bf16"]),
])
def test_the_executor_gives_the_python_walks_bits_and_issues_the_launches(monkeypatch, portion, contexts, H, Hk, d, window, launches):
    from allpaca_amd.engine.batch import Entry
    from allpaca_amd.engine.runner import ModelRunner
    from allpaca_amd.models import DecoderModel, describe_model
    from allpaca_amd.parts import Runtime
    import helpers
    cfg = dict(helpers.TINY_B, hidden_size=256, num_attention_heads=H, num_key_value_heads=Hk, head_dim=d, intermediate_size=512, num_hidden_layers=2,
               vocab_size=500, max_position_embeddings=4096, rope_scaling=None)
    rng = np.random.default_rng(portion)
    toks = [rng.integers(0, 500, size=n).tolist() for n in [portion + 77] + contexts]
    got = []
    for python_walk in (True, False):
        if python_walk:
            monkeypatch.setenv("ALLPACA_AMD_PYTHON_WALK", "1")
        else:
            monkeypatch.delenv("ALLPACA_AMD_PYTHON_WALK", raising=False)
        _, _, spec = describe_model(cfg)
        if window:
            for block in spec.blocks:
                block.parts["mixer"].params["window"] = window
        model = DecoderModel(spec)
        g = torch.Generator(device=DEV).manual_seed(1)
        tensors = {name: torch.randn(ps.shape, generator=g, device=DEV, dtype=BF).mul_(0.1) for name, ps in model.param_specs().items()}
        model.bind(tensors, Runtime(torch.device(DEV), BF, 4096))
        runner = ModelRunner(model, 16, 64 + sum(-(-len(t) // 16) + 1 for t in toks), len(toks))
        assert (runner.native is None) == python_walk
        for i, t in enumerate(toks):
            runner.admit(i)
            runner.step([Entry(i, t[:77] if i == 0 else t[:-1], [])])
        if not python_walk:
            runner.native.timing(True)
        got.append(runner.step([Entry(0, toks[0][77:], [portion - 1])] + [Entry(i, t[-1:], [0]) for i, t in enumerate(toks) if i]).cpu())
        if not python_walk:
            issued = [name for name, _ in runner.native.timing_report() if name.startswith("attention")]
            runner.native.timing(False)
            assert issued == launches * 2
    assert torch.isfinite(got[0]).all() and torch.equal(*got)
