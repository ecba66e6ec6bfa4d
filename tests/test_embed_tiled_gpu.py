"""Rows of an embedding kept in tiles: sizes on both sides of a piece of 8 elements, a tile of 32 and a block of 1,024,
both output types, output rows that 16-byte stores may not take; exact, since a table's element is only widened."""
import pytest
import torch

from test_kernels_tuned import BF, DEV, gen, pack

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [8, 24, 32, 41, 1016, 1024, 1032, 4104])
@pytest.mark.parametrize("dtype", [torch.float32, BF])
@pytest.mark.parametrize("pad", [0, 2, 4, 8])
def test_rows_of_the_table(dim, dtype, pad):
    from allpaca_amd.kernels import ops
    table = gen(37, dim, seed=dim, dtype=BF).to(DEV)
    toks = torch.tensor([36, 0, 15, 16, 31, 36, 5], dtype=torch.int32, device=DEV)
    rows = torch.full((7, dim + pad), 5.0, dtype=dtype, device=DEV)
    ops.embed_rows(pack(table), toks, rows[:, :dim])
    assert torch.equal(rows[:, :dim].float().cpu(), table.float().cpu()[toks.cpu().long()])
    assert bool((rows[:, dim:] == 5.0).all())


@pytest.mark.parametrize("dtype", [torch.float32, BF])
def test_a_table_that_begins_off_16_bytes(dtype):
    from allpaca_amd.kernels import ops
    from allpaca_amd.kernels.packing import PackedWeight
    table = gen(37, 264, seed=3, dtype=BF).to(DEV)
    tiles = pack(table)
    room = torch.zeros(tiles.data.numel() + 8, dtype=BF, device=DEV)
    moved = room[1:1 + tiles.data.numel()].view(tiles.data.shape)
    moved.copy_(tiles.data)
    toks = torch.tensor([36, 0, 15, 16, 31, 36, 5], dtype=torch.int32, device=DEV)
    rows = torch.empty(7, 264, dtype=dtype, device=DEV)
    ops.embed_rows(PackedWeight(moved, *[getattr(tiles, n) for n in ("N", "K")]), toks, rows)
    assert torch.equal(rows.float().cpu(), table.float().cpu()[toks.cpu().long()])
