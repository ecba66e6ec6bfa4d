"""The float32 kernel of both feed-forward products and their activation against the product of 2 F outputs and the
activation's own pass: the same sums in the same order, so the same bits; sizes on both sides of its tiles, few and many
rows, widths of K that leave waves without work, strided rows."""
import pytest
import torch

from test_kernels_tuned import DEV, gen

SIZES = [(1, 1, 4), (1, 16, 32), (4, 1000, 260), (4, 8192, 2048), (16, 17, 512), (17, 8200, 64), (40, 2048, 1028), (49, 4095, 96),
         (130, 1024, 288), (340, 8192, 512), (700, 9000, 36), (509, 2045, 132), (49, 4095, 132), (49, 100, 36), (700, 9000, 100),
         (30, 3000, 132), (1, 40, 100)]


def test_the_sizes_reach_every_tile():
    from allpaca_amd.kernels import lib
    L = lib.load("plain")
    for slices, tiles in ((lambda k: k > 128, {16016, 32016, 48016, 48032, 64032}),
                          (lambda k: 64 < k <= 128, {16016, 32016, 48016}), (lambda k: k <= 64, {16016, 32016, 48016})):
        assert {L.apc_swiglu_f32_tile(*s) for s in SIZES if slices(s[2])} >= tiles


@pytest.mark.gpu
@pytest.mark.parametrize("M,F,K", SIZES)
@pytest.mark.parametrize("pad", [0, 4])
def test_both_products_and_the_activation(M, F, K, pad):
    from allpaca_amd.kernels import ops
    h, w = gen(M, K + pad, seed=M).to(DEV)[:, :K], gen(2 * F, K + pad, seed=F, scale=2.0 * K ** -0.5).to(DEV)[:, :K]
    out = torch.full((M, F + pad), 7.0, device=DEV)
    assert ops._swiglu_f32(h, w, out[:, :F])
    both, want = torch.empty(M, 2 * F, device=DEV), torch.empty(M, F, device=DEV)
    ops.gemm_plain(h, w, both)
    ops.silu_mul(both, want)
    assert torch.equal(out[:, :F], want)
    assert bool((out[:, F:] == 7.0).all())


MORE_TILES = [(700, 9000, 132), (331, 9001, 256), (517, 2045, 388), (464, 2045, 520), (888, 1001, 580)]


def test_the_sizes_of_more_tiles_than_units_make_blocks_go_on():
    from allpaca_amd.kernels import lib
    L = lib.load("plain")
    assert all(L.apc_swiglu_f32_tiles_a_block(*s) > 1 for s in MORE_TILES)
    assert {L.apc_swiglu_f32_tile(*s) for s in MORE_TILES} == {48032, 64032}


@pytest.mark.gpu
@pytest.mark.parametrize("M,F,K", MORE_TILES + [(200, 8200, 520)])
def test_both_products_of_more_tiles_than_units(M, F, K):
    test_both_products_and_the_activation(M, F, K, 0)


@pytest.mark.gpu
def test_rows_that_are_no_pieces_of_16_bytes_are_left_alone():
    from allpaca_amd.kernels import ops
    h, w = gen(4, 63).to(DEV), gen(48, 63).to(DEV)
    out = torch.full((4, 24), 7.0, device=DEV)
    assert not ops._swiglu_f32(h, w, out)
    assert bool((out == 7.0).all())
    ops.swiglu(h, w, out)
    h, w, out = h.double().cpu(), w.double().cpu(), out.double().cpu()
    z, dz = h @ w.T, 64 * 2.0 ** -24 * (h.abs() @ w.abs().T)      # a sum of 63 float32 products
    g, u = z[:, :24], z[:, 24:]
    want = torch.nn.functional.silu(g) * u
    # |silu'| <= 1.1, and a handful of roundings of the activation itself
    bound = 1.1 * dz[:, :24] * u.abs() + torch.nn.functional.silu(g).abs() * dz[:, 24:] + 2.0 ** -20 * want.abs() + 1e-6
    assert bool(((out - want).abs() <= bound).all())
