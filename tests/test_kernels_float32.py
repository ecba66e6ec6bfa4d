"""The float32 products on the matrix cores and the float32 attention in 16-byte pieces, each at the edges of its tiles
against float64, and a row of a batch against the row alone, bit for bit."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
U = 2.0 ** -24


def ops():
    from allpaca_amd.kernels import ops as o
    return o


def gen(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


def product_bound(a, w):
    """A sum of at most K/8 + 32 rounded products and additions, then eight slices: each step is off by at most U of the
    sum of the magnitudes."""
    return (a.shape[1] / 8 + 32 + 8 + 1) * U * (a.double().abs() @ w.double().abs().T)


# rows and outputs of every tile's range (16 x 16, 32 x 16, 32 x 32, 48 x 32, 48 x 64, 64 x 64) and their remainders;
# widths with whole and ragged stages of 32 and slices with 0, 1, 2, several of them
@pytest.mark.parametrize("M,N,K", [(1, 16, 4), (3, 70, 36), (16, 515, 256), (17, 33, 260), (8, 2048, 2048), (24, 16384, 96),
                                   (100, 2041, 388), (160, 2048, 1028), (331, 2045, 516), (480, 2050, 320), (33, 100, 8192)])
def test_product_against_64_bits_and_rows_alone(M, N, K):
    o = ops()
    a, w = gen(M, K, seed=1), gen(N, K, seed=2)
    out = torch.empty(M, N, device=DEV)
    o.gemm_plain(a, w, out)
    want, bound = a.double() @ w.double().T, product_bound(a, w)
    assert ((out.double() - want).abs() <= bound).all()
    for r in sorted({0, M // 2, M - 1}):
        alone = torch.empty(1, N, device=DEV)
        o.gemm_plain(a[r:r + 1], w, alone)
        assert torch.equal(alone[0], out[r])
    add = gen(M, N, seed=3)
    both = add.clone()
    o.gemm_plain(a, w, both, accumulate=True)
    assert torch.equal(both, add + out)


def test_product_of_views_reads_nothing_past_their_width():
    """Rows of a wider matrix whose other columns hold NaN, outputs into a wider matrix, bfloat16 outputs."""
    o = ops()
    for K in (52, 64, 300):
        wide_a, wide_w = torch.full((37, 320), math.nan, device=DEV), torch.full((90, 320), math.nan, device=DEV)
        a, w = wide_a[:, :K], wide_w[:, :K]
        a.copy_(gen(37, K, seed=4)), w.copy_(gen(90, K, seed=5))
        wide = torch.full((37, 100), 7.0, device=DEV)
        o.gemm_plain(a, w, wide[:, :90])
        assert ((wide[:, :90].double() - a.double() @ w.double().T).abs() <= product_bound(a, w)).all()
        assert (wide[:, 90:] == 7.0).all()
        half = torch.empty(37, 90, dtype=torch.bfloat16, device=DEV)
        o.gemm_plain(a, w, half)
        assert torch.equal(half, wide[:, :90].to(torch.bfloat16))


def test_product_lets_infinities_and_nan_through():
    o = ops()
    a, w = gen(5, 36, seed=6), gen(20, 36, seed=7)
    a[1, 35], a[3, 0], w[19, 3] = math.inf, math.nan, -math.inf
    out = torch.empty(5, 20, device=DEV)
    o.gemm_plain(a, w, out)
    want = a.double() @ w.double().T
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
