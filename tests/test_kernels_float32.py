"""The float32 products on the matrix cores and the float32 attention in 16-byte pieces, each at the edges of its tiles
against float64, and a row of a batch against the row alone, bit for bit."""
import math

import numpy as np
import pytest
import torch

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
# widths with whole and ragged stages of 32 and slices with 0, 1, 2, several of them; widths of two, of four and of eight
# slices at the tiles that leave the empty ones out
SIZES = [(1, 16, 4), (3, 70, 36), (16, 515, 256), (17, 33, 260), (8, 2048, 2048), (24, 16384, 96), (100, 2041, 388),
         (160, 2048, 1028), (331, 2045, 516), (480, 2050, 320), (33, 100, 8192), (509, 2045, 324), (509, 2045, 4), (331, 2047, 32),
         (509, 4101, 36), (331, 2045, 64), (500, 4090, 68), (331, 2045, 128), (700, 4099, 128), (331, 2045, 132), (20, 130, 100)]


def test_the_sizes_reach_every_tile():
    from allpaca_amd.kernels import lib
    L = lib.load("plain")
    for slices, tiles in ((lambda k: k > 128, {16016, 32016, 32032, 48032, 48064, 64064}),
                          (lambda k: 64 < k <= 128, {16016, 32032, 48032}), (lambda k: k <= 64, {16016, 32032, 48032})):
        assert {L.apc_gemm_f32_tile(*s) for s in SIZES if slices(s[2])} >= tiles


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SIZES)
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


# more tiles than compute units, on every tile whose blocks go on: a block's second and third tile, with slices of no, one, two
# and several stages, tiles that a block has one more of than its neighbour, and outputs that are added to
MORE_TILES = [(700, 4099, 132), (700, 4099, 256), (331, 6145, 300), (720, 3100, 580), (1030, 2045, 776), (517, 2045, 132), (1047, 1001, 520),
              (305, 6145, 520), (623, 3100, 776)]


def test_the_sizes_of_more_tiles_than_units_make_blocks_go_on():
    from allpaca_amd.kernels import lib
    L = lib.load("plain")
    assert all(L.apc_gemm_f32_tiles_a_block(*s) > 1 for s in MORE_TILES)
    assert {L.apc_gemm_f32_tile(*s) for s in MORE_TILES} == {48032, 48064, 64064}
    # (a row behind a norm among them: the form with the rows' scales goes on alike)
    assert L.apc_gemm_f32_tiles_a_block(700, 4099, 256) > 1 and L.apc_gemm_f32_tiles_a_block(16, 128256, 2048) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", MORE_TILES + [(490, 3100, 580)])
def test_product_of_more_tiles_than_units(M, N, K):
    test_product_against_64_bits_and_rows_alone(M, N, K)
    a, w = gen(M, K, seed=3), gen(N, K, seed=4)
    out, added = torch.empty(M, N, device=DEV), torch.ones(M, N, device=DEV)
    ops().gemm_plain(a, w, out)
    ops().gemm_plain(a, w, added, accumulate=True)
    assert torch.equal(added, out + 1.0)


@pytest.mark.gpu
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


@pytest.mark.gpu
def test_product_lets_infinities_and_nan_through():
    o = ops()
    a, w = gen(5, 36, seed=6), gen(20, 36, seed=7)
    a[1, 35], a[3, 0], w[19, 3] = math.inf, math.nan, -math.inf
    out = torch.empty(5, 20, device=DEV)
    o.gemm_plain(a, w, out)
    want = a.double() @ w.double().T
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())


def paged(lengths, Hk, d, P, seed):
    """A cache with the keys and values of several sequences on shuffled pages, NaN in every slot without a key."""
    g = torch.Generator().manual_seed(seed)
    blocks = [-(-n // P) for n in lengths]
    order = torch.randperm(sum(blocks) + 2, generator=g)
    cache = torch.full((len(order), 2, Hk, P, d), math.nan, device=DEV)
    values = cache[:, 1].view(-1, Hk, d, P)
    table = torch.zeros(len(lengths), max(blocks), dtype=torch.int32)
    kv, at = [], 0
    for i, n in enumerate(lengths):
        k, v = gen(n, Hk, d, seed=seed + 2 * i), gen(n, Hk, d, seed=seed + 2 * i + 1)
        for b in range(blocks[i]):
            page, m = int(order[at + b]), min(P, n - b * P)
            table[i, b] = page
            cache[page, 0, :, :m] = k[b * P:b * P + m].transpose(0, 1)
            values[page, :, :, :m] = v[b * P:b * P + m].permute(1, 2, 0)
        at += blocks[i]
        kv.append((k.double(), v.double()))
    return cache, table.to(DEV), kv


# groups of 4, 2, 1 heads on a kv head (and 3, taken one by one); heads up to 64 and up to 128; pages under, at and over
# a chunk of 64 keys; lengths around a chunk and around eight of them
@pytest.mark.gpu
@pytest.mark.parametrize("H,Hk,d,P", [(8, 2, 64, 16), (6, 2, 32, 4), (4, 2, 128, 16), (3, 1, 100, 8), (4, 1, 80, 128)])
@pytest.mark.parametrize("window", [0, 70])
def test_attention_against_64_bits_and_rows_alone(H, Hk, d, P, window):
    o = ops()
    lengths = [577, 1, 63, 64, 65]
    cache, table, kv = paged(lengths, Hk, d, P, seed=11)
    pos = torch.tensor([p for n in lengths for p in range(n)], dtype=torch.int32, device=DEV)
    seg = torch.tensor([i for i, n in enumerate(lengths) for _ in range(n)], dtype=torch.int32, device=DEV)
    q = gen(len(pos), 8 + H * d, seed=5)
    out = torch.empty(len(pos), H * d, device=DEV)                    # (enough rows for the form of a row a wave)
    o.paged_attention_plain(q, 8, out, H, Hk, d, cache, P, table, pos, seg, window=window)
    for r in [0, 62, 63, 64, 69, 70, 511, 512, 576, 577, 578, 640, 641, 704, 705, len(pos) - 1]:
        alone = torch.empty(1, H * d, device=DEV)                     # (a block a row)
        o.paged_attention_plain(q[r:r + 1], 8, alone, H, Hk, d, cache, P, table, pos[r:r + 1], seg[r:r + 1], window=window)
        assert torch.equal(alone[0], out[r])
        p, (k, v) = int(pos[r]), kv[int(seg[r])]
        first = max(0, p - window + 1) if window else 0
        k, v = (x[first:p + 1].repeat_interleave(H // Hk, 1) for x in (k, v))
        qr = q[r, 8:].double().view(H, d)
        s = torch.einsum("hd,thd->ht", qr, k) / math.sqrt(d)
        want = torch.einsum("ht,thd->hd", s.softmax(-1), v)
        # a score is off by at most (d + 2) U of the sum of its products' magnitudes, a weight by twice that relatively
        # and by the exponential's few U, a sum of n weights and products by n + 16 U
        most = float((torch.einsum("hd,thd->ht", qr.abs(), k.abs()) / math.sqrt(d)).max())
        bound = (2 * (d + 2) * most + 2 * (p + 1 - first + 16) + 16) * U * float(v.abs().max())
        assert float((out[r].double().view(H, d) - want).abs().max()) <= bound


# the norm in the product (up to 16 rows of up to 4,096) and in front of it: both against float64, a row of a batch against
# the row alone bit for bit across that line, rows with more elements than they are used with, several tiles a block
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 16, 4), (4, 70, 36), (16, 515, 256), (17, 130, 260), (8, 3072, 2048), (33, 100, 4096),
                                   (5, 48, 4100), (331, 2045, 516), (700, 4099, 256), (20, 8200, 388)])
@pytest.mark.parametrize("gated", [False, True])
def test_product_of_normalised_rows(M, N, K, gated):
    o = ops()
    x, g, w = gen(M, K + 4, seed=1)[:, :K] * 3.0, 1.0 + 0.1 * gen(K, seed=2), gen(N * (2 if gated else 1), K, seed=3) * 2 * K ** -0.5
    x[M // 2] *= 1e-3
    eps = 1e-5
    fn = o.swiglu_normed if gated else o.linear_normed
    out = torch.full((M, N + 4), 7.0, device=DEV)
    assert fn(x, g, eps, w, out[:, :N])
    assert (out[:, N:] == 7.0).all()
    h = x.double() * torch.rsqrt(x.double().square().mean(1, keepdim=True) + eps) * g.double()
    y = h @ w.double().T
    # beside the product's own bound: the rounded x * g, the sum of squares, the root and the last product
    bound = product_bound(h, w) + (K / 16 + 16) * U * (h.abs() @ w.double().abs().T)
    if gated:
        s, u = y[:, :N], y[:, N:]
        want = torch.nn.functional.silu(s) * u
        # silu' is at most 1.1; its own rounding and that of the product
        bound = 1.1 * bound[:, :N] * u.abs() + bound[:, N:] * torch.nn.functional.silu(s).abs() + 1.1 * bound[:, :N] * bound[:, N:] + 8 * U * want.abs()
    else:
        want = y
    assert ((out[:, :N].double() - want).abs() <= bound).all()
    for r in sorted({0, M // 2, M - 1}):
        alone = torch.empty(1, N, device=DEV)
        assert fn(x[r:r + 1], g, eps, w, alone)
        assert torch.equal(alone[0], out[r, :N])


def test_tiles_of_few_rows():
    """Up to 16 rows take the tile of 16 rows, but for many outputs of a K up to 128, where tiles that leave the empty slices
    out are faster."""
    from allpaca_amd.kernels import lib
    L = lib.load("plain")
    for M in (1, 9, 16):
        for K in (32, 64, 128):
            assert L.apc_gemm_f32_tile(M, 2048, K) == 16016 and L.apc_gemm_f32_tile(M, 128256, K) == 32032, (M, K)
        for K in (132, 2048, 8192):
            assert {L.apc_gemm_f32_tile(M, N, K) for N in (16, 2048, 128256)} == {16016}, (M, K)


# few rows of a K up to 128: two and four slices, and 16 rows of eight, with the norm in the product and in front of it
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(16, 40003, 32), (3, 33000, 64), (9, 50010, 100), (1, 128256, 128), (40, 300, 128), (33, 100, 64)])
def test_few_rows_of_a_short_k(M, N, K):
    test_product_against_64_bits_and_rows_alone(M, N, K)
    for gated in (False, True):
        test_product_of_normalised_rows(M, N // 2 if gated else N, K, gated)
    o, x, g, w = ops(), gen(M, K, seed=1), 1.0 + 0.1 * gen(K, seed=2), gen(N, K, seed=3)
    many, few = torch.empty(M, N, device=DEV), torch.empty(M, 48, device=DEV)
    assert o.linear_normed(x, g, 1e-5, w, many) and o.linear_normed(x, g, 1e-5, w[:48], few)
    assert torch.equal(many[:, :48], few)                  # (48 outputs: the norm in the product up to 16 rows)


# where the norm stands: in the product, or in front of it (many outputs of a K up to 1,024) by two rows a wave or a row a block
# (rows of more than 512 numbers; of more than 4,096 for however many rows), whose last pass of a slice is whole or not
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(3, 32776, 300), (2, 16400, 1024), (16, 16384, 516), (1, 32776, 1028), (17, 40, 508), (17, 40, 516), (512, 40, 1156),
                                   (513, 40, 1156), (600, 24, 4100), (3, 40, 8196), (40, 24, 16388)])
def test_rows_behind_a_norm_in_every_form(M, N, K):
    o, eps = ops(), 1e-5
    x, g, w = gen(M, K, seed=1) * 2.0, 1.0 + 0.1 * gen(K, seed=2), gen(N, K, seed=3) * 2 * K ** -0.5
    out, few = torch.empty(M, N, device=DEV), torch.empty(M, 24, device=DEV)
    assert o.linear_normed(x, g, eps, w, out) and o.linear_normed(x, g, eps, w[:24].contiguous(), few)
    h = x.double() * torch.rsqrt(x.double().square().mean(1, keepdim=True) + eps) * g.double()
    bound = product_bound(h, w) + (K / 16 + 16) * U * (h.abs() @ w.double().abs().T)
    assert ((out.double() - h @ w.double().T).abs() <= bound).all()
    assert torch.equal(out[:, :24], few)
    for r in sorted({0, M // 2, M - 1}):
        alone = torch.empty(1, N, device=DEV)
        assert o.linear_normed(x[r:r + 1], g, eps, w, alone)
        assert torch.equal(alone[0], out[r])


# blocks of 8 outputs (up to 2,048) and tiles beyond, last blocks that are not full; slices with no, one and several stages, a last stage cut
# by K; outputs whose rows do not allow 16-byte stores
@pytest.mark.gpu
@pytest.mark.parametrize("N,K", [(8, 132), (40, 14340), (515, 256), (2048, 2048), (2047, 388), (2049, 1028), (4090, 2052), (4096, 1056), (1001, 132), (2040, 1024)])
def test_up_to_8_rows_are_the_bits_of_more(N, K):
    o = ops()
    a, w = gen(12, K, seed=1), gen(N, K, seed=2)
    many = torch.empty(12, N, device=DEV)
    o.gemm_plain(a, w, many)
    assert ((many.double() - a.double() @ w.double().T).abs() <= product_bound(a, w)).all()
    for M in (1, 2, 5, 8):
        for ld in (N, N + 3):
            out = torch.full((M, ld), 7.0, device=DEV)
            o.gemm_plain(a[:M], w, out[:, :N])
            assert torch.equal(out[:, :N], many[:M]) and (out[:, N:] == 7.0).all()
            o.gemm_plain(a[:M], w, out[:, :N], accumulate=True)
            assert torch.equal(out[:, :N], many[:M] + many[:M]) and (out[:, N:] == 7.0).all()


@pytest.mark.parametrize("M,N,K,stored,added", [(1, 2048, 1028, 1, 1), (8, 2048, 2048, 1, 1), (8, 8, 14336, 1, 1), (4, 2048, 1024, 0, 1), (4, 576, 132, 0, 1),
                                                (4, 576, 128, 0, 0), (9, 2048, 2048, 0, 0), (4, 2049, 2048, 0, 0), (4, 4096, 4096, 0, 0)])
def test_products_that_the_kernel_of_up_to_8_rows_takes(M, N, K, stored, added):
    from allpaca_amd.kernels import lib
    few = lib.load("plain").apc_gemm_f32_few
    assert (few(M, N, K, 0), few(M, N, K, 1)) == (stored, added)


@pytest.mark.gpu
@pytest.mark.parametrize("M,H,Hk,d,K,P", [(1, 32, 8, 64, 2048, 16), (4, 32, 8, 64, 2048, 16), (8, 4, 2, 128, 4096, 8), (5, 3, 1, 16, 132, 4),
                                          (7, 6, 2, 80, 1000, 24), (3, 5, 5, 32, 260, 5)])
def test_q_k_v_rotated_and_in_the_pages_are_the_bits_of_the_kernels_one_after_the_other(M, H, Hk, d, K, P):
    o = ops()
    rng = np.random.default_rng(M * 100 + d)
    x, g, w = gen(M, K + 4, seed=1)[:, :K] * 3.0, 1.0 + 0.1 * gen(K, seed=2), gen((H + 2 * Hk) * d, K, seed=3)
    blocks = 6
    places = rng.permutation(3 * blocks * P)[:M]
    seg = torch.tensor(places // (blocks * P), dtype=torch.int32, device=DEV)
    pos = torch.tensor(places % (blocks * P), dtype=torch.int32, device=DEV)
    table = torch.from_numpy(rng.permutation(3 * blocks).reshape(3, blocks).astype(np.int32)).to(DEV)
    angles = torch.arange(blocks * P, dtype=torch.float64)[:, None] * 300.0 ** (-torch.arange(d // 2, dtype=torch.float64) / (d // 2))
    cos_sin = torch.stack([angles.cos(), angles.sin()], 1).float().to(DEV)
    got, want = (torch.full((M, (H + 2 * Hk) * d + 4), 7.0, device=DEV) for _ in range(2))
    pages_got, pages_want = (torch.zeros(3 * blocks, 2, Hk, P, d, device=DEV) for _ in range(2))
    assert o.qkv_rope_normed(x, g, 1e-5, w, got, H, Hk, d, cos_sin, pos, seg, table, pages_got, P)
    assert o.linear_normed(x, g, 1e-5, w, want[:, :-4])
    o.rope_kv_write(want, 0, H * d, (H + Hk) * d, H, Hk, d, d, cos_sin, pos, seg, table, pages_want, P)
    assert torch.equal(got[:, :H * d], want[:, :H * d]) and torch.equal(pages_got, pages_want)
    assert (got[:, H * d:] == 7.0).all()


@pytest.mark.gpu
def test_q_k_v_that_are_left_to_the_kernels_one_after_the_other():
    o = ops()

    def taken(M=4, H=4, Hk=2, d=32, K=256):
        x, w = gen(M, K), gen((H + 2 * Hk) * d, K)
        ints = [torch.zeros(n, dtype=torch.int32, device=DEV) for n in (M, M)]
        return o.qkv_rope_normed(x, gen(K), 1e-5, w, torch.empty(M, (H + 2 * Hk) * d, device=DEV), H, Hk, d, torch.zeros(64, 2, d // 2, device=DEV),
                                 *ints, torch.zeros(1, 4, dtype=torch.int32, device=DEV), torch.zeros(4, 2, Hk, 16, d, device=DEV), 16)

    assert taken()
    assert not taken(M=9) and not taken(d=24) and not taken(K=128) and not taken(K=4100) and not taken(H=300)
