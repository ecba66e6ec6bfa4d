"""Rows whose top-k keeps at most 1,024 candidates, chosen in two launches: every token is the one that the kernel of one
block a row gives, which walks the same candidates in the same order with the same float32 sums."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def both_ways(logits, temperature, top_k, top_p, uniform):
    from allpaca_amd.kernels import ops
    R = logits.shape[0]
    f = lambda x, dt: torch.tensor(np.broadcast_to(np.asarray(x), R).copy(), dtype=dt, device=DEV)  # noqa: E731
    args = (f(temperature, torch.float32), f(top_k, torch.int32), f(top_p, torch.float32), f(uniform, torch.float32))
    got, want = (torch.full((R,), -7, dtype=torch.int32, device=DEV) for _ in range(2))
    ops.sample_rows(logits, *args, got, few_after_top_k=True)
    ops.sample_rows(logits, *args, want, one_block=True)
    return got.tolist(), want.tolist()


# vocabularies of one piece, of ragged pieces, of rows that start off 16 bytes; rows with many and with few pieces
@pytest.mark.parametrize("V,R", [(7, 3), (1003, 5), (4099, 9), (32001, 70), (128256, 8), (60000, 600)])
def test_random_rows(V, R):
    g = torch.Generator(device=DEV).manual_seed(V)
    rng = np.random.default_rng(V)
    logits = torch.randn(R, V, generator=g, device=DEV) * 3
    for top_k in (1, 40, 63, 64, 65, 1024):
        for top_p in (0.0, 0.5, 0.95, 1.0):
            if V >= 32001 and (top_k, top_p) not in ((1, 0.95), (40, 0.95), (64, 0.5), (65, 1.0), (1024, 0.95)):
                continue                                     # (a row of one block takes milliseconds there)
            got, want = both_ways(logits, 0.8, top_k, top_p, rng.random(R))
            assert got == want, (top_k, top_p)


@pytest.mark.parametrize("V", [513, 9001])
def test_equal_values_infinities_and_masked_rows(V):
    rng = np.random.default_rng(1)
    rows = [np.full(V, 1.5), np.round(rng.normal(size=V)), np.full(V, -np.inf), np.full(V, np.nan), rng.normal(size=V),
            rng.normal(size=V), rng.normal(size=V), np.where(np.arange(V) % 2, 0.0, -0.0), rng.normal(size=V) * 1e-30,
            rng.normal(size=V) * 1e30]
    rows[1][::3] = -0.0
    rows[4][rng.random(V) < 0.98] = -np.inf                  # fewer candidates than top-k keeps
    rows[5][[3, 77]] = np.inf
    rows[6][:] = -np.inf
    rows[6][[5, 500]] = 2.0, 2.0
    logits = torch.tensor(np.stack(rows), dtype=torch.float32, device=DEV)
    for top_k in (1, 40, 300, 1024):
        for top_p in (0.3, 0.95, 1.0):
            for u in (0.0, 0.37, 0.999999):
                got, want = both_ways(logits, 0.7, top_k, top_p, u)
                assert got == want, (top_k, top_p, u)


def test_greedy_rows_and_rows_the_callers_word_was_wrong_about():
    g = torch.Generator(device=DEV).manual_seed(5)
    logits = torch.randn(6, 20000, generator=g, device=DEV)
    logits[1, 19999] = logits[1, 44] = 50.0                  # greedy: the first of two maxima
    rng = np.random.default_rng(2)
    got, want = both_ways(logits, [0.8, 0.0, 1.3, 1e-6, 0.5, 0.9], [40, 0, 0, 7, 3000, 40], [0.9, 0.9, 0.9, 1.0, 0.9, 1.0], rng.random(6))
    assert got == want and got[1] == 44
    # a view of a wider matrix whose rows start off 16 bytes
    wide = torch.randn(6, 20003, generator=g, device=DEV)
    got, want = both_ways(wide[:, 1:20002], 0.8, 40, 0.95, rng.random(6))
    assert got == want


# options on the host, with the launch: every rule, one row, the most rows that go that way and one more, rows of unlike
# rules, a greedy row among others, numbers of tokens and seeds at the ends of their ranges
@pytest.mark.parametrize("R,V", [(1, 4099), (8, 32001), (64, 9001), (65, 5000)])
@pytest.mark.parametrize("rule", [(0.8, 40, 0.95), (0.7, 0, 0.9), (0.8, 0, 1.0), (1.1, 2000, 0.5), None])
def test_options_that_go_with_the_launch(R, V, rule, monkeypatch):
    from allpaca_amd.kernels import ops
    from allpaca_amd.sampling import GenerationParams
    from allpaca_amd.sampling.sampler import Sampler, uniforms_for
    logits = torch.randn(R, V, generator=torch.Generator(device=DEV).manual_seed(R), device=DEV) * 3
    rules = [rule or [(0.0, 0, 1.0), (0.8, 40, 0.95), (1.0, 0, 1.0), (0.6, 1, 0.3), (0.9, 0, 0.7)][r % 5] for r in range(R)]
    seeds = [(1 << 64) - 1 if r == 0 else None if r == 1 else 977 * r for r in range(R)]
    numbers = [(1 << 40) * (r % 2) + r for r in range(R)]
    params = [GenerationParams(temperature=t, top_k=k, top_p=p, seed=s) for (t, k, p), s in zip(rules, seeds)]
    f = lambda x, dt: torch.tensor(x, dtype=dt, device=DEV)  # noqa: E731
    want = torch.empty(R, dtype=torch.int32, device=DEV)
    ops.sample_rows(logits, f([t for t, _, _ in rules], torch.float32), f([k for _, k, _ in rules], torch.int32), f([p for _, _, p in rules], torch.float32),
                    torch.from_numpy(uniforms_for([5 if s is None else s for s in seeds], numbers)).to(DEV), want, one_block=True)
    sampler, sample_rows, went = Sampler(torch.device(DEV), 5), ops.sample_rows, []

    def seen(logits, temperature, *a, **kw):
        done = sample_rows(logits, temperature, *a, **kw)
        went.append((isinstance(temperature, list), done is not None))
        return done

    monkeypatch.setattr(ops, "sample_rows", seen)
    for _ in range(3):                                       # (both of the sampler's result buffers)
        pending = sampler.launch(logits, params, numbers)
        assert pending.wait() == want.tolist() == pending.device.tolist()
    by_value = R <= 64                                       # options with the launch, ids from the kernel to the host
    assert went == ([] if rule is None and R == 1 else [(by_value, by_value)] * 3)       # (one greedy row: no sampling)


def test_options_that_only_the_copy_to_the_device_takes():
    """A top-k that is a float and numbers of tokens beyond a signed 64-bit one, beside the same choice with the launch."""
    from allpaca_amd.sampling import GenerationParams
    from allpaca_amd.sampling.sampler import Sampler
    logits = torch.randn(3, 5000, generator=torch.Generator(device=DEV).manual_seed(3), device=DEV) * 3
    params = lambda k: [GenerationParams(temperature=0.9, top_k=k, top_p=0.95, seed=r) for r in range(3)]  # noqa: E731
    s = Sampler(torch.device(DEV), 5)
    assert s.sample(logits, params(40.0), [4, 5, 6]) == s.sample(logits, params(40), [4, 5, 6])
    assert s.sample(logits, params(40.7), [4.0, 5, 6]) == s.sample(logits, params(40), [4, 5, 6])
    top = (1 << 64) - 2
    ids = s.sample(logits, params(40), [top, 1 << 63, 0])
    assert ids[2] == s.sample(logits, params(40), [1, 2, 0])[2] and all(0 <= t < 5000 for t in ids)


def test_a_result_that_is_dropped_keeps_its_memory_until_the_kernel_is_through():
    """The memory of a dropped result is nobody else's while the kernel that writes it is behind other work."""
    from allpaca_amd.kernels import ops
    from allpaca_amd.sampling import GenerationParams
    from allpaca_amd.sampling.sampler import Sampler
    torch.cuda.synchronize()
    ops.PinnedIds(1)                                         # (what earlier tests left is taken back)
    held = len(ops._still_written)
    logits = torch.randn(4, 32000, device=DEV)
    a = torch.randn(8192, 8192, device=DEV)
    params = [GenerationParams(temperature=0.8, top_k=40, top_p=0.95, seed=r) for r in range(4)]
    sampler = Sampler(torch.device(DEV), 5)
    want = sampler.sample(logits, params, [0] * 4)           # (both buffers have been pinned and the kernels loaded)
    assert sampler.sample(logits, params, [0] * 4) == want
    for _ in range(8):
        a @ a
    pending = sampler.launch(logits, params, [0] * 4)
    memory, device = pending.pinned, pending.device
    addresses = {p.address for p in sampler._pinned}
    del pending, sampler
    assert len(ops._still_written) == held + 2 and {m.data_ptr() for m, _ in list(ops._still_written)[held:]} == addresses
    del memory
    new = torch.empty(64, dtype=torch.int32).pin_memory()
    assert new.data_ptr() not in addresses
    torch.cuda.synchronize()
    assert device.tolist() == want and list(ops._still_written)[-1][1][-1].query()
    ops.PinnedIds(1)
    assert len(ops._still_written) == 0


def with_the_launch(logits, temperature, top_k, top_p):
    """(ids by options that go with the launch, ids of the kernel of one block a row)"""
    from allpaca_amd.kernels import ops
    from allpaca_amd.sampling.sampler import uniforms_for
    R = logits.shape[0]
    temps, ks, tops = ([x] * R if np.isscalar(x) else list(x) for x in (temperature, top_k, top_p))
    seeds, numbers = [31 * r + top_k if np.isscalar(top_k) else r for r in range(R)], list(range(R))
    f = lambda x, dt: torch.tensor(x, dtype=dt, device=DEV)  # noqa: E731
    got, want = (torch.full((R,), -7, dtype=torch.int32, device=DEV) for _ in range(2))
    ops.sample_rows(logits, temps, ks, tops, (seeds, numbers), got, few_after_top_k=True)
    ops.sample_rows(logits, f(temps, torch.float32), f(ks, torch.int32), f(tops, torch.float32),
                    torch.from_numpy(uniforms_for(seeds, numbers)).to(DEV), want, one_block=True)
    return got.tolist(), want.tolist()


# the bound from waves' largest values: sets of 48 to 256 waves and of fours of waves; the largest top-k that they take and the next; pieces of
# several rounds (64 rows) and a ragged last one; rows that start off 16 bytes
@pytest.mark.parametrize("V,R", [(12289, 3), (32001, 8), (65536, 1), (128256, 16), (128255, 8), (60001, 64)])
def test_top_k_bounded_by_the_largest_values_of_groups(V, R):
    logits = torch.randn(R, V + 3, generator=torch.Generator(device=DEV).manual_seed(V), device=DEV) * 3
    for view in (logits[:, :V], logits[:, 1:V + 1]):
        for top_k in (1, 31, 32, 40, 85, 86):
            got, want = with_the_launch(view, 0.8, top_k, 0.95)
            assert got == want, top_k


@pytest.mark.parametrize("V", [20000, 70001])
def test_groups_of_unlike_and_of_like_values(V):
    """All large values in one group, equal values, values in order, few that are finite: more than the block holds stand at the bound."""
    rng = np.random.default_rng(3)
    rows = [np.full(V, 1.5), np.round(rng.normal(size=V)), np.sort(rng.normal(size=V)), -np.sort(rng.normal(size=V)), np.full(V, -np.inf),
            np.full(V, np.nan), rng.normal(size=V), np.where(np.arange(V) % 2, 0.0, -0.0), rng.normal(size=V) * 1e-38, rng.normal(size=V) * 1e38,
            np.full(V, -np.inf), np.full(V, -np.inf), rng.normal(size=V)]
    rows[1][::3] = -0.0
    rows[3][700:] = -np.inf
    rows[6][[3, 77]] = np.inf
    rows[10][[5, V - 1]] = 2.0, 2.0
    rows[11][np.arange(0, V, V // 30)] = rng.normal(size=np.arange(0, V, V // 30).size)
    rows[12][4096:4096 + 900] += 20.0                        # 900 values far above all others
    logits = torch.tensor(np.stack(rows), dtype=torch.float32, device=DEV)
    for top_k in (1, 40):
        for top_p in (0.3, 0.95, 1.0):
            got, want = with_the_launch(logits, 0.7, top_k, top_p)
            assert got == want, (top_k, top_p)
    got, want = with_the_launch(logits, [0.7, 0.0, 1e-6] * 4 + [1.5], [40, 7, 0] * 4 + [3], [0.9, 1.0, 0.5] * 4 + [0.4])
    assert got == want


@pytest.mark.parametrize("V,R,most", [(12289, 3, 42), (32001, 8, 85), (65536, 1, 170), (128256, 16, 85), (128255, 8, 85), (60001, 64, 85), (128256, 32, 170), (128256, 24, 58)])
def test_top_k_up_to_which_rows_are_bounded_by_groups(V, R, most):
    """Which pair of launches a call takes, and the same tokens at the largest top-k of either."""
    from allpaca_amd.kernels import lib
    L = lib.load("plain")
    assert L.apc_sample_rows_bounded(R, V, most) == 1 and L.apc_sample_rows_bounded(R, V, most + 1) == 0
    assert L.apc_sample_rows_bounded(R, V, 0) == 0 and L.apc_sample_rows_bounded(65, V, 1) == 0
    logits = torch.randn(R, V, generator=torch.Generator(device=DEV).manual_seed(R), device=DEV) * 3
    logits[0] = logits[0].sort(descending=True).values       # large values side by side: more than the block holds
    logits[R // 2, :900] += 25.0
    logits[-1] = logits[-1].round() / 2
    for top_k in (most // 2, most, most + 1):
        got, want = with_the_launch(logits, 0.8, top_k, 0.95)
        assert got == want, top_k


@pytest.mark.parametrize("temperature", [1.1e-5, 0.5, 3.0, 1e4])
def test_bounds_at_the_ends_of_float32(temperature):
    """Quotients that overflow (all infinite, told apart by their ids), that vanish, and values next to the bound."""
    rng = np.random.default_rng(7)
    V = 40000
    near = np.float32(2.0) + np.float32(2.0 ** -22) * rng.integers(0, 40, size=V).astype(np.float32)      # neighbours that a division may round together
    rows = [rng.normal(size=V) * 1e38, rng.normal(size=V) * 1e34, -np.abs(rng.normal(size=V)) * 3e38, rng.normal(size=V) * 1e-44, rng.normal(size=V) * 1e-36, near, -near,
            np.where(rng.random(V) < 0.01, 3.4028e38, rng.normal(size=V))]
    logits = torch.tensor(np.clip(np.stack(rows), -3.4028234e38, 3.4028234e38), dtype=torch.float32, device=DEV)
    for top_k in (1, 40, 85):
        got, want = with_the_launch(logits, temperature, top_k, 0.9)
        assert got == want, top_k


def test_rows_of_equal_values_take_no_multiple_of_random_ones():
    """A row with more values at the bound than a block holds: some 2.5 times as long as random logits, and not 30."""
    from allpaca_amd.kernels import ops
    out = torch.zeros(8, dtype=torch.int32, device=DEV)

    def us(logits):
        least = 1e9
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                ops.sample_rows(logits, [0.8] * 8, [40] * 8, [0.95] * 8, (list(range(8)), [0] * 8), out, few_after_top_k=True)
            b.record()
            b.synchronize()
            least = min(least, a.elapsed_time(b) * 100.0)
        return least

    random = us(torch.randn(8, 128256, device=DEV) * 3)
    for like in (torch.zeros(8, 128256, device=DEV), torch.full((8, 128256), -1.7, device=DEV)):
        assert us(like) < 8 * random
