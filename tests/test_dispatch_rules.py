"""Host-side rules that choose a kernel's shape from a step's sizes (no GPU): into how many ranges the keys of a tile
of prompt rows are cut, and which launches the sampler is told to leave out."""
from types import SimpleNamespace

import pytest


def _step(segments, tile=128):
    """A step of prompt portions: (position of the first row, rows) per segment."""
    n_tiles = sum(-(-n // tile) for _, n in segments if n > 1)
    return SimpleNamespace(n_tiles=n_tiles, host_pos0=[p for p, _ in segments], host_rows=[n for _, n in segments])


def test_key_ranges_of_a_step():
    from allpaca_amd.kernels import tuned
    ks = tuned._key_splits
    # a chunk of 512 rows at 32 heads is 128 blocks: cut in two from 4,096 keys on, never more (256 compute units)
    assert ks(_step([(0, 512)]), 32, 0) == 1
    assert ks(_step([(2048 - 512, 512)]), 32, 0) == 1
    assert ks(_step([(4096 - 512, 512)]), 32, 0) == 2
    assert ks(_step([(131072 - 512, 512)]), 32, 0) == 2
    # 128 rows are 32 blocks: ranges of 1,024 keys while the chip stays half empty, of 2,048 beyond, 8 at most
    assert [ks(_step([(n - 128, 128)]), 32, 0) for n in (1000, 2048, 3072, 4096, 8192, 16384, 65536)] == [1, 2, 3, 4, 4, 8, 8]
    # a whole-prompt step has blocks enough
    assert ks(_step([(0, 2048)]), 32, 0) == 1 and ks(_step([(30720, 2048)]), 32, 0) == 1
    # 64 heads: a chunk of 512 fills the chip by itself; 8 heads: 32 blocks
    assert ks(_step([(32768 - 512, 512)]), 64, 0) == 1
    assert ks(_step([(8192 - 512, 512)]), 8, 0) == 4
    # the longest prompt of the step counts, single rows (decoding requests) do not; a window bounds the keys
    assert ks(_step([(100, 128), (8000, 128), (50000, 1)]), 32, 0) == 3
    assert ks(_step([(50000, 1), (10, 128)]), 32, 0) == 1
    assert ks(_step([(32768 - 128, 128)]), 32, 1000) == 1
    assert ks(_step([(32768 - 128, 128)]), 32, 4096) == 4
    # nothing known of the step's positions: no cutting
    assert ks(SimpleNamespace(n_tiles=1), 32, 0) == 1


def test_key_ranges_can_be_switched_off(monkeypatch):
    from allpaca_amd.kernels import tuned
    monkeypatch.setattr(tuned, "KEY_SPLITS_MAX", 0)
    assert tuned._key_splits(_step([(32768 - 128, 128)]), 32, 0) == 1


@pytest.mark.parametrize("rules,want", [
    # (temperature, top-k, top-p) per row -> (some top-k, some top-p, few survivors everywhere)
    ([(0.8, 40, 0.95)], (True, True, True)),
    ([(0.8, 0, 1.0)], (False, False, False)),
    ([(0.8, 0, 0.9), (0.0, 0, 1.0)], (False, True, False)),
    ([(0.8, 40, 1.0), (0.0, 0, 1.0)], (True, False, True)),      # a greedy row needs no launch of its own
    ([(0.8, 2000, 1.0)], (True, False, False)),
    ([(0.8, 40, 0.95), (0.7, 0, 0.95)], (True, True, False)),
])
def test_what_the_sampler_tells_the_kernels(monkeypatch, rules, want):
    """`Sampler.launch` passes on which cuts its rows ask for, so that the kernels leave out the launches nobody needs."""
    import torch
    from allpaca_amd.kernels import ops
    from allpaca_amd.sampling import GenerationParams
    from allpaca_amd.sampling import sampler as S
    seen = {}

    def fake_sample_rows(logits, t, k, p, u, out, **kw):
        seen.update(kw)

    monkeypatch.setattr(ops, "sample_rows", fake_sample_rows)
    monkeypatch.setattr(S.Sampler, "_upload", lambda self, params, indices: torch.zeros(4, 64))
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda self: self)
    monkeypatch.setattr(torch.cuda, "Event", lambda *a, **k: SimpleNamespace(record=lambda: None, synchronize=lambda: None))
    s = S.Sampler(torch.device("cpu"), 0)
    params = [GenerationParams(max_tokens=1, temperature=t, top_k=k, top_p=p) for t, k, p in rules]
    s.launch(torch.zeros(len(rules), 16), params, [0] * len(rules))
    assert (seen["any_top_k"], seen["any_top_p"], seen["few_after_top_k"]) == want


@pytest.mark.parametrize("rows,k,number,by_value", [
    (2, 40, 7, True), (64, -1, 0, True), (65, 40, 7, False), (2, (1 << 31) - 1, (1 << 63) - 1, True),
    # what only the copy to the device takes: floats, numbers beyond a signed 64-bit one; and what it refuses
    (2, 40.0, 7, False), (2, 40, 7.0, False), (2, 40, 1 << 63, False), (2, 1 << 31, 7, False), (2, -(1 << 31) - 1, 7, False), (2, 40, -1, False)])
def test_options_of_few_rows_go_with_the_launch_if_its_types_hold_them(rows, k, number, by_value):
    import torch
    from allpaca_amd.kernels import ops
    from allpaca_amd.sampling.sampler import Sampler
    s = Sampler(torch.device("cuda"), 0)
    temps, tops, ks, numbers = [0.8] * rows, [0.95] * rows, [5] * (rows - 1) + [k], [3] * (rows - 1) + [number]
    assert s._by_value((rows, 32000), temps, ks, tops, numbers) == by_value
    assert not s._by_value((rows - 1, 32000), temps, ks, tops, numbers)          # (more options than rows)
    if by_value:
        ops._packed_options(rows).pack(*temps, *tops, *ks, *range(rows), *numbers)


def test_memory_that_a_queued_kernel_writes_is_kept_until_it_has(monkeypatch):
    """Token ids come back through pinned memory whose address a kernel gets.  Dropped with kernels queued, on two streams, the
    block is given back only when both are through."""
    import gc
    import weakref

    import torch
    from allpaca_amd.kernels import lib, ops
    kernels, through, stream = [], set(), [1]

    class Event:
        def record(self):
            self.kernel = len(kernels) - 1

        def query(self):
            return self.kernel in through

    L = SimpleNamespace(apc_sample_rows_scratch_kib=lambda n: 1, apc_sample_rows_host=lambda *a: kernels.append(a[6]) or 0)
    monkeypatch.setattr(lib, "load", lambda name: L)
    monkeypatch.setattr(ops, "_gpu", lambda *a: None)
    monkeypatch.setattr(ops, "_stream", lambda: stream[0])
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda self: self)
    monkeypatch.setattr(torch.cuda, "Event", Event)
    ids = ops.PinnedIds(64)
    tensor, address = weakref.ref(ids.tensor), ids.address

    def choose(on):
        stream[0] = on
        return ops.sample_rows(torch.zeros(2, 16), [0.8] * 2, [40] * 2, [0.9] * 2, ([1, 2], [0, 1]), torch.zeros(2, dtype=torch.int32), out_host=ids)

    events = [choose(1), choose(2), choose(2)]
    assert kernels == [address] * 3 and all(isinstance(e, Event) for e in events)
    del ids
    for done in ({2}, {0, 1}):
        gc.collect()
        through.clear()
        through.update(done)
        ops.PinnedIds(64)
        assert tensor() is not None and tensor().data_ptr() == address
    through.update({0, 2})
    ops.PinnedIds(64)
    gc.collect()
    assert tensor() is None


def test_memory_for_ids_is_pinned_by_threads_at_a_time_and_kept_by_an_event_that_raises(monkeypatch):
    import collections
    import torch
    from allpaca_amd.kernels import ops
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda self: self)
    waiting = collections.deque()
    monkeypatch.setattr(ops, "_still_written", waiting)

    class Emptied:                      # what a thread sees whose last entry another one has just taken
        def __len__(self):
            return 1

        def popleft(self):
            raise IndexError

    def refuses():
        raise RuntimeError("capturing")

    monkeypatch.setattr(ops, "_still_written", Emptied())
    assert ops.PinnedIds(4).size == 4
    monkeypatch.setattr(ops, "_still_written", waiting)
    entry = (torch.zeros(1), [SimpleNamespace(query=refuses)])
    waiting.append(entry)
    with pytest.raises(RuntimeError, match="capturing"):
        ops.PinnedIds(4)
    assert list(waiting) == [entry]


@pytest.mark.parametrize("Hk,d,page,takes", [(8, 128, 16, 1), (8, 64, 32768, 1), (255, 128, 32768, 1), (256, 128, 32768, 0), (511, 64, 32768, 1),
                                             (512, 64, 32768, 0), (2048, 128, 4096, 0), (8, 128, 65536, 0), (8, 128, 8, 0), (8, 96, 16, 0), (8, 64, 48, 0)])
def test_pages_that_the_attention_kernel_of_128_rows_takes(Hk, d, page, takes):
    """The question that room for ranges of keys hangs on is the dispatch's own: a page of 4 GiB goes to the narrower kernels."""
    from allpaca_amd.kernels import lib
    assert lib.load("tuned").apc_attention_prefill_wide_takes(Hk, d, page, 2, 256) == takes


@pytest.mark.parametrize("parts,one", [(64, True), (32, True), (16, True), (8, False), (1, False)])
def test_gated_recurrence_in_one_launch_for_parts_of_up_to_128_channels(monkeypatch, parts, one):
    """A block reads all gates of a part: of 256 channels three launches are faster (parts of 32 to 2,048 channels here)."""
    import torch
    from allpaca_amd.kernels import ops
    from allpaca_amd.parts.gated_recurrence import GatedRecurrence
    C, went = 2048, []
    monkeypatch.setattr(ops, "recurrent_step", lambda *a: went.append("one") or True)
    for name in ("conv_channels", "heads_linear", "gated_recurrence"):
        monkeypatch.setattr(ops, name, lambda *a, name=name, **kw: went.append(name))
    mixer = SimpleNamespace(C=C, B=parts, w=C // parts, rt=SimpleNamespace(dtype=torch.bfloat16),
                            **{n: None for n in ("x_b", "y_b", "conv_w", "conv_b", "w_gates", "gates_b", "rate")})
    view = SimpleNamespace(writes=True, state=None, slots=None)
    proj, out = torch.zeros(2, 2 * C, dtype=torch.bfloat16), torch.zeros(2, C, dtype=torch.bfloat16)
    GatedRecurrence.core(mixer, proj, None, {"mixer": view, "mixer.state": view}, out)
    assert went == (["one"] if one else ["conv_channels", "heads_linear", "gated_recurrence"])


def test_entry_points_that_launch_nothing_are_not_timed_as_kernels():
    """A kernel's last argument is its stream; what has none answers a question about sizes."""
    from allpaca_amd.kernels import lib
    asked = {n for group, entries in lib.SIGNATURES.items() if group != "host"
             for n, args in entries.items() if not args or args[-1] is not lib.P}
    assert "apc_swiglu_f32_takes" in asked and asked <= lib.NOT_KERNELS


def test_the_room_kept_out_of_the_cache_holds_the_samplers_scratch():
    from allpaca_amd.engine import Engine
    from allpaca_amd.kernels import lib
    L = lib.load("plain")
    model = SimpleNamespace(spec=SimpleNamespace(hidden_size=64, vocab_size=0), blocks=[])
    room = lambda n: Engine.reserve_bytes(model, SimpleNamespace(max_batch_tokens=8, max_active_requests=n))  # noqa: E731
    for rows in (1, 2, 7, 16, 17, 64, 300, 1024):
        assert room(rows) - room(0) >= 1024 * L.apc_sample_rows_scratch_kib(rows), rows


def test_ranges_the_decode_attention_cuts_a_rows_keys_into():
    """Four ranges a block, as many blocks a (row, kv head) pair as keep the launch within the chip's compute units,
    and no range under 64 keys."""
    from allpaca_amd.kernels import tuned as t
    got = {(n, ctx): t._decode_parts(n * 8, ctx) for n, ctx in
           [(1, 2048), (4, 2048), (8, 2048), (8, 2063), (12, 2048), (16, 2048), (24, 2048), (8, 8192), (16, 8192),
            (1, 32768), (8, 512), (1, 10), (40, 2048)]}
    assert got == {(1, 2048): 32, (4, 2048): 32, (8, 2048): 16, (8, 2063): 16, (12, 2048): 8, (16, 2048): 8,
                   (24, 2048): 4, (8, 8192): 16, (16, 8192): 8, (1, 32768): 128, (8, 512): 8, (1, 10): 1, (40, 2048): 4}
    for pairs in (1, 8, 64, 100, 255, 256, 1000):
        for span in (1, 64, 65, 2048, 1 << 20):
            parts = t._decode_parts(pairs, span)
            blocks = pairs * -(-parts // t.WHOLE_WAVES)
            assert parts >= 1 and (blocks <= max(pairs, t.CHIP_UNITS)) and (parts == 1 or span / parts >= 32)


def test_the_executors_rules_are_the_wrappers_rules():
    """The compiled plan executor (csrc/host/rules.h) chooses slices of K, keys a wave and ranges of keys by the same
    rules as the Python wrappers of the kernels: held against each other over the shapes either may meet."""
    from allpaca_amd.kernels import host, tuned
    L = host.load()
    for M in (17, 24, 32, 48, 64, 100, 128, 129, 200, 256, 384, 500, 512, 640, 768, 1000, 1024, 1025, 2048):
        for N in (192, 1000, 2048, 3072, 4096, 5120, 6144, 8192, 14336, 16384, 28672, 57344, 128256):
            for K in (120, 192, 512, 2048, 3072, 4096, 8192, 14336, 28672):
                assert L.apc_host_rule_tiled_k_split(M, N, K) == tuned._tiled_k_split(M, N, K), (M, N, K)
    for pairs in (1, 2, 3, 8, 12, 16, 24, 31, 64, 100, 255, 256, 257, 2040):
        for span in (1, 63, 64, 65, 2048, 2049, 8192, 32768, 131072):
            assert L.apc_host_rule_decode_parts(pairs, span) == tuned._decode_parts(pairs, span), (pairs, span)
    for rows in (2, 100, 128, 129, 256, 512, 1024, 2048):
        for pos0 in (0, 500, 1920, 3584, 8000, 32640, 130000):
            for heads in (4, 8, 24, 32, 64):
                for window in (0, 1000, 4096):
                    step = _step([(pos0, rows), (7, 1)])
                    want = tuned._key_splits(step, heads, window)
                    got = L.apc_host_rule_key_splits(step.n_tiles, heads, pos0 + rows, window, tuned.KEY_SPLITS_MAX,
                                                     tuned.KEY_RANGE_MIN)
                    assert got == want, (rows, pos0, heads, window)


@pytest.mark.parametrize("M,N,slices", [(896, 6144, 3), (384, 5120, 6), (300, 5120, 3), (300, 5120, 6), (896, 2048, 6), (512, 4096, 4),
                                        (512, 6144, 2), (1024, 8192, 4)])
def test_slices_without_weights_in_lds_fill_their_rounds_by_the_busiest_xcd(M, N, slices):
    """The tiles of a launch are dealt out to 8 XCDs of 32 compute units by eighths, all slices of a tile to one XCD: the
    bands a wave takes are not such that a round beyond the first serves a few blocks of one XCD."""
    from allpaca_amd.kernels import host
    bands = host.load().apc_host_rule_direct_bands(M, N, slices)
    busiest = -(-(-(-M // 128) * -(-N // (64 * bands))) // 8) * slices
    assert busiest / (32 * -(-busiest // 32)) >= 0.7, (bands, busiest)


@pytest.mark.parametrize("M,N,K,slices,direct", [
    # K without many divisors: as many slices as the 128 x 128 tile wants (measured: 33, 40, 48, 64 and 37 us; in the two
    # slices that the kernel without weights in LDS has 84, 68, 67, 72 and 67)
    (384, 640, 15104, 5, False), (500, 2048, 11008, 4, False), (384, 3072, 11008, 3, False), (384, 4096, 11008, 2, False), (384, 1280, 11008, 5, False),
    # slices on the kernel without weights in LDS
    (512, 4096, 14336, 4, True), (512, 6144, 4096, 2, True), (384, 3072, 8192, 4, True),
    # at 1,024 rows K in one piece is that kernel's too, and its time counts, not the tile's
    (1024, 5120, 3072, 1, False), (1024, 4096, 14336, 2, True),
    # below 257 rows, K no multiple of 128
    (256, 4096, 14336, 4, False), (300, 640, 1288, 5, False)])
def test_slices_of_k_for_some_hundred_rows(M, N, K, slices, direct):
    from allpaca_amd.kernels import tuned
    assert tuned._slices_many_rows(M, N, K) == (slices, direct)


def test_the_kernel_library_takes_the_slices_that_the_wrappers_mean_for_it():
    from allpaca_amd.kernels import host, tuned
    L = host.load()
    for M in (129, 200, 256, 257, 300, 384, 500, 512, 640, 768, 896, 1000, 1023, 1024):
        for N in (192, 640, 1000, 1002, 1920, 2048, 3072, 4096, 5120, 6144, 8192, 11008, 28672):
            for K in (128, 192, 512, 768, 1152, 1288, 2048, 3072, 4096, 5376, 8192, 11008, 14336, 15104):
                s, direct = tuned._slices_many_rows(M, N, K)
                assert (L.apc_host_rule_tiled_k_split(M, N, K), bool(L.apc_host_rule_slices_direct(M, N, K))) == (s, direct), (M, N, K)
                assert not direct or (s > 1 and K % (128 * s) == 0)


@pytest.mark.parametrize("kind,M,N,K,bands", [
    # few columns and a long K (0: plain, 1: gated, 2: q, k and v): a few blocks read everything, in slices many share it
    (2, 32, 640, 8192, 0), (2, 48, 640, 5440, 0), (2, 32, 1280, 8192, 0), (2, 64, 640, 4096, 0), (1, 32, 320, 8192, 0), (0, 48, 320, 5440, 0),
    # more than a round of blocks, where the tiled kernel needs no slices
    (1, 64, 14336, 1024, 0), (1, 17, 32000, 1024, 0), (0, 64, 32000, 1024, 0),
    # what one launch is for
    (0, 64, 4096, 4096, 1), (0, 64, 3072, 3072, 1), (2, 64, 5120, 3072, 2), (1, 64, 8192, 3072, 4), (0, 32, 3072, 2048, 1), (0, 32, 3072, 8192, 1), (2, 17, 3072, 2048, 2),
    # (the tiled kernel with a few blocks more than compute units)
    (0, 17, 10240, 2048, 4), (0, 37, 8320, 4032, 4)])
def test_products_of_17_to_64_rows_in_one_launch_where_that_is_faster(kind, M, N, K, bands):
    from allpaca_amd.kernels import host
    assert host.load().apc_host_rule_rows_bands(M, N, K, kind) == bands


def test_bands_of_gated_products_in_one_launch_do_not_depend_on_the_rows():
    """Which block an output is in is a matter of N, not of the rows beside a row."""
    from allpaca_amd.kernels import host
    rule = host.load().apc_host_rule_rows_bands
    for N in (16, 320, 1024, 2560, 4080, 4096, 4112, 5120, 8192, 11008, 14336):
        for K in (1024, 1536, 2048, 3072, 4096, 5440, 8192, 14336):
            assert {rule(M, N, K, 1) for M in range(17, 65)} <= {0, 4 if N > 4096 else 2}, (N, K)


def test_gated_products_and_the_sums_behind_a_norm_by_the_executors_rules():
    from allpaca_amd.kernels import host, tuned
    L = host.load()
    for M in (17, 64, 65, 128, 129, 200, 256, 257, 384, 512, 640, 1000, 1024, 1025, 2048):
        assert L.apc_host_rule_ss_parts_max(M) == tuned._ss_parts_max(M)
        for N in (192, 640, 1000, 2048, 4096, 8192, 16384, 28672):
            for K in (120, 512, 1088, 2048, 4096, 11008, 14336):
                assert L.apc_host_rule_gated_k_split(M, N, K) == tuned._tiled_k_split(M, N, K, True), (M, N, K)
                assert 128 < M <= 1024 or tuned._tiled_k_split(M, N, K, True) == tuned._tiled_k_split(M, N, K)


def test_the_expected_times_of_a_size_are_worked_out_once(monkeypatch):
    """A step's products come in the same few sizes, and the rule is 8 us of Python a product."""
    from allpaca_amd.kernels import tuned
    want = tuned._tiled_k_split(517, 4100, 4224)
    monkeypatch.setattr(tuned, "_direct_slices_us", lambda *a: pytest.fail("worked out again"))
    assert tuned._tiled_k_split(517, 4100, 4224) == want


@pytest.mark.parametrize("H,G,dk,dv,rows", [(32, 16, 64, 64, 64), (32, 32, 64, 64, 64), (32, 8, 64, 64, 32), (48, 16, 64, 64, 21), (64, 16, 128, 64, 16), (4, 1, 64, 64, 256)])
def test_single_rows_of_the_delta_rule_in_one_launch_while_the_chip_is_not_full(H, G, dk, dv, rows):
    from allpaca_amd.kernels import lib
    takes = lib.load("plain").apc_delta_step_takes
    assert takes(H, G, dk, dv, 4, 0, 1) and takes(H, G, dk, dv, 4, 0, rows) and not takes(H, G, dk, dv, 4, 0, rows + 1)
    assert not takes(H, G, dk, dv, 9, 0, 1) and not takes(H, G, dk, dv, 4, 8, 1) and not takes(5 * G, G, dk, dv, 4, 0, 1) and not takes(H, G, dk, 68, 4, 0, 1)


@pytest.mark.parametrize("M,H,Hk,d,K,together", [
    (2048, 32, 8, 128, 4096, 1), (1153, 24, 8, 128, 3072, 1), (1500, 32, 8, 64, 2048, 1), (2048, 16, 8, 128, 1024, 1), (1024, 4, 2, 64, 128, 1),
    # few columns in one round of blocks: tiles of 3 bands a wave, which the product that rotates does not have, end sooner
    (1025, 8, 1, 128, 2048, 0), (2048, 16, 2, 64, 2048, 0), (1300, 8, 2, 128, 2048, 0), (1025, 16, 2, 128, 2048, 0), (1025, 14, 2, 64, 896, 0),
    (64, 32, 8, 128, 4096, 0), (2048, 32, 8, 96, 4096, 0), (2048, 32, 8, 128, 4100, 0)])
def test_q_k_v_of_many_rows_rotated_by_the_product_where_that_is_faster(M, H, Hk, d, K, together):
    from allpaca_amd.kernels import lib
    assert lib.load("tuned").apc_gemm_direct_qkv_takes(0, K, 0, (H + 2 * Hk) * d, M, K, H, Hk, d, 0, 0) == together


@pytest.mark.parametrize("M,N,K,slices", [
    # a short K, columns so few that tiles of 3 bands would be needed to fill the chip
    (1025, 2048, 2048, 2), (1153, 3072, 3072, 2), (1300, 1024, 2048, 2),
    # a longer K: the slices' way through memory (48.5 / 49.7, 88 / 92, 139 / 146, 87 / 90, 51 / 54 us)
    (1025, 4096, 4096, 1), (1153, 4096, 8192, 1), (1153, 5120, 11008, 1), (2400, 2048, 8192, 1), (3000, 1536, 4096, 1), (2048, 2048, 2048, 1),
    # what products that leave no row take in slices
    (1153, 3072, 8192, 2), (1025, 1024, 4096, 2), (2048, 2048, 8192, 2), (1023, 2048, 8192, 1), (1025, 2048, 2200, 1),
    (1500, 4096, 14336, 2)])
def test_slices_of_k_of_products_into_the_residual_of_more_than_1024_rows(M, N, K, slices):
    from allpaca_amd.kernels import lib
    L = lib.load("tuned")
    assert L.apc_gemm_direct_emit_k_split(M, N, K) == slices >= L.apc_gemm_direct_k_split(M, N, K)


@pytest.mark.parametrize("tiles,heads,splits,d,pairs,last,one", [
    (4, 32, 1, 128, 64, 1, 1), (8, 32, 1, 128, 128, 1, 1), (8, 32, 1, 128, 128, 0, 1),           # a round of decode blocks at most
    (4, 32, 1, 128, 512, 0, 1), (12, 32, 1, 128, 1024, 0, 1), (4, 32, 1, 64, 1024, 0, 1),        # more, where the tiles leave units free
    (8, 32, 1, 128, 512, 0, 0), (4, 32, 2, 128, 256, 0, 0), (8, 32, 2, 64, 256, 0, 0),           # tiles that fill whole rounds
    (15, 32, 1, 128, 512, 0, 1), (4, 32, 1, 128, 2048, 0, 0), (1, 32, 1, 128, 2048, 0, 0), (4, 32, 1, 64, 2048, 0, 0)])
def test_decoded_rows_in_the_launch_of_the_prompt_rows_where_that_is_faster(tiles, heads, splits, d, pairs, last, one):
    from allpaca_amd.kernels import host
    assert host.load().apc_host_rule_decode_beside_tiles(tiles * heads * splits, d, pairs, last) == one
