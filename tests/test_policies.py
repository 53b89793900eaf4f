"""Decisions the host takes about a launch, checked without a GPU: how many workgroups share the keys
of a decode step's requests."""
import ctypes

import pytest

from tiny_llm_amd.kernels import library, ops


@pytest.fixture
def waves(monkeypatch):
    # eight waves a workgroup up to heads of 64, four beyond (what the library answers on the GPU)
    monkeypatch.setattr(ops, "flash_waves", lambda head_dim, groups=1 << 20: 8 if head_dim <= 64 else 4)


def test_short_contexts_are_not_split(waves):
    for rows in (1, 8, 64):
        assert ops.decode_key_splits(rows, 1024, 4, 64) == 1          # 16 key tiles: two a wave
        assert ops.decode_key_splits(rows, 512, 8, 128) == 1          # 8 key tiles: two a wave


def test_one_request_is_split_down_to_a_tile_a_wave_within_64(waves):
    assert ops.decode_key_splits(1, 2048, 4, 64) == 4
    assert ops.decode_key_splits(1, 8192, 4, 64) == 16
    assert ops.decode_key_splits(1, 32768, 4, 64) == 64
    assert ops.decode_key_splits(1, 1 << 20, 4, 64) == 64
    assert ops.decode_key_splits(1, 131072, 8, 128) == 32             # 8 kv heads: 256 workgroups


def test_splits_stay_within_one_round_of_workgroups_where_one_is_enough(waves):
    for rows, kv, hd in ((8, 4, 64), (8, 8, 128), (16, 8, 128), (64, 4, 64)):
        for ctx in (2048, 8192, 131072):
            assert rows * kv * ops.decode_key_splits(rows, ctx, kv, hd) <= 256


def test_a_mostly_empty_last_round_is_split_away_at_long_contexts(waves):
    # 8 requests x 40 kv heads: 320 workgroups are two rounds for the work of 1.25
    assert ops.decode_key_splits(8, 2048, 40, 128) == 1               # too short to pay for a merge
    assert ops.decode_key_splits(8, 8192, 40, 128) == 4
    assert ops.decode_key_splits(8, 131072, 40, 128) == 4
    # 64 x 8 = 512 workgroups are two full rounds: nothing to gain
    assert ops.decode_key_splits(64, 131072, 8, 128) == 1


def test_more_context_never_means_fewer_splits(waves):
    for rows, kv, hd in ((1, 4, 64), (8, 4, 64), (8, 40, 128), (16, 8, 128), (3, 5, 96)):
        got = [ops.decode_key_splits(rows, ctx, kv, hd) for ctx in (64, 640, 1280, 4224, 8192, 32768, 131072)]
        assert got == sorted(got) and 1 <= got[0] and got[-1] <= 64


def test_prompt_portions_split_their_keys_where_it_was_measured_to_pay():
    heads = dict(num_heads=32, num_kv_heads=8)
    assert ops.prefill_key_splits(2048, 2048, tile_waves=8, **heads) == 1          # a whole prompt: enough workgroups
    assert ops.prefill_key_splits(512, 512, tile_waves=4, **heads) == 1            # 8 key tiles: too short
    assert ops.prefill_key_splits(512, 8192, tile_waves=4, **heads) == 4
    assert ops.prefill_key_splits(512, 131072, tile_waves=4, **heads) == 8         # from 32,768 tokens of context on
    assert ops.prefill_key_splits(2048, 32768, tile_waves=8, **heads) == 1
    assert ops.prefill_key_splits(8192, 131072, tile_waves=8, **heads) == 4        # the same quarter of the keys together
    assert ops.prefill_key_splits(131072, 131072, tile_waves=8, **heads) == 1      # a whole prompt of that length
    for rows in (16, 100, 512, 2048, 8192):
        for ctx in (rows, 4096, 32768, 131072):
            if ctx >= rows:
                assert 1 <= ops.prefill_key_splits(rows, ctx, tile_waves=4, **heads) <= 8


def test_small_experts_products_go_by_rows():
    """Which experts' weights are read once for all their rows: large ones, and any in the second product of one or two
    tokens (small ones took up to four times as long that way)."""
    by_expert = library.load(verbose=False).tl_table_moe_by_expert
    up = lambda N, K, act=0: by_expert(0, 6, 4, N, K, act)
    down = lambda n_tokens, top, N, K: by_expert(1, n_tokens, top, N, K, 0)
    gate = 2
    assert up(2 * 704, 2048, gate) and up(704, 2048) and up(1408, 2048) and up(2048, 512, gate)
    assert not up(128, 512) and not up(2048, 1024) and not up(2 * 256, 1024, gate) and not up(256, 2048)
    assert down(6, 4, 2048, 704) and down(32, 2, 1024, 1024) and not down(8, 8, 1024, 256) and not down(64, 1, 512, 1536)
    assert down(1, 8, 256, 64) and down(2, 2, 64, 32) and not down(2, 1, 512, 128) and not down(3, 2, 256, 128)


def test_split_products_keep_their_number_of_parts():
    """How many float32 parts a split product's sums are added in, and so what its results round to: sizes of the ring
    kernel (two to sixteen parts), and of 128 x 128 tiles, shared out over 256 workgroups with at least four steps of 64 each."""
    plan = library.load(verbose=False).tl_splitk_plan
    ring = {(66, 1024, 512): 2, (80, 2048, 2048): 8, (128, 4096, 4096): 4, (150, 4096, 1024): 2, (200, 2048, 512): 2,
            (256, 2560, 2048): 3, (128, 1408, 2048): 8}
    for sizes, parts in ring.items():
        assert plan(*sizes) == parts, sizes
    for M in (257, 300, 400, 512, 640, 700, 1000, 1944, 2500):
        for N in (256, 518, 704, 1280, 2048, 2560, 4096, 6144, 11264):
            for K in (256, 512, 520, 1024, 1096, 2048, 4096, 5632, 14336):
                tiles, steps, parts = -(-M // 128) * -(-N // 128), -(-K // 64), 1
                if K >= 512 and tiles < 160:
                    share = max(-(-steps // -(-256 // tiles)), 4)
                    parts = -(-steps // share)
                assert plan(M, N, K) == parts, (M, N, K)


def test_operands_go_straight_into_lds_where_it_is_the_faster_way():
    """128 x 128 tiles: through registers beyond 256 workgroups of fewer than 32 steps, also where splitting the inner size makes
    them so many; every tile: through registers for inner sizes that end within a step."""
    mode = library.load(verbose=False).tl_tile_mode
    tail, whole, direct, quarters = 0, 1, 2, 3
    for M, N, K, share in ((1500, 1408, 1088, 576), (300, 2048, 2048, 384), (66, 11264, 2048, 704), (2102, 3968, 1984, 0),
                           (300, 2048, 128, 0), (128, 257 * 128, 4096, 2048)):
        assert mode(3, M, N, K, share) == whole, (M, N, K, share)
    for M, N, K, share in ((1500, 1408, 1088, 0), (300, 2048, 2048, 512), (128, 256 * 128, 256, 0), (2102, 3968, 2048, 0)):
        assert mode(3, M, N, K, share) == direct, (M, N, K, share)
    assert mode(2, 2102, 3968, 256, 0) == direct and mode(2, 2102, 3968, 192, 0) == whole
    assert mode(1, 100, 300, 64, 0) == quarters and mode(4, 100, 300, 4096, 0) == whole
    assert all(mode(t, 300, 300, K, 0) == tail for t in (1, 2, 3, 4) for K in (8, 72, 1000, 4104))


def test_large_tiles_are_worth_less_for_few_steps():
    """Products of fewer than eight steps choose among the tiles by other rates: their first loads and epilogues outweigh the
    loop."""
    best = library.load(verbose=False).tl_best_tile
    for M, N in ((2102, 3968), (2200, 3712), (700, 11264)):
        assert all(best(M, N, K) == 4 for K in (8, 64, 72, 128, 192, 200, 256, 328, 448, 504)), (M, N)
        assert all(best(M, N, K) == 1 for K in (512, 520, 704, 1000, 1024, 4104)), (M, N)
    for K in (64, 72, 256, 512, 1000, 2048):
        assert best(2048, 28672, K) == 1 and best(2048, 4096, K) == 2 and best(2048, 2048, K) == 3 and best(512, 2048, K) == 4, K


def _places(tiles_m, tiles_n, banded):
    place = library.load(verbose=False).tl_tile_place
    at, places = (ctypes.c_int * 2)(), []
    for t in range(tiles_m * tiles_n):
        place(t, tiles_m, tiles_n, banded, at)
        places.append((at[0], at[1]))
    assert sorted(places) == [(m, n) for m in range(tiles_m) for n in range(tiles_n)]      # every tile, once
    return places


@pytest.mark.parametrize("tiles_m", list(range(1, 45)) + [64, 101])
def test_tiles_through_registers_and_few_rows_of_tiles_stand_in_columns(tiles_m):
    columns = [(m, n) for n in range(5) for m in range(tiles_m)]
    assert _places(tiles_m, 5, 0) == columns
    assert (_places(tiles_m, 5, 1) == columns) == (tiles_m < 8)


def test_time_mix_runs_in_chunks_where_its_longest_portion_pays_for_them():
    """The steps beside the rule, and sizes that the chunks do not take."""
    pays = lambda lens, heads=32, dim=64: ops.time_mix_chunks_pay(sum(lens), len(lens), max(lens), heads, dim, dim)  # noqa: E731
    for lens in ([48] * 8, [48] * 64, [30] * 32, [31] * 16, [1] * 40 + [32] * 3, [1] * 64, [1]):      # chunks took 1.1 to 2.2 times as long
        assert not pays(lens), lens
    for lens in ([64], [2047], [67, 801, 143, 411, 205, 317], [1] * 8 + [512], [1] * 64 + [512], [1] * 64 + [1024]):
        assert pays(lens), lens
    assert pays([24] * 16, 16, 128) and pays([31] * 16, 16, 128) and not pays([24] * 8, 8, 128) and not pays([1] * 256, 16, 128)
    assert not pays([2047], 16, 32) and not pays([2047], 16, 129)


def test_a_step_is_known_by_the_forms_its_parts_choose():
    """Parts that choose a form by a step's own sizes are asked, those within a parallel mixer too, and no others."""
    from tiny_llm_amd.engine.step import StepContext, StepSizes
    from tiny_llm_amd.models.decoder import Decoder
    from tiny_llm_amd.parts import base, parallel

    class ByLength(base.Mixer):
        def form(self, sizes):
            return sizes.longest > 10

    plain, chooses = base.Mixer("a", None, None), ByLength("b", None, None)
    side = object.__new__(parallel.ParallelMixer)
    side.branches = [plain, chooses]
    d = object.__new__(Decoder)
    d._formed, d.parts = None, lambda: [plain, chooses, plain, side]
    assert d.forms(StepSizes(40, 4, 10)) == (False, (None, False)) and d.forms(StepSizes(40, 2, 30)) == (True, (None, True))
    d._formed, d.parts = None, lambda: [plain]
    assert d.forms(StepSizes(40, 4, 10)) == ()
    bare = dict.fromkeys(("tokens", "positions", "req_of_token", "cu_seqlens_q", "seq_lens", "state_slots", "logit_rows", "block_tables", "slot_mappings"))
    assert StepContext(num_tokens=9, num_requests=2, max_q_len=8, **bare).sizes == (9, 2, 8)
    assert StepContext(num_tokens=16, num_requests=2, max_q_len=16, sizes=StepSizes(9, 2, 8), **bare).sizes == (9, 2, 8)


def test_the_delta_rule_runs_in_chunks_where_its_longest_portion_pays_for_them():
    """The steps beside the rule, and sizes that the chunks do not take."""
    pays = lambda lens, heads=16, dim=128, vdim=128, taps=4: ops.delta_chunks_pay(sum(lens), len(lens), max(lens), heads, dim, vdim, taps)  # noqa: E731
    for lens in ([8] * 8, [24] * 8, [16], [1] * 40 + [32] * 3, [1] * 64, [1] * 256, [1]):
        assert not pays(lens), lens
    for lens in ([32] * 8, [48] * 8, [13] * 64, [48] * 64, [48], [2047], [67, 801, 143, 411, 205, 317], [1] * 8 + [128], [1] * 16 + [256],
                 [1] * 40 + [512], [1] * 64 + [512], [1] * 64 + [1024]):
        assert pays(lens), lens
    assert not pays([1] * 239 + [62], 32, 48, 64) and not pays([1] * 94 + [43], 64, 33, 33)
    assert not pays([2047], dim=32) and not pays([2047], dim=129) and not pays([2047], vdim=129) and not pays([2047], taps=5)


def test_no_plan_is_kept_for_rows_that_have_none():
    """A product of more rows than the kernel of whole lines takes leaves nothing behind: prompts have any length."""
    kept = len(ops._WHOLE)
    assert not any(ops.linear_whole(rows, 2048, 2048) for rows in range(65, 600))
    assert len(ops._WHOLE) == kept
    assert ops.linear_whole(64, 2048, 2048) and ops.linear_whole(9, 2048, 2048) and not ops.linear_whole(5, 2560, 2048)


def test_few_rows_of_short_inner_sizes_keep_their_kernel():
    """Where the kernel of whole lines was timed slower than the few-row one (inner sizes of up to 2,048): products of one and of several
    rounds of workgroups; odd multiples of 64 and longer inner sizes, whose sums are closer to 64 bits so, stay with whole lines."""
    whole = ops.linear_whole
    for rows, cols, inner in ((9, 32000, 2048), (16, 32000, 2048), (12, 128256, 2048), (9, 8192, 2048), (10, 6144, 1024), (8, 8192, 2048),
                              (6, 4704, 640), (8, 2560, 512), (16, 560, 256), (12, 2048, 640), (17, 3072, 256), (24, 4096, 512), (32, 2560, 256),
                              (9, 18432, 2048), (16, 40960, 1024)):
        assert not whole(rows, cols, inner), (rows, cols, inner)
    for rows, cols, inner in ((9, 32000, 2112), (9, 28672, 4096), (16, 28672, 1536), (11, 8192, 2048), (8, 8192, 2560), (8, 2560, 2048), (16, 560, 320),
                              (16, 1024, 512), (16, 2560, 704), (17, 2048, 256), (25, 4096, 512), (33, 3072, 256), (16, 11264, 2048),
                              (8, 11264, 2048), (64, 2560, 128)):
        assert whole(rows, cols, inner), (rows, cols, inner)


def test_norms_of_short_float32_rows_ride_where_a_block_is_one_request():
    """The float32 product with a norm inside: by whole lines only where a wave has more than the one or two blocks that the other
    kernel asks for at once."""
    lines = lambda rows, cols, inner: ops.linear_f32_lines(rows, cols, inner, inner, norm=True)
    assert not any(lines(rows, cols, inner) for rows in (1, 8, 12) for cols in (64, 2048, 6144) for inner in (64, 256, 512, 640, 768))
    assert not lines(16, 512, 512) and lines(16, 512, 768) and lines(1, 512, 896) and lines(8, 2048, 2048) and lines(16, 6144, 4096)
    assert not lines(1, 4096, 1152) and lines(8, 4096, 1152) and lines(1, 4096, 2048) and lines(1, 2048, 1152)
    assert all(ops.linear_f32_lines(rows, 512, inner, inner) for rows in (1, 16) for inner in (64, 512, 2048))      # without a norm
