"""Which kernel a projection goes to is decided on the host from its sizes alone; the
decisions are checked here without a GPU."""

import pytest

from zig_ai_amd.kernels import ops


@pytest.mark.parametrize("M,N,K,plan", [
    (8, 2048, 2048, 4),          # few outputs: K in ranges until some 512 workgroups run
    (8, 2048, 8192, 4),
    (1, 64, 4096, 8),
    (8, 6144, 12288, 2),         # a wide model: outputs alone fill the chip, K is too long
    (3, 8192, 28672, 4),
    (16, 5136, 9216, 2),
    (2, 48, 8200, 0),            # no cut of 8200 is a multiple of 32: the product comes back
    (17, 2048, 2048, 0),         # more than a decode batch
    (8, 2048, 2052, 0),          # rows that do not start on 16-byte boundaries
])
def test_how_a_decode_product_reaches_the_stream(M, N, K, plan):
    assert ops.accumulate_plan(M, N, K, False) == plan


def test_every_plan_fits_the_kernel():
    """Whatever the sizes, a plan's ranges are what the decode kernel takes: no longer than a
    workgroup covers, and a multiple of 32 when K is cut."""
    for N in (16, 100, 2048, 5136, 6144, 8192, 65536, 200000):
        for K in range(8, 70000, 8):
            plan = ops.accumulate_plan(8, N, K, False)
            if plan == 0:
                continue
            assert (K + plan - 1) // plan <= ops.ROWS16_MAX_K_PER_WORKGROUP, (N, K, plan)
            assert plan == 1 or K % (plan * 32) == 0, (N, K, plan)


def test_the_kernel_that_runs_the_norm_covers_k_alone():
    assert ops.accumulate_plan(8, 2048, 2048, True) == 1
    assert ops.normed_rows_pay(8, 2048, 2048) and not ops.normed_rows_pay(8, 2048, 4608)
    assert ops.normed_rows_pay(16, 2048, 2048) and not ops.normed_rows_pay(17, 16384, 2048)


def test_when_the_output_projection_merges_the_context_ranges():
    """Few rows in few ranges: every workgroup of the projection merges its slice of every
    row, which pays while rows x ranges stays small."""
    from zig_ai_amd.kernels import ops
    assert ops.merged_rows_pay(1, 8) and ops.merged_rows_pay(3, 8) and ops.merged_rows_pay(8, 2)
    assert ops.merged_rows_pay(2, 2) and ops.merged_rows_pay(4, 4) and ops.merged_rows_pay(8, 3)
    assert not ops.merged_rows_pay(8, 4) and not ops.merged_rows_pay(5, 8) and not ops.merged_rows_pay(4, 8)
    assert ops.merged_rows_pay(1, 12) and ops.merged_rows_pay(2, 12) and not ops.merged_rows_pay(2, 16)
    assert not ops.merged_rows_pay(3, 12)
    assert not ops.merged_rows_pay(1, 1) and not ops.merged_rows_pay(1, 17) and not ops.merged_rows_pay(9, 2)



def test_where_the_kernel_for_17_to_64_rows_is_taken():
    """The feed-forward's fused first product up to 48 rows, up to 64 on a stream no wider
    than 1,024, for widths whose K is spans of 512 (at least two) up to 4096; the mixer's
    closing product of such a step adds itself to the stream (through the library, see the
    next test; this package's kernel, where the library has nothing, when K is short and
    enough workgroups come of it)."""
    assert ops.rows64_swiglu_fusable(17, 2048) and ops.rows64_swiglu_fusable(32, 1024)
    assert ops.rows64_swiglu_fusable(33, 1024) and ops.rows64_swiglu_fusable(64, 1024)
    assert not ops.rows64_swiglu_fusable(65, 1024) and not ops.rows64_swiglu_fusable(49, 1536)
    assert ops.rows64_swiglu_fusable(20, 1536) and ops.rows64_swiglu_fusable(24, 4096)
    assert not ops.rows64_swiglu_fusable(16, 2048)      # the decode kernel's
    assert ops.rows64_swiglu_fusable(48, 2048)
    assert not ops.rows64_swiglu_fusable(49, 2048)      # measured no faster than the library's path
    assert not ops.rows64_swiglu_fusable(20, 512) and not ops.rows64_swiglu_fusable(20, 1280)
    assert not ops.rows64_swiglu_fusable(20, 4608)
    assert ops.rows64_add_splits(2048, 2048) == 2       # 32 tiles x 2 ranges of 1,024
    assert ops.rows64_add_splits(2048, 4096) == 4
    assert ops.rows64_add_splits(2048, 8192) == 0       # the library's ranges of K are faster
    assert ops.rows64_add_splits(1024, 1024) == 0       # 16 workgroups: too few
    assert ops.rows64_add_splits(4096, 1024) == 1
    assert ops.rows64_add_splits(2048, 1280) == 0       # no cut into spans of 512
    for K in range(512, 9000, 256):
        for N in (1024, 2048, 4096):
            ks = ops.rows64_add_splits(N, K)
            assert ks == 0 or ops.rows64_takes(32, K, ks)


def test_where_the_library_adds_a_product_to_the_stream_itself():
    """Many rows (beyond those whose K the library gets in ranges): only with a long K, the
    feed-forward's closing product.  Few rows (17 to 64): only with a short K, a mixer's
    closing product, and only where a feed-forward that runs its norm itself can follow on a
    stream of that width.  Elsewhere the product comes back and the next norm adds it."""
    assert ops.library_adds(2048, 2048, 8192) and ops.library_adds(1025, 1024, 4608)
    assert ops.library_adds(4096, 2560, 10752)
    assert not ops.library_adds(2048, 2048, 2048)          # the mixers' closing products
    assert not ops.library_adds(1024, 2048, 8192)          # K in ranges instead
    assert not ops.library_adds(2048, 2048, 4100)          # rows that do not start on 16 bytes
    for M in (17, 64, 512, 1024):
        assert not ops.library_adds(M, 2048, 8192)
    # few rows
    for M in (17, 24, 32):
        assert ops.library_adds(M, 2048, 2048) and ops.library_adds(M, 1024, 1024)
        assert ops.library_adds(M, 2048, 1024)
    for M in (33, 48, 64):
        assert ops.library_adds(M, 1024, 1024) and ops.library_adds(M, 2048, 2048) == (M <= 48)
    for M in (16, 65, 128, 512):
        assert not ops.library_adds(M, 1024, 1024)
    assert not ops.library_adds(24, 1280, 1024)            # no fused feed-forward at that width
    assert not ops.library_adds(24, 2048, 4096)            # a long K stays in ranges


def test_the_batch_sizes_that_recordings_are_kept_for():
    """A decode batch without a recording of its own is filled up to 1, 2, 4, 8, 16 requests
    or, beyond, to a multiple of 8: never by more than 7 rows."""
    from zig_ai_amd.engine.runner import ModelRunner
    sizes = [ModelRunner.padded_size(n) for n in range(1, 70)]
    assert sizes[:17] == [1, 2, 4, 4, 8, 8, 8, 8, 16, 16, 16, 16, 16, 16, 16, 16, 24]
    assert all(0 <= s - n <= 7 for n, s in zip(range(1, 70), sizes))
    assert all(s % 8 == 0 for s in sizes[16:]) and sizes[63] == 64 and sizes[64] == 72


def test_where_the_tiles_for_17_to_64_rows_are_taken():
    """Products whose K comes in ranges, products with enough outputs to occupy the chip, and
    gated ones with half as many."""
    from zig_ai_amd.kernels import ops
    for M in (17, 64):
        assert ops.tiles_take(M, 2048, 8192, 8) and ops.tiles_take(M, 512, 4096, 8)
        assert not ops.tiles_take(M, 200, 4096, 8)          # 32 workgroups
        assert not ops.tiles_take(M, 512, 2048, 4)          # as many
        assert ops.tiles_take(M, 65536, 2048, 1) and not ops.tiles_take(M, 6144, 2048, 1)
        assert not ops.tiles_take(M, 2048, 1000, 4)         # ranges that are no steps of 64
        assert ops.tiles_take_gated(M, 8192, 2048) and ops.tiles_take_gated(M, 4608, 1024)
        assert not ops.tiles_take_gated(M, 2048, 2048) and not ops.tiles_take_gated(M, 8192, 2044)
    for M in (16, 65):
        assert not ops.tiles_take(M, 2048, 8192, 8) and not ops.tiles_take(M, 65536, 2048, 1)
        assert not ops.tiles_take_gated(M, 8192, 2048)


def test_where_a_router_runs_in_one_kernel():
    """Few blocks of 16 weight rows and a short K; with more of either the product's own kernel, which
    many workgroups share, is faster."""
    pays = ops.route_linear_pays
    assert pays(8, 8, 2048) and pays(20, 8, 2048) and pays(64, 16, 2048) and pays(16, 16, 8192)
    assert not pays(17, 16, 2560) and not pays(64, 8, 4096)
    assert pays(8, 33, 2048) and pays(1, 32, 2048) and pays(64, 80, 512) and pays(1, 64, 512)
    assert not pays(9, 33, 2048) and not pays(8, 33, 2560) and not pays(64, 32, 1024)
    assert not pays(1, 64, 1024) and not pays(64, 80, 4096) and not pays(20, 64, 2048)
    # steps beyond 64 tokens, where a launch costs more
    assert pays(65, 80, 1024) and pays(1777, 48, 2048) and pays(8192, 16, 4096)
    assert not pays(65, 64, 2048) and not pays(1777, 32, 2560) and not pays(4096, 16, 5120)


def test_how_far_portions_over_planes_are_cut():
    """Beyond one workgroup a compute unit where walks differ in length and two workgroups share a
    compute unit; not where ranges only add a merge."""
    from zig_ai_amd.parts.attention import planes_target
    most, least = planes_target(128, 64, 1200, True, True), planes_target(128, 128, 1200, True, True)
    assert (most, least) == (400, 256)
    assert planes_target(64, 64, 1200, True, True) == planes_target(96, 96, 5000, True, False) == most
    assert planes_target(128, 64, 3000, False, False) == planes_target(72, 8, 800, False, False) == most
    assert planes_target(128, 64, 1028, False, True) == planes_target(64, 64, 3000, False, False) == least
    assert planes_target(128, 64, 700, True, False) == planes_target(192, 96, 3000, True, False) == least
    assert planes_target(136, 64, 3000, False, False) == planes_target(128, 104, 3000, True, False) == least


@pytest.mark.parametrize("outputs,rank", [(4096, 512), (4096, 128), (32768, 512), (2560, 1024)])
def test_how_many_rows_keys_and_values_are_formed_for(outputs, rank):
    """Any sum of contexts leaves the library few numbers of rows, none of them far more than there are."""
    from zig_ai_amd.parts.latent_attention import FORMING_BLOCK, forming_rows
    asked = set()
    for rows in range(1, 33000):
        room = forming_rows(rows, outputs, rank)
        assert rows <= room < rows + max(FORMING_BLOCK, rows / 4)
        assert forming_rows(room, outputs, rank) == room
        if room > FORMING_BLOCK and not ops.half_plan(room, outputs, rank, False)[0]:
            asked.add(room)
    assert len(asked) <= 25


@pytest.mark.parametrize("tokens,top,experts,outputs,inner,once", [
    (1, 4, 32, 1024, 2048, False),       # a token's four experts of 32
    (1, 4, 32, 512, 1024, False),
    (1, 2, 8, 2048, 1024, False),
    (1, 2, 8, 4096, 2048, True),
    (2, 4, 32, 1024, 2048, True),
    (8, 4, 32, 512, 1024, True),
    (8, 2, 8, 1024, 1024, False),        # all of them together are no more
    (20, 2, 8, 4096, 2048, True),
    (400, 4, 32, 1024, 2048, True),
    (640, 4, 32, 1024, 2048, False),     # many rows an expert
])
def test_which_experts_are_read_past_the_caches(tokens, top, experts, outputs, inner, once):
    """By the bytes that a launch can read, not by those of experts that no token of the step goes to."""
    rule = ops.build.load("experts").za_grouped_reads_once
    assert bool(rule(tokens * top, experts, outputs, inner)) == once


def test_where_a_token_gate_runs_in_its_product():
    """Up to a round of loads, or whole ones and few rows: part of a round costs as much as a whole one."""
    assert all(ops.table_gate_fuses(T, K) for T in (1, 8, 16) for K in (8, 1024, 1544, 2048))
    assert all(ops.table_gate_fuses(T, K) for T in (1, 8) for K in (4096, 8192))
    assert not any(ops.table_gate_fuses(T, K) for T in (1, 8, 16) for K in (2056, 2560, 3072, 5120))
    assert not any(ops.table_gate_fuses(T, K) for T, K in ((9, 4096), (16, 8192), (17, 1024), (4, 1028)))


def test_where_a_decode_batch_shares_k_out_to_waves():
    """What the host takes for the kernels' own line between their two forms is that line."""
    import os
    import re
    with open(os.path.join(ops.build.CSRC_DIR, "latent.hip")) as f:
        line, = re.findall(r"#define HL_SPLIT_MIN_K (\d+)", f.read())
    assert int(line) == ops.HEAD_SPLIT_MIN_K
