"""Where the GEMM planner's lines lie, at the sizes on either side of each (host only): the plans that sweeps over cold weights
found faster, and scratch that covers whatever a call may run."""
import itertools
import re

import pytest

from nanovllm import _qlinear as Q

G, S, R, A, NARROW = Q.QL_PLAN_GROUP, Q.QL_PLAN_SILU, Q.QL_PLAN_ROPE, Q.QL_PLAN_W8A8, Q.QL_PLAN_NARROW
I8, F8 = Q.QL_INT8, Q.QL_FP8


def wide(p):
    return p[1:] == (8, 1, 8, 1)


@pytest.fixture()
def no_table():
    lib = Q.load()
    lib.ql_gemm_plan_clear()
    yield lib
    Q.load_plan_table(Q.PLAN_TABLE)


@pytest.mark.parametrize("form,dtype,group,M,N,K,expected", [
    (G, F8, 64, 600, 4096, 2048, True), (G, I8, 64, 600, 4096, 2048, False), (G, I8, 32, 4096, 6144, 2560, False), (G, I8, 96, 4096, 6144, 2304, False),
    (G, I8, 192, 4096, 6144, 2304, False), (G, I8, 256, 4096, 6144, 2560, True), (A, F8, 0, 4096, 6144, 2560, True), (A | NARROW, F8, 0, 4096, 6144, 2560, False),
    (NARROW, I8, 0, 4096, 6144, 2560, False), (A | S | NARROW, I8, 0, 4096, 6144, 2560, False), (A, I8, 0, 4096, 6144, 2432, False), (0, I8, 0, 4096, 6144, 2432, True)])
def test_a_query_answers_for_the_call(no_table, form, dtype, group, M, N, K, expected):
    """The weight type, the group size and what the call does with its activations decide, not the form alone."""
    assert wide(Q.plan_query(form, M, N, K, dtype, group)) == expected


@pytest.mark.parametrize("form,dtype,M,N,K,expected", [
    (0, I8, 1, 36864, 4096, False), (0, I8, 32, 36864, 4096, False), (0, I8, 33, 36864, 4096, True), (0, I8, 1, 51200, 5120, True),
    (A, F8, 1, 36864, 4096, False), (A, F8, 4, 151936, 1024, False), (A, F8, 33, 151936, 1024, True), (A, F8, 1, 65536, 2048, True),
    (G | S, I8, 32, 51200, 5120, False), (G | S, I8, 64, 51200, 5120, True), (G, I8, 32, 51200, 5120, True),
    (0, I8, 640, 4096, 12288, False), (0, F8, 640, 4096, 12288, True), (0, I8, 704, 4096, 12288, True), (A, F8, 576, 4096, 12288, True),
    (R, F8, 1280, 4096, 1024, False), (R, I8, 1280, 4096, 1024, True), (R, F8, 1600, 4096, 1024, True), (R, F8, 640, 4096, 1024, True),
    (G, F8, 1280, 2048, 2048, False), (G, F8, 1600, 2048, 2048, True), (G, F8, 140, 12288, 3584, False), (G, F8, 640, 4096, 2048, True)])
def test_the_line_to_the_prefill_tiles(no_table, form, dtype, M, N, K, expected):
    assert wide(Q.plan_query(form, M, N, K, dtype)) == expected


@pytest.mark.parametrize("form", [G, G | S])
@pytest.mark.parametrize("M", [960, 961, 1000, 1024, 1025])
@pytest.mark.parametrize("N", [8192, 16384, 24576])
def test_what_the_cost_rule_refuses_goes_to_the_tile_it_compared_with(no_table, form, M, N):
    """Groups: the 128 x 256 tile where it is the cheaper one, at any row count; nothing falls through to the 64 x 128 tile."""
    p = Q.plan_query(form, M, N, 4096)
    assert wide(p) or p == (4, 8, 1, 2, 1)


@pytest.mark.parametrize("dtype", [I8, F8])
@pytest.mark.parametrize("M,N,K,there", [(1792, 4096, 4096, True), (1024, 6144, 2560, True), (1088, 6144, 2560, True), (1089, 6144, 2560, False),
                                         (1000, 6144, 2560, False), (1280, 6144, 1024, False), (900, 6144, 2560, False), (960, 4096, 4096, False)])
def test_one_round_of_128_row_tiles_with_groups_of_64(no_table, dtype, M, N, K, there):
    """Taken where two rounds of the prefill tile stand against it and its last row tile is whole, or at most half full."""
    p = Q.plan_query(G, M, N, K, dtype, 64)
    assert (p == (4, 8, 1, 2, 1)) == there and (there or wide(p))


@pytest.mark.parametrize("form,group", [(0, 0), (G, 64), (G, 128)])
@pytest.mark.parametrize("M,N,K,mt", [(4500, 1024, 512, 3), (9000, 1024, 512, 3), (4500, 2048, 768, 3), (3300, 1024, 512, 2), (16000, 480, 640, 2)])
def test_fewer_rounds_of_taller_tiles_over_short_k(no_table, form, group, M, N, K, mt):
    p = Q.plan_query(form, M, N, K, I8, group)
    assert wide(p) and (p[0] >= mt if not group else p[0] == mt)


@pytest.mark.parametrize("form,dtype,M,N,K", [(0, I8, 1024, 19456, 512), (0, I8, 1500, 13312, 768), (S, I8, 1500, 13312, 768), (S, F8, 1500, 13312, 768),
                                              (S, I8, 769, 19456, 768)])
def test_four_rounds_over_short_k_stay_in_low_tiles(no_table, form, dtype, M, N, K):
    assert Q.plan_query(form, M, N, K, dtype) == (2, 8, 1, 8, 1)


MID, MID64 = (1, 2, 4, 4), (2, 2, 4, 4)


@pytest.mark.parametrize("form,dtype,M,N,K,expected", [
    # 8-bit activations: by the ladder's pick (256 x 2048: one round of 32 x 64 tiles)
    (A, F8, 256, 2048, 6144, False), (A, F8, 128, 4096, 4096, False), (A, F8, 64, 6144, 2560, False), (A, F8, 192, 2560, 4096, False),
    (A, F8, 96, 5120, 6144, True), (A, I8, 96, 10240, 4096, True), (A, I8, 224, 5120, 5120, False), (A, F8, 192, 1024, 12288, True),
    (A, F8, 64, 1024, 8192, False), (A, I8, 160, 2048, 6144, True), (A, F8, 256, 2312, 9024, True), (A, I8, 96, 4104, 4160, True),
    (A, I8, 129, 7200, 2112, False), (A, I8, 224, 5120, 2560, True), (A, F8, 192, 2560, 8192, False), (A, F8, 160, 2816, 8256, True),
    (A, I8, 256, 4104, 4160, False), (A, F8, 128, 2312, 4160, True), (A, I8, 256, 640, 9024, False),
    (A, I8, 64, 2560, 10240, True),
    # 16-bit activations
    (0, I8, 128, 4096, 4096, False), (0, I8, 128, 2560, 6144, True), (0, F8, 128, 2560, 6144, True), (0, I8, 192, 6144, 5120, False),
    (0, I8, 96, 5120, 6144, True), (0, I8, 160, 4096, 4096, False), (0, F8, 160, 4096, 4096, True), (0, I8, 64, 10240, 12288, False),
    (0, I8, 192, 1024, 12288, True), (0, I8, 64, 1024, 8192, False), (0, I8, 96, 10240, 9728, False), (0, F8, 180, 3584, 11008, False),
    (0, I8, 128, 4104, 2112, True), (0, F8, 33, 9216, 3584, True), (0, I8, 256, 2048, 4096, False), (0, I8, 256, 4104, 8256, False), (0, I8, 256, 4104, 2112, True),
    (0, I8, 192, 5136, 2112, False), (0, I8, 192, 5120, 2304, True), (0, I8, 128, 2312, 4160, True), (0, F8, 96, 2816, 4160, True),
    # groups
    (G, I8, 128, 8192, 9728, True), (G, I8, 128, 10240, 4096, False), (G, I8, 96, 2048, 2560, False), (G, I8, 48, 2048, 6144, True),
    (G, F8, 64, 5120, 12288, False), (G, I8, 40, 9216, 13824, False), (G, I8, 64, 8192, 12288, True),
    # outside: few rows, many rows, short K
    (0, I8, 32, 2560, 9728, False), (0, I8, 257, 2560, 9728, False), (0, I8, 64, 5120, 2048, False)])
def test_the_tile_of_33_to_256_rows_over_long_k(no_table, form, dtype, M, N, K, expected):
    got = Q.plan_query(form, M, N, K, dtype)[:4]
    assert (got == (MID64 if form & G and M > 64 else MID)) == expected, got


@pytest.mark.parametrize("M,N,K,expected", [(64, 19456, 2048, True), (33, 24576, 4096, True), (64, 16384, 4096, False), (64, 12288, 2048, False),
                                            (33, 6144, 3072, False), (64, 19456, 1536, False), (65, 19456, 2048, False)])
def test_silu_of_8_bit_activations_at_33_to_64_rows(no_table, M, N, K, expected):
    assert (Q.plan_query(A | S, M, N, K, F8) == (2, 2, 2, 8, 1)) == expected


def test_calls_that_the_prefill_tiles_are_not_built_for_take_their_own_entries():
    """Groups of 32, operands off 16 bytes, staged quantization and row maxima keep the measured plans of their shapes."""
    Q.load()
    for form, M, N, K, group, plan in [(G | S, 768, 19456, 2560, 32, (4, 8, 1, 2, 1)), (G | R, 768, 6144, 2560, 32, (4, 8, 1, 2, 1)),
                                       (G, 2048, 2560, 4096, 96, (4, 8, 1, 2, 1)), (S | NARROW, 384, 19456, 2560, 0, (4, 8, 1, 4, 1)),
                                       (A | S | NARROW, 64, 19456, 2560, 0, (1, 4, 2, 16, 1)), (R | NARROW, 640, 4096, 1024, 0, (2, 4, 1, 4, 1))]:
        assert Q.plan_query(form, M, N, K, I8, group) == plan, (form, M, N, K, group)
        if form & NARROW:
            assert Q.plan_query(form & ~NARROW, M, N, K, I8, group) != plan
        else:
            assert wide(Q.plan_query(form, M, N, K, I8, 128))


def test_an_entry_for_narrow_calls_only_serves_them(no_table):
    lib, N, K = no_table, 6144, 2560
    before = Q.plan_query(0, 512, N, K)
    assert wide(before)
    assert lib.ql_gemm_plan_set(NARROW, 400, 600, N, K, 2, 4, 2, 4, 1) == 0
    assert Q.plan_query(0, 512, N, K) == before and Q.plan_query(NARROW, 512, N, K) == (2, 4, 2, 4, 1)
    assert lib.ql_gemm_plan_set(0, 400, 600, N, K, 4, 8, 1, 4, 1) == 0              # an entry of the form itself comes first
    assert Q.plan_query(0, 512, N, K) == Q.plan_query(NARROW, 512, N, K) == (4, 8, 1, 4, 1)
    assert lib.ql_gemm_plan_set(NARROW | Q.QL_PLAN_PARTIAL, 1, 32, N, K, 1, 1, 8, 4, 1) == -1
    out = (Q._c_int * 5)()
    for bad in [(0, I8, 128), (G, I8, 0), (64, I8, 0), (0, 2, 0)]:
        assert lib.ql_gemm_plan_of_call(*bad, 512, N, K, out) == -1


@pytest.mark.parametrize("table", [True, False])
@pytest.mark.parametrize("N,K", [(2560, 9728), (2560, 4096), (4096, 12288), (6144, 2560), (1024, 3072), (3584, 11008), (5120, 5120), (19456, 2560)])
def test_scratch_covers_every_plan_of_a_row_count(N, K, table):
    """A workspace is asked for by shape and granularity alone: it has to hold the plan of either weight type, of any group size,
    on and off 16 bytes."""
    lib = Q.load()
    if not table:
        lib.ql_gemm_plan_clear()
    try:
        for M in (1, 32, 33, 64, 65, 96, 128, 160, 192, 256, 320, 512, 700, 961, 1024, 1280, 2048):
            for grp, epi, dt, narrow in itertools.product((0, G), (0, S, R), (I8, F8), (0, NARROW)):
                for act, group in itertools.product((0,) if grp else (0, A), (32, 64, 128, 256)):
                    if K % group or (epi == R and N % 128):
                        continue
                    mt, wn, _, _, split = Q.plan_query(grp | epi | act | narrow, M, N, K, dt, group)
                    tiles = -(-M // (32 * mt)) * -(-N // (32 * wn))
                    slabs = tiles * split if split > 1 else (-split + tiles if split < 0 else 0)
                    need = 65536 + slabs * wn * mt * 4096 if slabs else 0
                    have = lib.ql_gemm_workspace_bytes(M, N, K, Q.QL_PER_GROUP if grp else Q.QL_PER_ROW)
                    assert have >= need, (M, grp, epi, act, dt, group, narrow)
    finally:
        if not table:
            Q.load_plan_table(Q.PLAN_TABLE)


@pytest.mark.parametrize("form,dtype", [(0, I8), (0, F8), (A, I8), (A, F8)])
def test_costs_choose_one_plan_for_every_32_rows(no_table, form, dtype):
    """Scratch is asked for by the last row count of 32: all of them have to run on its plan."""
    for N, K in [(8192, 12288), (4096, 9728), (2048, 12288), (3072, 3072), (1344, 7104)]:
        for last in (32, 64, 96, 160, 256):
            assert len({Q.plan_query(form, M, N, K, dtype) for M in range(last - 31, last + 1)}) == 1


@pytest.mark.parametrize("form,dtype,M,N,K,plan", [
    (A, F8, 33, 8192, 12288, (2, 2, 4, 8, 2)), (A, I8, 64, 6144, 8192, (2, 2, 4, 8, 2)), (0, I8, 64, 2048, 12288, (1, 2, 4, 8, 4)),
    (A | S, F8, 64, 19456, 2560, (2, 4, 2, 8, 1)), (A | S, F8, 64, 16384, 2560, (2, 2, 4, 8, 1))])
def test_plans_that_costs_and_long_gates_take(no_table, form, dtype, M, N, K, plan):
    assert Q.plan_query(form, M, N, K, dtype) == plan


MODELS = {"0.6b": [(4096, 1024), (1024, 2048), (1024, 3072)], "1.7b": [(4096, 2048), (2048, 2048), (2048, 6144)],
          "4b": [(6144, 2560), (2560, 4096), (2560, 9728)], "8b": [(6144, 4096), (4096, 4096), (4096, 12288)]}


@pytest.mark.parametrize("form,dtype", [(0, I8), (0, F8), (A, I8), (A, F8)])
@pytest.mark.parametrize("model", MODELS)
def test_costs_of_a_layers_shapes_are_worked_out_once(no_table, model, form, dtype):
    """The linears of a layer in turn: each finds its answer of the step before."""
    lib = Q.load()
    for M in (1, 32, 33, 64, 100, 256):
        def layer():
            return [Q.plan_query(form, M, N, K, dtype) for N, K in MODELS[model]]
        first, before = layer(), lib.ql_gemm_plans_costed()
        for _ in range(3):
            assert layer() == first
        assert lib.ql_gemm_plans_costed() == before


def test_costs_of_measured_and_forced_plans_are_not_worked_out(no_table):
    lib = Q.load()
    assert lib.ql_gemm_plan_set(A, 1, 32, 5024, 7072, 1, 2, 4, 8, 3) == 0
    before = lib.ql_gemm_plans_costed()
    assert Q.plan_query(A, 32, 5024, 7072, F8) == (1, 2, 4, 8, 3)
    try:
        assert lib.ql_gemm_force_config(1, 1, 8, 4, 1) == 0
        assert Q.plan_query(A, 32, 5056, 7072, F8) == (1, 1, 8, 4, 1)
    finally:
        lib.ql_gemm_force_config(0, 0, 0, 0, 0)
    assert lib.ql_gemm_plans_costed() == before
    Q.plan_query(A, 32, 5056, 7072, F8)
    assert lib.ql_gemm_plans_costed() == before + 1


@pytest.mark.parametrize("M,N,K", [(33, 8192, 12288), (64, 6144, 8192), (8, 4096, 9728), (48, 1344, 7104), (16, 5120, 8192), (200, 1024, 5120)])
@pytest.mark.parametrize("dtype", [I8, F8])
@pytest.mark.parametrize("entry", [None, A, A | NARROW])
def test_a_query_of_staged_quantization_answers_for_the_call(no_table, entry, dtype, M, N, K):
    """The call says what scratch its plan needs, and launches nothing without it."""
    import ctypes
    lib = Q.load()
    if entry is not None:
        assert lib.ql_gemm_plan_set(entry, M, M, N, K, 1, 2, 4, 4, 4) == 0
    mt, wn, wk, cp, split = Q.plan_query(A | Q.QL_PLAN_STAGED, M, N, K, dtype)
    assert split > 1 and (entry is None) != ((mt, wn, wk, cp, split) == (1, 2, 4, 4, 4))
    here = ctypes.create_string_buffer(64)
    at = ctypes.addressof(here)
    assert lib.ql_gemm_w8a8_dynq(dtype, at, at, 1, at, at, None, at, M, N, K, None, 0, None) != 0
    tiles = -(-M // (32 * mt)) * -(-N // (32 * wn))
    slabs = tiles * split * wn * mt * 16 * 64 * 4
    need, slices = re.search(r"workspace of (\d+) bytes needed for split-K=(\d+)", lib.ql_last_error().decode()).groups()
    assert int(slices) == split and int(need) == 65536 + slabs              # (a ticket for each of 16384 tiles in front)


def test_what_a_query_of_staged_quantization_refuses(no_table):
    import ctypes
    lib, out = Q.load(), (ctypes.c_int * 5)()
    for form in (Q.QL_PLAN_STAGED, A | S | Q.QL_PLAN_STAGED, A | R | Q.QL_PLAN_STAGED, A | Q.QL_PLAN_PARTIAL | Q.QL_PLAN_STAGED):
        assert lib.ql_gemm_plan_of_call(form, I8, 0, 33, 8192, 12288, out) != 0
    assert lib.ql_gemm_plan_set(A | Q.QL_PLAN_STAGED, 1, 32, 8192, 12288, 1, 2, 4, 4, 1) != 0


@pytest.mark.parametrize("form", [S, S | A, S | G, S | NARROW, S | A | NARROW])
def test_gates_under_silu_have_one_slice_by_the_rules(no_table, form):
    """Their plans may change inside a block of 32 rows (at 48): the block's last row count need not stand for their scratch."""
    for N, K in [(384, 256), (2048, 1024), (6144, 1024), (12288, 2048), (19456, 2560), (24576, 4096), (32768, 4096), (65536, 8192), (8192, 12288), (28672, 14336)]:
        for dtype in (I8, F8):
            for M in (1, 8, 16, 32, 33, 47, 48, 49, 64, 65, 96, 128, 129, 200, 256, 257, 512, 1024, 1025, 4096):
                assert Q.plan_query(form, M, N, K, dtype)[4] == 1


@pytest.mark.parametrize("form", [0, A, G, A | Q.QL_PLAN_STAGED])
def test_one_plan_for_every_32_rows(no_table, form):
    """Scratch is asked for by the last row count of 32, whatever the form (but gates under SiLU, above)."""
    for N, K in [(1024, 2048), (4096, 1024), (4096, 4096), (2560, 9728), (18496, 2560), (24576, 4096), (8192, 12288), (1344, 7104), (3072, 3072)]:
        for dtype in (I8, F8):
            for last in (32, 64, 96, 128, 160, 224, 256, 288, 512):
                assert len({Q.plan_query(form, M, N, K, dtype) for M in range(last - 31, last + 1)}) == 1
