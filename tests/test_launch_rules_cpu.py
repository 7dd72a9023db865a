"""The launch rules on the host: which sizes take which kernel."""
import ctypes

import launch_rules

CUS = 256


def test_wide_tiles_do_not_leave_half_a_round_empty():
    """Two rounds of wide tiles, each at least 1.5 narrow tiles' time, are kept
    only where they are shorter than the rounds of twice as many narrow tiles."""
    L = launch_rules.lib()
    for tiles_m in (1, 8, 16, 17, 28, 32, 40, 64):
        for cols in range(1, 49):
            tiles = tiles_m * cols
            wide = L.rule_mxg_wide(1, tiles_m, 256 * cols, 1, 0, 1024)
            if tiles < CUS:
                assert not wide
                continue
            rounds_wide, rounds_narrow = -(-tiles // CUS), -(-2 * tiles // CUS)
            if rounds_wide == 2:
                assert wide == (1.5 * rounds_wide < rounds_narrow)
            else:
                assert wide
    # the joined projections of 8 x 512 tokens, 16 heads of 64
    assert not L.rule_mxg_wide(1, 32, 3072, 1, 0, 1024)
    assert not L.rule_mxg_wide(1, 32, 3072, 1, 1, 1024)
    assert L.rule_mxg_wide(1, 32, 3072, 1, 1, 4096)  # FP4, long rows
    assert not L.rule_mxg_wide(1, 32, 3072 + 128, 1, 0, 1024)  # no multiple of the width
    assert L.rule_mxg_wide(64, 2, 1024, 1, 0, 1024)  # 64 members: two full rounds


def test_joined_projections_stay_within_the_large_tiles():
    """Three matrices below 2 GiB each whose joined rows reach it: mha_join, which
    asks this rule, must leave them apart (the product refuses the joined one)."""
    fit = launch_rules.lib().rule_mxg_weights_fit
    fit.argtypes = [ctypes.c_longlong, ctypes.c_longlong]
    d = 26880  # FP8, full heads
    assert fit(d, d) and not fit(3 * d, d)
    assert fit(3 * 26624, 26624) and not fit(3 * 26880, 26880)
    assert fit((1 << 31) // 32768 - 256, 32768) and not fit((1 << 31) // 32768 - 255, 32768)


FORMATS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 16, 17]


def test_format_waves_load_what_they_have():
    """The runs of sub-blocks that a wave of the small-batch kernel loads ahead:
    a built (waves, depth), and less than one sub-block per run past its last."""
    built = {(4, 2), (4, 3), (4, 4), (8, 3), (8, 4), (16, 2), (16, 3), (16, 4)}
    seen = set()
    for fmt, rows, nsub in [(f, r, n) for f in (2, 8) for r in (16, 8192) for n in range(1, 400)]:
        p = launch_rules.format_plan(fmt, rows, 32 * nsub, 16)
        assert p.kernel == launch_rules.ROWS
        seen.add((p.waves, p.depth))
        per = -(-nsub // p.waves)
        runs = -(-per // p.depth)
        assert runs * p.depth - per < max(runs, 3 - per)  # (2 is the least depth)
    assert seen == built


def test_format_kernels_by_size():
    plan = launch_rules.format_plan
    for fmt in FORMATS:
        for batch in (1, 2, 3):
            assert plan(fmt, 4096, 4096, batch).kernel == launch_rules.PER_ROW
        for out, inp in ((256, 512), (8192, 256), (448, 768), (4096, 4096)):
            assert plan(fmt, out, inp, 8).kernel == plan(fmt, out, inp, 16).kernel == launch_rules.ROWS
        # narrow inputs at many rows: one launch while it is the shorter one
        assert plan(fmt, 256, 512, 300).kernel == launch_rules.ROWS
        assert plan(fmt, 256, 512, 1000).kernel == launch_rules.ROWS
        assert plan(fmt, 448, 768, 300).kernel == launch_rules.ROWS
        assert plan(fmt, 8192, 256, 64).kernel == launch_rules.GEMM
        assert plan(fmt, 1024, 1024, 100).kernel == launch_rules.ROWS
        assert plan(fmt, 1024, 1024, 300).kernel == launch_rules.GEMM
        assert plan(fmt, 4096, 4096, 17).kernel == launch_rules.GEMM
        # (the grid's second dimension holds 65535 blocks of 16 batch rows)
        assert plan(fmt, 16, 32, 1 << 20).kernel == launch_rules.GEMM
        assert [plan(fmt, 4096, 4096, b)[3:5] for b in (64, 128, 256, 512)] == [(1, 1), (1, 2), (2, 2), (2, 4)]
