"""Double-buffered rounds: single problems of up to 8M padded entries with
default tuning run each round as one phase (one launch, or one barrier of the
persistent launch).  Checked bit for bit against the round-synchronous oracle
and against the three-phase rounds, which an explicit work-item size selects,
at the sizes where the plan changes: entries per lane (64K and 512K padded
entries), workgroup size of the persistent launch (1024 and 2048 items), the
largest problem of the rule and the first one beyond it.
"""
import numpy as np
import pytest

import fixtures
from gdp_amd import interface as I
from gdp_amd.instances import from_rows, powerlaw_mip, small_mip

pytestmark = pytest.mark.gpu

SYNCS = [I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL]


def _check(inst, oracle, syncs=SYNCS, max_rounds=100, tunings=(None,)):
    exp = oracle.jacobi(inst, max_rounds=max_rounds)
    for tuning in tunings:
        p = I.Problem(inst, tuning)
        try:
            for sync in syncs:
                got = p.propagate(inst.lb, inst.ub, sync, max_rounds)
                label = f"{inst.name} m={inst.m} nnz={inst.nnz} tuning={tuning} sync={sync} cap={max_rounds}"
                np.testing.assert_array_equal(got.lbs, exp[0], err_msg=label)
                np.testing.assert_array_equal(got.ubs, exp[1], err_msg=label)
                assert (got.rounds, got.infeasible, got.capped) == exp[2:], label
        finally:
            p.close()
    return exp


def _rows_of(width, m, n, seed):
    """m rows of one width over n columns, mixed column types."""
    rng = np.random.default_rng(seed)
    x = small_mip(seed=seed, m=m, n=n, len_lo=width, len_hi=width)
    return x if width > 1 else from_rows(m, n, [[int(c)] for c in rng.integers(0, n, m)],
                                         [[float(v)] for v in rng.integers(1, 9, m)], [-1e20] * m,
                                         rng.integers(1, 40, m).astype(float), [0.0] * n, [50.0] * n,
                                         rng.choice([0, 1, 3], n))


@pytest.mark.parametrize("width", [1, 2, 3, 4, 8, 17, 33, 65, 129, 256, 257, 513])
@pytest.mark.parametrize("m", [1, 63, 65])
def test_widths_and_remainders(gpu, oracle, width, m):
    print(f"rounds: width {width} rows {m}", flush=True)
    _check(_rows_of(width, m, max(700, 2 * width), width + m), oracle, tunings=(None, {"item_nnz": 1024}))


# about 11 nonzeros a row, 12.5 padded entries
@pytest.mark.parametrize("m", [5000, 6000, 40000, 44000, 130000, 330000, 380000, 650000, 700000])
def test_plan_thresholds(gpu, oracle, m):
    inst = small_mip(seed=m, m=m, n=m // 2 + 1)
    print(f"rounds: m {m} nnz {inst.nnz}", flush=True)
    _check(inst, oracle, tunings=(None, {"item_nnz": 1024}) if m < 100000 else (None,))


def test_split_rows_every_cap(gpu, oracle):
    """Split rows whose gate passes (a second phase in the round), stopped by
    every round cap: the last round's block is the one returned."""
    inst = powerlaw_mip(seed=5, m=4000, n=2000, len_hi=1900, s=1.7)
    rounds = _check(inst, oracle)[2]
    for cap in range(1, min(rounds, 8) + 1):
        _check(inst, oracle, max_rounds=cap)


@pytest.mark.parametrize("make", [fixtures.infeasible_instance, fixtures.int32_overflow,
                                  lambda: fixtures.tiny_integer(3), lambda: fixtures.tiny_integer(11)],
                         ids=["infeasible", "int32_overflow", "tiny3", "tiny11"])
def test_crossed_bounds_at_and_around_the_cap(gpu, oracle, make):
    """Crossed bounds are found one round late, from the other block: with the
    cap at the crossing round, before it and after it."""
    inst = make()
    rounds = _check(inst, oracle)[2]
    for cap in range(max(1, rounds - 2), min(100, rounds + 2) + 1):
        _check(inst, oracle, max_rounds=cap)


def test_no_records_of_a_class(gpu, oracle):
    """Only integer columns, only continuous ones, and FP64 records only."""
    _check(small_mip(seed=1, m=500, n=301, int_frac=1.0), oracle)
    _check(small_mip(seed=2, m=500, n=301, int_frac=0.0), oracle)
    _check(small_mip(seed=3, m=500, n=301), oracle, tunings=({"compact_bounds": 0},))


def test_state_without_room_for_the_second_block(gpu, oracle):
    """An allocation-free call whose run state fits the fixed array only
    without the rounds' arrays takes the three-phase rounds."""
    rows, n = 2000, 900_000
    per = n // rows
    rng = np.random.default_rng(4)
    inst = from_rows(rows, n, [list(range(i * per, (i + 1) * per)) for i in range(rows)],
                     [list(rng.integers(1, 9, per).astype(float)) for _ in range(rows)], [-1e20] * rows,
                     list(rng.integers(5, 500, rows).astype(float)), [0.0] * n, [60.0] * n,
                     list(np.where(rng.random(n) < 0.8, 1, 3)))
    exp = oracle.jacobi(inst)
    p = I.Problem(inst)
    try:
        assert p.stats().run_state_bytes <= 64 << 20
        for sync in SYNCS:
            dl, du = I.DeviceArray(inst.lb), I.DeviceArray(inst.ub)
            info = p.propagate_device_no_alloc(dl.ptr, du.ptr, sync)
            np.testing.assert_array_equal(dl.numpy(), exp[0])
            np.testing.assert_array_equal(du.numpy(), exp[1])
            assert (info.rounds, bool(info.infeasible)) == (exp[2], exp[3])
            dl.free()
            du.free()
    finally:
        p.close()
