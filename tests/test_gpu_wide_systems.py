"""Systems of many more columns than entries, against the round-synchronous
oracle, and the rules that look at the number of columns."""
import re
import time

import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import small_mip

pytestmark = pytest.mark.gpu

SYNCS = [I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL]


def _traced(make, monkeypatch, capfd):
    """The problem, and whether its persistent and its launched runs take the
    double-buffered rounds."""
    monkeypatch.setenv("GDP_TRACE_CREATE", "1")
    capfd.readouterr()
    p = make()
    monkeypatch.delenv("GDP_TRACE_CREATE")
    err = capfd.readouterr().err
    return p, tuple(int(re.search(rf" {k}=(\d+)", err).group(1)) > 0 for k in ("with_rounds", "rounds_launched"))


# 5000 items look for unmoved rows: launches up to 2.6M columns, persistent runs
# up to 5.2M; few items never look
@pytest.mark.parametrize("m,n,route", [
    (100_000, 5 << 19, (True, True)), (100_000, (5 << 19) + 33, (True, False)), (100_000, 10 << 19, (True, False)),
    (100_000, (10 << 19) + 33, (False, False)), (30, 1_000_003, (True, True)), (50_000, 6_000_001, (True, True))])
def test_routes_of_wide_systems(gpu, oracle, monkeypatch, capfd, m, n, route):
    inst = small_mip(seed=3, m=m, n=n)
    exp = oracle.jacobi(inst)
    p, got = _traced(lambda: I.Problem(inst), monkeypatch, capfd)
    try:
        assert got == route
        for sync in SYNCS + [I.MEGAKERNEL, I.CPU_LOOP]:  # the routes share a run state
            out = p.propagate(inst.lb, inst.ub, sync)
            np.testing.assert_array_equal(out.lbs, exp[0])
            np.testing.assert_array_equal(out.ubs, exp[1])
            assert (out.rounds, out.infeasible, out.capped) == exp[2:]
    finally:
        p.close()


# beyond 2^26 columns a round's records would need offsets of more than 31 bits
@pytest.mark.parametrize("n,rounds", [(1 << 26, True), ((1 << 26) + 1, False)])
def test_columns_of_the_rounds(gpu, oracle, monkeypatch, capfd, n, rounds):
    small = small_mip(seed=2, m=40, n=60)
    at = np.sort(np.random.default_rng(1).choice(n, 60, replace=False))
    lb, ub, vt = np.zeros(n), np.ones(n), np.zeros(n, np.int32)
    lb[at], ub[at], vt[at] = small.lb, small.ub, small.vartype
    inst = small.__class__(**{**small.__dict__, "n": n, "col": at[small.col].astype(np.int32), "lb": lb, "ub": ub,
                              "vartype": vt})
    exp = oracle.jacobi(small)
    p, got = _traced(lambda: I.Problem(inst), monkeypatch, capfd)
    try:
        assert got == (rounds, rounds)
        for sync in SYNCS:
            out = p.propagate(lb, ub, sync)
            np.testing.assert_array_equal(out.lbs[at], exp[0])
            np.testing.assert_array_equal(out.ubs[at], exp[1])
            assert (out.rounds, out.infeasible, out.capped) == exp[2:]
            out.lbs[at], out.ubs[at] = 0.0, 1.0
            assert not out.lbs.any() and (out.ubs == 1.0).all()
    finally:
        p.close()


def test_routes_of_a_wide_batch(gpu, oracle, monkeypatch, capfd):
    xs = [small_mip(seed=k, m=14_000 + k, n=700_000 + k) for k in range(8)]
    exp = [oracle.jacobi(x) for x in xs]
    b, got = _traced(lambda: I.Batch(xs), monkeypatch, capfd)
    try:
        assert got == (False, False)
        for sync in SYNCS:
            for out, e in zip(b.propagate(sync_type=sync), exp):
                np.testing.assert_array_equal(out.lbs, e[0])
                np.testing.assert_array_equal(out.ubs, e[1])
                assert (out.rounds, out.infeasible, out.capped) == e[2:]
    finally:
        b.close()


def test_wide_systems_are_not_slower_than_the_three_phases(gpu):
    """3.1M entries over 12M columns: rounds that copy the bitmap of the columns
    for every workgroup took 1.6 to 2.5 times as long."""
    inst = small_mip(seed=1, m=100_000, n=12_000_000, len_hi=60)
    took = {}
    for tuning in (None, {"item_nnz": 1024}):
        p = I.Problem(inst, tuning)
        lb, ub = I.DeviceArray(inst.lb), I.DeviceArray(inst.ub)
        for sync in SYNCS:
            times = []
            for _ in range(7):
                lb.upload(inst.lb)
                ub.upload(inst.ub)
                t = time.perf_counter()
                p.propagate_device(lb.ptr, ub.ptr, sync)
                times.append(time.perf_counter() - t)
            took[tuning is None, sync] = sorted(times)[2]
        p.close()
        lb.free()
        ub.free()
    print(took, flush=True)
    for sync in SYNCS:
        assert took[True, sync] < 1.4 * took[False, sync], took


def test_a_candidate_marks_at_least_its_row(gpu, oracle):
    """8000 rows of 2 entries over 800,000 columns: round 1 accepts candidates in
    more than an eighth of the rows, so round 2 processes all of them."""
    inst = small_mip(seed=5, m=8000, n=800_000, len_lo=2, len_hi=2)
    p = I.Problem(inst)
    try:
        out, rows, _, _, accepted = p.work_profile(inst.lb, inst.ub)
        assert inst.m / 8 < accepted[0] < inst.m * inst.n / (8 * inst.nnz), accepted
        assert rows[0] == rows[1] == inst.m, rows
        exp = oracle.jacobi(inst)
        np.testing.assert_array_equal(out.lbs, exp[0])
        np.testing.assert_array_equal(out.ubs, exp[1])
    finally:
        p.close()
