"""Which rounds a problem's runs take, as GDP_TRACE_CREATE reports it at
creation (with_rounds: bytes of the run state with the arrays of the
double-buffered rounds, 0 where runs take the three phases)."""
import re
import time

import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import INF, Instance, small_mip

pytestmark = pytest.mark.gpu


def _bytes(make, monkeypatch, capfd):
    """The problem and its reported bytes: (least state, with lists, with rounds)."""
    monkeypatch.setenv("GDP_TRACE_CREATE", "1")
    capfd.readouterr()
    p = make()
    monkeypatch.delenv("GDP_TRACE_CREATE")
    err = capfd.readouterr().err
    return p, tuple(int(re.search(rf" {k}=(\d+)", err).group(1)) for k in ("state_bytes", "with_lists", "with_rounds"))


# every option of the three phases selects them; the others leave the rounds
@pytest.mark.parametrize("tuning,rounds", [
    (None, True), ({"graph_rounds": 4}, True), ({"compact_bounds": 0}, True), ({"row_marking": 0}, False),
    ({"mark_limit": 1 << 30}, False), ({"mark_limit": 64}, False), ({"item_nnz": 1024}, False),
    ({"mega_threads": 256}, False), ({"mega_blocks_per_cu": 1}, False), ({"max_split_segs": 0}, False)])
def test_options_reach_the_phases_they_describe(gpu, oracle, monkeypatch, capfd, tuning, rounds):
    inst = small_mip(seed=4, m=3000, n=1500)
    exp = oracle.jacobi(inst)
    for make in (lambda: I.Problem(inst, tuning), lambda: I.Batch([inst, inst], tuning)):
        p, got = _bytes(make, monkeypatch, capfd)
        try:
            assert (got[2] > 0) == rounds, (tuning, got)
            if isinstance(p, I.Problem):
                out = p.propagate(inst.lb, inst.ub)
            else:
                out = p.propagate()[1]
            np.testing.assert_array_equal(out.lbs, exp[0])
            np.testing.assert_array_equal(out.ubs, exp[1])
        finally:
            p.close()


STATE_BYTES, ARRAY_BYTES = 64 << 20, 128 << 20  # of the allocation-free call


def _blocks(rows, n):
    """`rows` rows over disjoint columns, 80% of them integer, the others continuous."""
    per = n // rows
    rng = np.random.default_rng(4)
    val = rng.integers(1, 9, n).astype(float)
    return Instance(rows, n, np.arange(n, dtype=np.int32), (np.arange(rows + 1) * per).astype(np.int32), val,
                    np.full(rows, -INF), rng.integers(5, 500, rows).astype(float), np.zeros(n), np.full(n, 60.0),
                    np.where(rng.random(n) < 0.8, 1, 3).astype(np.int32))


# what the array holds beside the run state: lists of marked rows and the rounds'
# arrays, or only the lists (always: the marks leave room for them)
@pytest.mark.parametrize("make,rounds", [
    (lambda: _blocks(2000, 1_000_000), True), (lambda: _blocks(2000, 1_900_000), False),
    (lambda: small_mip(seed=6, m=2_000_000, n=1_800_000, len_lo=2, len_hi=2), False)],
    ids=["rounds", "lists", "many rows"])
def test_what_the_allocation_free_array_holds(gpu, oracle, monkeypatch, capfd, make, rounds):
    inst = make()
    exp = oracle.jacobi(inst)
    p, got = _bytes(lambda: I.Problem(inst), monkeypatch, capfd)
    try:
        print(got, flush=True)
        assert got[0] == p.stats().run_state_bytes <= STATE_BYTES
        assert got[1] <= ARRAY_BYTES and got[2] > 0 and (got[2] <= ARRAY_BYTES) == rounds, got
        for sync in (I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL):
            dl, du = I.DeviceArray(inst.lb), I.DeviceArray(inst.ub)
            for _ in range(2):  # from the bounds, then from their fixpoint
                info = p.propagate_device_no_alloc(dl.ptr, du.ptr, sync)
                np.testing.assert_array_equal(dl.numpy(), exp[0])
                np.testing.assert_array_equal(du.numpy(), exp[1])
            assert info.rounds == 1
            dl.upload(inst.lb)
            du.upload(inst.ub)
            info = p.propagate_device_no_alloc(dl.ptr, du.ptr, sync)
            assert (info.rounds, bool(info.infeasible), bool(info.capped)) == exp[2:]
            dl.free()
            du.free()
        assert p.stats().n_units == 0
    finally:
        p.close()


def test_many_rows_keep_their_marks_without_allocation(gpu):
    """11M nonzeros, a state of 64.4 MB and lists beyond 64 MiB: without the lists,
    every step processed all rows and took 1.8 times as long."""
    inst = small_mip(seed=1, m=1_000_000, n=2_000_000)
    p = I.Problem(inst)
    dl, du = I.DeviceArray(inst.lb), I.DeviceArray(inst.ub)
    took = []
    try:
        assert p.stats().run_state_bytes <= STATE_BYTES
        for fn in (p.propagate_device, p.propagate_device_no_alloc):
            times = []
            for _ in range(7):
                dl.upload(inst.lb)
                du.upload(inst.ub)
                t = time.perf_counter()
                fn(dl.ptr, du.ptr, I.CPU_LOOP)
                times.append(time.perf_counter() - t)
            took.append(sorted(times)[2] * 1e3)
        print(f"own state {took[0]:.2f} ms, array {took[1]:.2f} ms", flush=True)
        assert took[1] < 1.3 * took[0]
    finally:
        p.close()
        dl.free()
        du.free()
