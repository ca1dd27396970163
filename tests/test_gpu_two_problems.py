"""Problems in use from two threads at once.  The process shares the staging of
bulk copies, the pinned slots and blocks and the device memory cache between
them: every result is compared with the oracle, bit for bit, for vectors that
cross through a pinned block (up to 128 KiB each), through the staging while it
is free (below 1 MiB) and as bulk copies, with problems created and destroyed
meanwhile.
"""
import threading

import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import powerlaw_mip, small_mip

pytestmark = pytest.mark.gpu

SYNCS = [I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL]


def _instances(seed):
    return [small_mip(seed=seed, m=1500, n=900),
            small_mip(seed=seed + 1, m=9000, n=40_000),
            powerlaw_mip(seed=seed + 2, m=20_000, n=150_000, len_hi=3000, s=2.0)]


def _same(got, exp, label):
    np.testing.assert_array_equal(got.lbs, exp[0], err_msg=label)
    np.testing.assert_array_equal(got.ubs, exp[1], err_msg=label)
    assert (got.rounds, got.infeasible) == exp[2:4], label


@pytest.mark.parametrize("kept", [True, False])
def test_two_threads(gpu, oracle, kept):
    """kept: each thread's problems live as long as it runs; else every run has
    a problem of its own (the stateless call)."""
    work = [_instances(10), _instances(20)]
    expected = [[oracle.jacobi(x) for x in insts] for insts in work]
    print(f"two threads, problems kept: {kept}", flush=True)
    start, errors = threading.Barrier(2), []

    def run(t):
        problems = []
        try:
            problems = [I.Problem(x) for x in work[t]] if kept else []
            start.wait(60)
            for k in range(12):
                i, sync = (k + t) % 3, SYNCS[(k // 3) % 3]
                inst = work[t][i]
                got = problems[i].propagate(inst.lb, inst.ub, sync) if kept else I.gpu_propagate(inst, sync)
                _same(got, expected[t][i], f"thread {t} run {k}: {inst.name} n={inst.n} sync={sync}")
        except BaseException as e:  # reported below
            errors.append(e)
            start.abort()
        finally:
            for p in problems:
                p.close()

    threads = [threading.Thread(target=run, args=(t,)) for t in range(2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors, errors


def test_graphs_beside_synchronising_calls(gpu, oracle):
    """New graphs of launches are made while another thread copies through the
    null stream and waits for the device: neither disturbs the other.  (Captures
    were ended by such calls, which failed themselves.)"""
    inst = small_mip(seed=3, m=300, n=200)
    exp = oracle.jacobi(inst)
    stop, errors, copies = threading.Event(), [], [0]
    array = I.DeviceArray(inst.lb)

    def copy():
        try:
            while not stop.is_set():
                array.upload(inst.lb)
                copies[0] += 1
        except BaseException as e:  # reported below
            errors.append(e)

    th = threading.Thread(target=copy)
    th.start()
    try:
        for k in range(60):
            _same(I.gpu_propagate(inst, I.GPU_LOOP), exp, f"run {k}")
        b = I.Batch([inst] * 3)
        for k in range(20):
            for got in b.propagate(sync_type=I.GPU_LOOP, max_rounds=100 - k):
                np.testing.assert_array_equal(got.lbs, exp[0], err_msg=f"batch {k}")
        b.close()
    finally:
        stop.set()
        th.join()
        array.free()
    assert not errors, errors
    assert copies[0] > 60
