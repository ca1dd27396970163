"""Node vectors of which one works for many rounds while the others have
nothing left: bit for bit the round-synchronous oracle's, and the whole chip
works on the one that is left, from 64 vectors on (where an XCD's workgroups
take pieces that lie together) as below.
"""
import time

import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import powerlaw_mip, small_mip

pytestmark = pytest.mark.gpu

SYNCS = [I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL]


# around the 64 vectors of the rule, not multiples of 8, more than the 1024 of a window
@pytest.mark.parametrize("count", [63, 64, 67, 200, 1100])
@pytest.mark.parametrize("make", [lambda: small_mip(seed=2, m=3000, n=1500),
                                  lambda: powerlaw_mip(seed=5, m=4000, n=2000, len_hi=1500, s=1.8)],
                         ids=["short rows", "split rows"])
def test_one_long_vector(gpu, oracle, make, count):
    inst = make()
    exp = oracle.jacobi(inst)
    done = oracle.jacobi(inst, lb=exp[0], ub=exp[1])
    p = I.Problem(inst)
    try:
        for at, sync in [(k, s) for k in (0, count // 2, count - 1) for s in SYNCS]:
            lbs, ubs = [exp[0]] * count, [exp[1]] * count
            lbs[at], ubs[at] = inst.lb, inst.ub
            hints = [np.array([k % inst.n], np.int32) for k in range(count)]
            hints[at] = np.zeros(0, np.int32)
            label = f"{inst.name} count={count} at={at} sync={sync}"
            print(label, flush=True)
            for k, g in enumerate(p.propagate_nodes(lbs, ubs, hints=hints, sync_type=sync)):
                want = exp if k == at else done
                np.testing.assert_array_equal(g.lbs, want[0], err_msg=f"{label} vector {k}")
                np.testing.assert_array_equal(g.ubs, want[1], err_msg=f"{label} vector {k}")
                assert (g.rounds, g.infeasible, g.capped) == want[2:], f"{label} vector {k}"
    finally:
        p.close()


def test_one_long_vector_has_the_chip(gpu):
    """4.4M nonzeros, one vector of 32 rounds and 62 or 63 that end at once:
    an eighth of the chip takes 2.2 times as long as all of it."""
    inst = small_mip(seed=1, m=400_000, n=300_000)
    p = I.Problem(inst)
    root = p.propagate(inst.lb, inst.ub, I.MEGAKERNEL)
    took = {}
    try:
        for sync in SYNCS:
            for count in (63, 64):
                p.reserve(count)
                lb = [I.DeviceArray(inst.lb)] + [I.DeviceArray(root.lbs) for _ in range(count - 1)]
                ub = [I.DeviceArray(inst.ub)] + [I.DeviceArray(root.ubs) for _ in range(count - 1)]
                hints = [np.zeros(0, np.int32)] + [np.array([k], np.int32) for k in range(count - 1)]
                times = []
                for _ in range(7):
                    lb[0].upload(inst.lb)
                    ub[0].upload(inst.ub)
                    t = time.perf_counter()
                    p.propagate_nodes_device([x.ptr for x in lb], [x.ptr for x in ub], hints, sync)
                    times.append(time.perf_counter() - t)
                took[sync, count] = sorted(times)[2]
                for x in lb + ub:
                    x.free()
            print(f"sync={sync}: 63 vectors {took[sync, 63] * 1e6:.0f} us, 64 {took[sync, 64] * 1e6:.0f} us", flush=True)
            assert took[sync, 64] < 1.5 * took[sync, 63]
    finally:
        p.close()
