"""Double-buffered rounds that leave out the rows none of whose columns moved
(from 4096 work items): bit for bit the round-synchronous oracle's.

Sizes: a bit per column in LDS (up to 512K columns) and shared bits (beyond);
split rows, of which only the segments with moved columns are summed again;
every early round cap; batches, whose last rounds fall below the line.
"""
import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import chain_mip, powerlaw_mip, small_mip

pytestmark = pytest.mark.gpu

SYNCS = [I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL]


def _same(got, exp, label):
    np.testing.assert_array_equal(got.lbs, exp[0], err_msg=label)
    np.testing.assert_array_equal(got.ubs, exp[1], err_msg=label)
    assert (got.rounds, got.infeasible, got.capped) == exp[2:], label


@pytest.mark.parametrize("make", [lambda: chain_mip(seed=2, m=60_000, n=300_000),
                                  lambda: chain_mip(seed=3, m=60_000, n=700_001),
                                  lambda: powerlaw_mip(seed=5, m=90_000, n=40_000, len_hi=9000, s=1.8),
                                  lambda: small_mip(seed=6, m=100_000, n=64_000)],
                         ids=["own bits", "shared bits", "split rows", "mixed"])
def test_single(gpu, oracle, make):
    inst = make()
    exp = oracle.jacobi(inst)
    p = I.Problem(inst)
    try:
        for cap in [100, 1, 2, 3, 4] + [r for r in (exp[2] - 1, exp[2]) if r > 4]:
            want = exp if cap == 100 else oracle.jacobi(inst, max_rounds=cap)
            for sync in SYNCS:
                label = f"{inst.name} n={inst.n} nnz={inst.nnz} sync={sync} cap={cap}"
                print(label, flush=True)
                _same(p.propagate(inst.lb, inst.ub, sync, cap), want, label)
    finally:
        p.close()


def test_batch(gpu, oracle):
    xs = [chain_mip(seed=4, m=9000, n=45_000), powerlaw_mip(seed=7, m=30_000, n=14_000, len_hi=3000, s=1.8),
          small_mip(seed=8, m=60_000, n=30_000), small_mip(seed=9, m=300, n=200)]
    exp = [oracle.jacobi(x) for x in xs]
    p = I.Batch(xs)
    try:
        for cap in (100, 3):
            want = exp if cap == 100 else [oracle.jacobi(x, max_rounds=cap) for x in xs]
            for sync in SYNCS:
                for i, (g, e) in enumerate(zip(p.propagate(sync_type=sync, max_rounds=cap), want)):
                    _same(g, e, f"instance {i} sync={sync} cap={cap}")
    finally:
        p.close()
