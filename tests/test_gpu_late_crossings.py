"""Bounds that cross after several double-buffered rounds of a system large
enough for many workgroups a launch: the launch that finds the crossing of the
round before is run whole, whichever of its waves see the report, and the next
one stops.  Bit for bit the round-synchronous oracle's, several times over.
"""
import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import INF, Instance, small_mip

pytestmark = pytest.mark.gpu


def _with_chain(inst, length, top):
    """inst and y[i + 1] >= y[i] + 1 over `length` new integer columns in [0, top]."""
    k = length - 1
    col = np.stack([inst.n + np.arange(k), inst.n + np.arange(1, length)], 1).ravel().astype(np.int32)
    return Instance(inst.m + k, inst.n + length, np.concatenate([inst.col, col]),
                    np.concatenate([inst.row_ptr, inst.nnz + 2 * np.arange(1, length)]).astype(np.int32),
                    np.concatenate([inst.val, np.tile([-1.0, 1.0], k)]), np.concatenate([inst.lhs, np.ones(k)]),
                    np.concatenate([inst.rhs, np.full(k, INF)]), np.concatenate([inst.lb, np.zeros(length)]),
                    np.concatenate([inst.ub, np.full(length, float(top))]),
                    np.concatenate([inst.vartype, np.ones(length, np.int32)]), f"{inst.name}+chain")


# below and above the 4096 items from which the rounds look for unmoved rows
@pytest.mark.parametrize("m", [20_000, 120_000])
@pytest.mark.parametrize("top", [5, 9])
def test_late_crossing(gpu, oracle, m, top):
    inst = _with_chain(small_mip(seed=m, m=m, n=m // 2), 2 * top + 4, top)
    exp = oracle.jacobi(inst)
    assert exp[3] and exp[2] > 2, exp[2:]
    p = I.Problem(inst)
    try:
        for sync in (I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL):
            for cap in (100, exp[2] + 1, exp[2], exp[2] - 1):
                want = exp if cap == 100 else oracle.jacobi(inst, max_rounds=cap)
                for _ in range(3):
                    label = f"m={m} top={top} sync={sync} cap={cap}"
                    print(label, flush=True)
                    got = p.propagate(inst.lb, inst.ub, sync, cap)
                    np.testing.assert_array_equal(got.lbs, want[0], err_msg=label)
                    np.testing.assert_array_equal(got.ubs, want[1], err_msg=label)
                    assert (got.rounds, got.infeasible, got.capped) == want[2:], label
    finally:
        p.close()
