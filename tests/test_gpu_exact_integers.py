"""Candidates beyond the int32 range in runs that follow each other: the exact
integer accumulators of a run state start clean in every run, whatever the
runs before left in them.  Each run bit for bit the round-synchronous oracle's.
"""
import numpy as np
import pytest

import fixtures
from gdp_amd import interface as I

pytestmark = pytest.mark.gpu

SYNCS = [I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL]


def _vectors(oracle):
    """int32_overflow's bounds, and with w from -8e8 on: candidates of 3e9 and
    5e9, then of 2.2e9 and 4.2e9 (the larger ones would win over them)."""
    inst = fixtures.int32_overflow()
    out = []
    for w in (0.0, -8e8):
        lb = inst.lb.copy()
        lb[4] = w
        out.append((lb, inst.ub, oracle.jacobi(inst, lb=lb)))
    assert not np.array_equal(out[0][2][0], out[1][2][0])
    return inst, out


def _same(got, want, label):
    np.testing.assert_array_equal(got.lbs, want[0], err_msg=label)
    np.testing.assert_array_equal(got.ubs, want[1], err_msg=label)
    assert (got.rounds, got.infeasible, got.capped) == want[2:], label


@pytest.mark.parametrize("tuning", [None, {"item_nnz": 1024}], ids=["rounds", "three phases"])
def test_runs_in_turn(gpu, oracle, tuning):
    inst, vectors = _vectors(oracle)
    p, b = I.Problem(inst, tuning), I.Batch([inst, inst], tuning)
    try:
        for sync in SYNCS:
            for k in (0, 1, 1, 0, 1):
                lb, ub, want = vectors[k]
                label = f"sync={sync} vector {k}"
                _same(p.propagate(lb, ub, sync), want, label)
                dl, du = I.DeviceArray(lb), I.DeviceArray(ub)
                p.propagate_device_no_alloc(dl.ptr, du.ptr, sync)
                np.testing.assert_array_equal(dl.numpy(), want[0], err_msg=label + " no alloc")
                np.testing.assert_array_equal(du.numpy(), want[1], err_msg=label + " no alloc")
                dl.free()
                du.free()
                for g in p.propagate_nodes([lb] * 3, [ub] * 3, sync_type=sync):
                    _same(g, want, label + " nodes")
                other = vectors[1 - k]
                for g, e in zip(b.propagate([lb, other[0]], [ub, other[1]], sync), (want, other[2])):
                    _same(g, e, label + " batch")
    finally:
        p.close()
        b.close()
