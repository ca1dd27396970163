"""Column ids made on the device (single problems of 16,384 columns and more)
and on the host (below): the storage classes of envelopes at the edges of every
class, and the propagated bounds bit for bit the round-synchronous oracle's.

Sizes: one column below and above the line, the last tile of the sort full
(16,384 = 4 x 4096), one column into the next, and several tiles.
"""
import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import small_mip

pytestmark = pytest.mark.gpu

# (vartype, lower, upper, key): 0 binary, 1 int16, 2 int32, 3 FP64 records
EDGES = [(0, 0.0, 1.0, 0), (1, 0.0, 1.0, 0), (1, -0.0, 0.0, 0), (1, 1.0, 1.0, 0), (1, 0.0, 2.0, 1), (1, -1.0, 1.0, 1),
         (1, -32767.0, 32767.0, 1), (1, 0.0, 32768.0, 2), (1, -32768.0, 0.0, 2), (1, -2147483647.0, 2147483647.0, 2),
         (1, 0.0, 2147483648.0, 3), (1, -2147483648.0, 0.0, 3), (1, 0.5, 3.0, 3), (1, 0.0, 2.5, 3), (3, 0.0, 1.0, 3),
         (1, 0.0, 1e20, 3), (1, -1e20, 4.0, 3)]


def _instance(n):
    inst = small_mip(seed=n, m=n // 2 + 3, n=n)
    lb, ub, vt = inst.lb.copy(), inst.ub.copy(), inst.vartype.copy()
    for k, (v, l, u, _) in enumerate(EDGES * 3):
        j = (k * 331 + k // len(EDGES)) % n
        vt[j], lb[j], ub[j] = v, l, u
    vt[n - 1], lb[n - 1], ub[n - 1] = 1, 0.0, 1.0
    return inst.__class__(**{**inst.__dict__, "lb": lb, "ub": ub, "vartype": vt})


def _keys(inst):
    l, u = inst.lb, inst.ub
    with np.errstate(invalid="ignore"):
        integral = (np.abs(l) <= 2147483647.0) & (np.abs(u) <= 2147483647.0) & (l == np.floor(l)) & (u == np.floor(u))
    key = np.where(integral & (inst.vartype != 3), 2, 3)
    key[(key == 2) & (np.abs(l) <= 32767) & (np.abs(u) <= 32767)] = 1
    key[(key == 1) & (l >= 0) & (u <= 1)] = 0
    return key


@pytest.mark.parametrize("n", [16383, 16384, 16385, 40000])
@pytest.mark.parametrize("compact", [1, 0])
def test_classes_and_bounds(gpu, oracle, n, compact):
    inst = _instance(n)
    key = _keys(inst)
    print(f"column order: n={n} compact={compact}", flush=True)
    p = I.Problem(inst, {"compact_bounds": compact})
    try:
        st = p.stats()
        got = p.propagate(inst.lb, inst.ub, I.CPU_LOOP)
    finally:
        p.close()
    count = np.bincount(key, minlength=4) if compact else [0, 0, 0, n]
    assert [st.n_binary, st.n16, st.n32, st.nf] == [count[0], count[0] + count[1], count[2], count[3]]
    exp = oracle.jacobi(inst)
    np.testing.assert_array_equal(got.lbs, exp[0])
    np.testing.assert_array_equal(got.ubs, exp[1])
    assert (got.rounds, got.infeasible, got.capped) == exp[2:]
