"""Systems of many more columns than entries, against the round-synchronous
oracle, and the rules that look at the number of columns."""
import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import small_mip

pytestmark = pytest.mark.gpu


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
