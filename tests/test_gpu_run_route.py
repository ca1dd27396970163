"""Which rounds a problem's runs take, as GDP_TRACE_CREATE reports it at
creation (with_rounds: bytes of the run state with the arrays of the
double-buffered rounds, 0 where runs take the three phases)."""
import re

import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import small_mip

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
