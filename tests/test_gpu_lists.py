"""Steps of marked rows through the lists of marked work, with many bound
vectors in a launch: each vector bit for bit the round-synchronous oracle's.

Sizes: fewer vectors than one XCD group needs (63), from 64 on the groups of
the XCDs (a count not divisible by 8), and more than one LDS window of every
group (8,300).  Hinted vectors start from a reference's segment partials; a
vector that has nothing to do with it drops them all, and a single one
computes its own.
"""
import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import powerlaw_mip, small_mip, tighten_node

pytestmark = pytest.mark.gpu


def _nodes(inst, oracle, count, seed, k_hi):
    lb, ub = oracle.jacobi(inst)[:2]
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        l, u, cols = tighten_node(inst, rng, 1, k_hi, lb, ub)
        out.append((l, u, cols, oracle.jacobi(inst.with_bounds(l, u))))
    return out


def _run(inst, nodes, pick, sync, hints=True, tuning=None):
    print(f"lists: {inst.name} m={inst.m} vectors={len(pick)} sync={sync} hints={hints}", flush=True)
    p = I.Problem(inst, tuning)
    try:
        got = p.propagate_nodes([nodes[k][0] for k in pick], [nodes[k][1] for k in pick],
                                hints=[nodes[k][2] for k in pick] if hints else None, sync_type=sync)
    finally:
        p.close()
    for k, g in zip(pick, got):
        exp = nodes[k][3]
        np.testing.assert_array_equal(g.lbs, exp[0])
        np.testing.assert_array_equal(g.ubs, exp[1])
        assert (g.rounds, g.infeasible, g.capped) == exp[2:]


@pytest.mark.parametrize("sync", [I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL])
@pytest.mark.parametrize("count", [1, 2, 3, 63, 64, 75])
def test_children_with_split_rows(gpu, oracle, count, sync):
    inst = powerlaw_mip(seed=6, m=6000, n=3000, len_hi=2900, s=1.8)
    nodes = _nodes(inst, oracle, min(count, 16), 7, 12)
    _run(inst, nodes, [k % len(nodes) for k in range(count)], sync)


@pytest.mark.parametrize("tuning", [None, {"max_split_segs": 0}, {"mark_limit": 1 << 30}, {"item_nnz": 4096}])
def test_unhinted_and_tuned(gpu, oracle, tuning):
    inst = powerlaw_mip(seed=6, m=6000, n=3000, len_hi=2900, s=1.8)
    nodes = _nodes(inst, oracle, 9, 8, 12)
    _run(inst, nodes, list(range(9)), I.MEGAKERNEL, hints=False, tuning=tuning)
    _run(inst, nodes, list(range(9)), I.MEGAKERNEL, tuning=tuning)


def test_vectors_unlike_the_reference(gpu, oracle):
    """Children of the propagated root among children of a far deeper node:
    their hints hold, but 287 of the 3000 columns, in most bitmap words, differ
    from the reference."""
    inst = powerlaw_mip(seed=9, m=6000, n=3000, len_hi=2900, s=1.8)
    near = _nodes(inst, oracle, 3, 1, 6)
    rng = np.random.default_rng(2)
    l, u, _ = tighten_node(inst, rng, 40, 41, *oracle.jacobi(inst)[:2])
    deep = oracle.jacobi(inst.with_bounds(l, u))
    far = []
    for _ in range(3):
        cl, cu, cols = tighten_node(inst, rng, 1, 6, deep[0], deep[1])
        far.append((cl, cu, cols, oracle.jacobi(inst.with_bounds(cl, cu))))
    assert not deep[3]
    _run(inst, near + far, list(range(6)), I.MEGAKERNEL)
    _run(inst, far + near, list(range(6)), I.CPU_LOOP)


@pytest.mark.parametrize("count", [1100, 8300])
def test_many_windows(gpu, oracle, count):
    inst = small_mip(seed=4, m=300, n=150)
    nodes = _nodes(inst, oracle, 12, 5, 5)
    _run(inst, nodes, [k % 12 for k in range(count)], I.MEGAKERNEL)
    if count < 2000:
        _run(inst, nodes, [k % 12 for k in range(count)], I.CPU_LOOP)


@pytest.mark.parametrize("seed", [2, 3, 5, 7])
def test_rounds_after_few_candidates_process_marked_rows(gpu, seed):
    """A round processes every row after max(64, m n / (6 (nnz + n))) accepted
    candidates or more, else marked rows.  These runs have a round between an
    eighth and a sixth."""
    inst = small_mip(seed=seed, m=8000, n=40_000, len_hi=60, fixed_frac=0.02)
    p = I.Problem(inst)
    try:
        out, rows, _, _, accepted = p.work_profile(inst.lb, inst.ub)
    finally:
        p.close()
    limit = max(64, inst.m * inst.n // (6 * (inst.nnz + inst.n)))
    between = [a for a in accepted if inst.m * inst.n // (8 * (inst.nnz + inst.n)) <= a < limit]
    assert between, (list(accepted), limit)
    for k in range(out.rounds - 1):
        assert (rows[k + 1] == inst.m) == (accepted[k] >= limit), (k, list(rows), list(accepted), limit)
