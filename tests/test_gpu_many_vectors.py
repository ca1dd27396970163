"""Loads, unpacks and publishes of many bound vectors, and what a run state
keeps from one run to the next: each vector bit for bit the round-synchronous
oracle's.

Sizes: vectors around the line from which a vector's workgroups share an XCD
(64) and not a multiple of 8; columns around a workgroup's 1024 and a wave's
64, binary columns ending inside a wave; as many bitmap words as make a
publishing wave take 64 of them.
"""
import numpy as np
import pytest

import fixtures
from gdp_amd import interface as I
from gdp_amd.instances import powerlaw_mip, small_mip, tighten_node

pytestmark = pytest.mark.gpu

SYNCS = [I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL]


def _children(inst, oracle, count, seed):
    lb, ub = oracle.jacobi(inst)[:2]
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        l, u, cols = tighten_node(inst, rng, 1, 9, lb, ub)
        out.append((l, u, cols, oracle.jacobi(inst.with_bounds(l, u))))
    return out


def _run(p, nodes, pick, sync, hints=True):
    got = p.propagate_nodes([nodes[k][0] for k in pick], [nodes[k][1] for k in pick],
                            hints=[nodes[k][2] for k in pick] if hints else None, sync_type=sync)
    for i, (k, g) in enumerate(zip(pick, got)):
        exp = nodes[k][3]
        np.testing.assert_array_equal(g.lbs, exp[0], err_msg=f"vector {i} of {len(pick)} sync={sync}")
        np.testing.assert_array_equal(g.ubs, exp[1], err_msg=f"vector {i} of {len(pick)} sync={sync}")
        assert (g.rounds, g.infeasible, g.capped) == exp[2:]


@pytest.mark.parametrize("n", [63, 64, 65, 1023, 1025, 4100])
def test_columns_and_vectors(gpu, oracle, n):
    inst = powerlaw_mip(seed=n, m=2 * n + 30, n=n, len_hi=max(8, n // 2), s=1.7)
    nodes = _children(inst, oracle, 7, n)
    print(f"many vectors: n={n}", flush=True)
    p = I.Problem(inst)
    try:
        for count in (1, 15, 16, 63, 64, 67):
            for sync in SYNCS:
                _run(p, nodes, [k % 7 for k in range(count)], sync, hints=count != 67)
    finally:
        p.close()


@pytest.mark.parametrize("hints", [True, False])
def test_wide_publish(gpu, oracle, hints):
    inst = small_mip(seed=8, m=9000, n=30000, len_hi=9)
    nodes = _children(inst, oracle, 5, 3)
    p = I.Problem(inst)
    try:
        for sync in SYNCS:
            print(f"many vectors: 300, sync={sync} hints={hints}", flush=True)
            _run(p, nodes, [k % 5 for k in range(300)], sync, hints)
    finally:
        p.close()


def test_integers_beyond_int32_and_back(gpu, oracle):
    """A run that needs the exact integer accumulators, then runs of the same
    state that must find them clean, several times over."""
    inst = fixtures.int32_overflow()
    tight_ub = inst.ub.copy()
    ints = np.flatnonzero((inst.vartype != 3) & (inst.ub < 1e9) & (inst.lb > -1e9))
    tight_ub[ints] = inst.lb[ints]
    nodes = [(inst.lb, inst.ub, np.arange(inst.n, dtype=np.int32), oracle.jacobi(inst)),
             (inst.lb, tight_ub, ints.astype(np.int32), oracle.jacobi(inst.with_bounds(inst.lb, tight_ub)))]
    p = I.Problem(inst)
    try:
        for sync in SYNCS:
            for pick in ([1, 1, 1], [1, 0, 1], [1, 1, 0], [0, 1, 1], [1, 1, 1]):
                _run(p, nodes, pick, sync, hints=False)
    finally:
        p.close()


@pytest.mark.parametrize("n_bin", [1, 15, 16, 17, 63, 64, 65, 200])
def test_binary_codes(gpu, oracle, n_bin):
    """Binary columns read from their codes: counts around a code word (16
    columns) and a 16-byte group (64), before other classes, one vector and
    several."""
    inst = small_mip(seed=n_bin, m=600, n=300)
    lb, ub, vt = inst.lb.copy(), inst.ub.copy(), inst.vartype.copy()
    ints = np.flatnonzero(vt != 3)
    ub[ints] = np.maximum(ub[ints], lb[ints] + 2)
    pick = np.random.default_rng(n_bin).permutation(inst.n)[:n_bin]
    vt[pick], lb[pick], ub[pick] = 1, 0.0, 1.0
    inst = inst.__class__(**{**inst.__dict__, "lb": lb, "ub": ub, "vartype": vt})
    exp = oracle.jacobi(inst)
    p = I.Problem(inst, {"item_nnz": 512})
    try:
        assert p.stats().n_binary == n_bin
        for sync in SYNCS:
            for count in (1, 3):
                for g in p.propagate_nodes([lb] * count, [ub] * count, sync_type=sync):
                    np.testing.assert_array_equal(g.lbs, exp[0])
                    np.testing.assert_array_equal(g.ubs, exp[1])
                    assert (g.rounds, g.infeasible, g.capped) == exp[2:]
    finally:
        p.close()


@pytest.mark.parametrize("n, slots", [(63, 5), (65, 70), (4100, 12), (30000, 3)])
def test_server_changes(gpu, oracle, n, slots):
    """A server's changed columns, listed by the unpack: columns around a wave,
    more requests than slots, full vectors beside deltas, and (30,000 columns
    from the unpropagated bounds) more changes than a list holds."""
    inst = small_mip(seed=n, m=2 * n, n=n, len_hi=9)
    base = oracle.jacobi(inst) if n < 30000 else (inst.lb, inst.ub)
    rng = np.random.default_rng(n)
    p = I.Problem(inst)
    server = I.Server(p, 4 << 30, slots)
    try:
        server.set_base(base[0], base[1])
        print(f"server changes: n={n} slots={server.slots}", flush=True)
        want = []
        for k in range(2 * slots if n < 30000 else slots):
            l, u, cols = tighten_node(inst, rng, 1, 9, base[0], base[1])
            exp = oracle.jacobi(inst.with_bounds(l, u))
            if n == 30000:  # the base is no fixpoint: every row in round 1
                want.append((server.submit(l, u), True, exp))
            elif k % 3 == 2:
                want.append((server.submit(l, u, hints=cols), True, exp))
            else:
                want.append((server.submit_delta(cols, l[cols], u[cols]), False, exp))
        if n == 30000:
            every = np.arange(n, dtype=np.int32)
            want.append((server.submit_delta(every, inst.lb, inst.ub), False, oracle.jacobi(inst)))
            assert int(np.sum((want[-1][2][0] != inst.lb) | (want[-1][2][1] != inst.ub))) > 4096
        while server.pending():
            server.step()
        for ticket, full, exp in want:
            if full:
                got = server.result(ticket)
                lb, ub, info = got.lbs, got.ubs, got
            else:
                cols, cl, cu, info = server.result_changes(ticket)
                lb, ub = base[0].copy(), base[1].copy()
                lb[cols], ub[cols] = cl, cu
                assert len(np.unique(cols)) == len(cols)
            np.testing.assert_array_equal(lb, exp[0])
            np.testing.assert_array_equal(ub, exp[1])
            assert (info.rounds, bool(info.infeasible), bool(info.capped)) == exp[2:]
    finally:
        server.close()
        p.close()
