"""Batches in double-buffered rounds (default tuning, up to 256 instances):
every instance bit for bit the round-synchronous oracle's, and the same as in
the three-phase rounds, which an explicit work-item size selects.

Sizes: the number of instances around a word of the barrier's bits (31, 62), a
wave (64), the largest batch of the rule and the first one beyond it (256,
257); instances that stop in different rounds, cross their bounds in different
rounds, are crossed on entry, and are stopped by a cap; split rows.
"""
import numpy as np
import pytest

import fixtures
from gdp_amd import interface as I
from gdp_amd.instances import powerlaw_mip, small_mip

pytestmark = pytest.mark.gpu

SYNCS = [I.CPU_LOOP, I.GPU_LOOP, I.MEGAKERNEL]
THREE_PHASES = {"item_nnz": 1024}


def _check(instances, exp, max_rounds=100, tunings=(None,), syncs=SYNCS):
    for tuning in tunings:
        p = I.Batch(instances, tuning)
        try:
            for sync in syncs:
                for again in range(2):
                    got = p.propagate(sync_type=sync, max_rounds=max_rounds)
                    for i, (g, e) in enumerate(zip(got, exp)):
                        label = f"instance {i} of {len(instances)} tuning={tuning} sync={sync} cap={max_rounds}"
                        np.testing.assert_array_equal(g.lbs, e[0], err_msg=label)
                        np.testing.assert_array_equal(g.ubs, e[1], err_msg=label)
                        assert (g.rounds, g.infeasible, g.capped) == e[2:], label
        finally:
            p.close()


def _mixture():
    """Uneven instances: long and short runs, split rows, crossings."""
    out = [small_mip(seed=k, m=40 + 37 * k, n=30 + 17 * k) for k in range(6)]
    out += [fixtures.infeasible_instance(), fixtures.int32_overflow(), powerlaw_mip(seed=5, m=900, n=700, len_hi=650, s=1.6)]
    out += [fixtures.tiny_integer(s) for s in (3, 11, 4)] + [fixtures.varied(2), small_mip(seed=77, m=2500, n=900)]
    return out


@pytest.mark.parametrize("count", [1, 2, 31, 32, 62, 63, 64, 65, 256, 257])
def test_number_of_instances(gpu, oracle, count):
    pool = [small_mip(seed=k, m=5 + 11 * k, n=4 + 7 * k) for k in range(12)]
    exp = [oracle.jacobi(x) for x in pool]
    print(f"batch rounds: {count} instances", flush=True)
    _check([pool[(5 * k) % 12] for k in range(count)], [exp[(5 * k) % 12] for k in range(count)])


def test_uneven_instances_and_every_cap(gpu, oracle):
    mix = _mixture()
    exp = [oracle.jacobi(x) for x in mix]
    _check(mix, exp, tunings=(None, THREE_PHASES))
    for cap in [1, 2, 3, 4, 5] + sorted({e[2] + d for e in exp for d in (-1, 0, 1) if 5 < e[2] + d <= 100}):
        print(f"batch rounds: cap {cap}", flush=True)
        _check(mix, [oracle.jacobi(x, max_rounds=cap) for x in mix], max_rounds=cap)


def test_crossed_on_entry_and_outside_the_envelope(gpu, oracle):
    mix = _mixture()
    exp = [oracle.jacobi(x) for x in mix]
    for tuning in (None, THREE_PHASES):
        p = I.Batch(mix, tuning)
        try:
            for sync in SYNCS:
                lbs, ubs = [x.lb.copy() for x in mix], [x.ub.copy() for x in mix]
                j = int(np.flatnonzero(mix[2].vartype == 3)[0])
                lbs[2][j], ubs[2][j] = 2.0, 1.0
                got = p.propagate(lbs, ubs, sync)
                assert got[2].infeasible
                for i, (g, e) in enumerate(zip(got, exp)):
                    if i == 2:
                        continue
                    np.testing.assert_array_equal(g.lbs, e[0])
                    np.testing.assert_array_equal(g.ubs, e[1])
                    assert (g.rounds, g.infeasible, g.capped) == e[2:]
                whole = np.flatnonzero((mix[3].vartype != 3) & (mix[3].ub < 1e4) & (mix[3].lb > -1e4))
                lbs, ubs = [x.lb.copy() for x in mix], [x.ub.copy() for x in mix]
                ubs[3][int(whole[0])] = 40000.0  # beyond an int16 record
                with pytest.raises(RuntimeError, match="envelope"):
                    p.propagate(lbs, ubs, sync)
        finally:
            p.close()
