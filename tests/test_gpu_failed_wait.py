"""A wait inside a launch that is given up (here because the bound of waits is
0 us, so that every kernel still ends normally) is an error that leaves the
caller's vectors as they were; the same problem then propagates through
launches that do not wait."""
import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import powerlaw_mip, small_mip

pytestmark = pytest.mark.gpu


@pytest.fixture
def no_waiting(monkeypatch):
    monkeypatch.setenv("GDP_WAIT_US", "0")


def _fails_and_recovers(run, lb, ub, want, label):
    dl, du = I.DeviceArray(lb), I.DeviceArray(ub)
    try:
        print(label, flush=True)
        with pytest.raises(RuntimeError, match="wait timed out"):
            run(dl.ptr, du.ptr, I.MEGAKERNEL)
        np.testing.assert_array_equal(dl.numpy(), lb, err_msg=label)
        np.testing.assert_array_equal(du.numpy(), ub, err_msg=label)
        run(dl.ptr, du.ptr, I.CPU_LOOP)
        np.testing.assert_array_equal(dl.numpy(), want[0], err_msg=label)
        np.testing.assert_array_equal(du.numpy(), want[1], err_msg=label)
    finally:
        dl.free()
        du.free()


# the rounds' barrier, without and with split rows, and the three phases'
@pytest.mark.parametrize("tuning", [None, {"item_nnz": 1024}], ids=["rounds", "three phases"])
@pytest.mark.parametrize("make", [lambda: small_mip(seed=3, m=60_000, n=30_000),
                                  lambda: powerlaw_mip(seed=5, m=60_000, n=30_000, len_hi=3000, s=1.8)],
                         ids=["short rows", "split rows"])
def test_single(gpu, oracle, no_waiting, make, tuning):
    inst = make()
    want = oracle.jacobi(inst)
    p = I.Problem(inst, tuning)
    try:
        _fails_and_recovers(p.propagate_device, inst.lb, inst.ub, want, f"{inst.name} {tuning}")
        _fails_and_recovers(p.propagate_device_no_alloc, inst.lb, inst.ub, want, f"{inst.name} {tuning} no alloc")
    finally:
        p.close()


@pytest.mark.parametrize("tuning", [None, {"item_nnz": 1024}], ids=["rounds", "three phases"])
def test_batch(gpu, oracle, no_waiting, tuning):
    xs = [small_mip(seed=k, m=20_000 + k, n=9000) for k in range(5)]
    lb, ub = np.concatenate([x.lb for x in xs]), np.concatenate([x.ub for x in xs])
    exp = [oracle.jacobi(x) for x in xs]
    want = [np.concatenate([e[k] for e in exp]) for k in (0, 1)]
    b = I.Batch(xs, tuning)
    try:
        _fails_and_recovers(b.propagate_device, lb, ub, want, f"batch {tuning}")
    finally:
        b.close()


def test_nodes(gpu, oracle, no_waiting):
    inst, count = small_mip(seed=9, m=20_000, n=9000), 20
    exp = oracle.jacobi(inst)
    p = I.Problem(inst)

    def run(lp, up, sync):
        ptrs = [[q + 8 * inst.n * k for k in range(count)] for q in (lp, up)]
        p.propagate_nodes_device(ptrs[0], ptrs[1], None, sync)

    try:
        p.reserve(count)
        _fails_and_recovers(run, np.tile(inst.lb, count), np.tile(inst.ub, count),
                            [np.tile(exp[k], count) for k in (0, 1)], "nodes")
    finally:
        p.close()
