"""A wait inside a launch that is given up (here because GDP_FAIL_WAITS sets the
error word before the run; every kernel still ends normally) is an error that
leaves the caller's vectors as they were."""
import numpy as np
import pytest

from gdp_amd import interface as I
from gdp_amd.instances import powerlaw_mip, small_mip

pytestmark = pytest.mark.gpu


@pytest.fixture
def no_waiting(monkeypatch):
    monkeypatch.setenv("GDP_FAIL_WAITS", "1")


def _fails(run, lb, ub, label):
    dl, du = I.DeviceArray(lb), I.DeviceArray(ub)
    try:
        print(label, flush=True)
        for sync in (I.MEGAKERNEL, I.CPU_LOOP, I.GPU_LOOP):
            with pytest.raises(RuntimeError, match="wait timed out"):
                run(dl.ptr, du.ptr, sync)
            np.testing.assert_array_equal(dl.numpy(), lb, err_msg=f"{label} sync={sync}")
            np.testing.assert_array_equal(du.numpy(), ub, err_msg=f"{label} sync={sync}")
    finally:
        dl.free()
        du.free()


# the rounds' barrier, without and with split rows, and the three phases'
@pytest.mark.parametrize("tuning", [None, {"item_nnz": 1024}], ids=["rounds", "three phases"])
@pytest.mark.parametrize("make", [lambda: small_mip(seed=3, m=60_000, n=30_000),
                                  lambda: powerlaw_mip(seed=5, m=60_000, n=30_000, len_hi=3000, s=1.8)],
                         ids=["short rows", "split rows"])
def test_single(gpu, no_waiting, make, tuning):
    inst = make()
    p = I.Problem(inst, tuning)
    try:
        _fails(p.propagate_device, inst.lb, inst.ub, f"{inst.name} {tuning}")
        _fails(p.propagate_device_no_alloc, inst.lb, inst.ub, f"{inst.name} {tuning} no alloc")
    finally:
        p.close()


@pytest.mark.parametrize("tuning", [None, {"item_nnz": 1024}], ids=["rounds", "three phases"])
def test_batch(gpu, no_waiting, tuning):
    xs = [small_mip(seed=k, m=20_000 + k, n=9000) for k in range(5)]
    lb, ub = np.concatenate([x.lb for x in xs]), np.concatenate([x.ub for x in xs])
    b = I.Batch(xs, tuning)
    try:
        _fails(b.propagate_device, lb, ub, f"batch {tuning}")
    finally:
        b.close()


def test_nodes(gpu, no_waiting):
    inst, count = small_mip(seed=9, m=20_000, n=9000), 20
    p = I.Problem(inst)

    def run(lp, up, sync):
        ptrs = [[q + 8 * inst.n * k for k in range(count)] for q in (lp, up)]
        p.propagate_nodes_device(ptrs[0], ptrs[1], None, sync)

    try:
        p.reserve(count)
        _fails(run, np.tile(inst.lb, count), np.tile(inst.ub, count), "nodes")
    finally:
        p.close()
