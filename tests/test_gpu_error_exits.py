"""What a stepping call leaves when it fails: refreshed ghosts, as when it
succeeds.  Failures are the ordinary ones of the main loop (dt below dt_min, a
step redone too often), at the first step and after completed ones."""
import numpy as np
import pytest

import piernik_amd as pk
from piernik_amd import setups

pytestmark = pytest.mark.gpu

# dt_max_grow = 0.5 halves each step's dt: a limit under the second dt fails there
FAILS = {"first step": dict(dt_initial=1e-4, dt_min=1e-3), "second step": dict(dt_initial=1e-4, dt_max_grow=0.5, dt_min=7e-5)}


def block(cfg, seed=3):
    """A block whose ghosts are not the periodic images of its interior."""
    cg = setups.smooth_random((12, 9, 10), nb=4, seed=seed, magnetized=cfg.magnetized, gamma=cfg.gamma)
    for a in (cg.u, cg.b):
        if a is not None:
            a[:, :4] *= 1.25
            a[:, :, -4:] *= 1.5
    return cg


def arrays(cg):
    return [a for a in (cg.u, cg.b, cg.psi) if a is not None]


def assert_periodic(cg):
    was = [a.copy(order="F") for a in arrays(cg)]
    setups.fill_ghosts_periodic(cg)
    for a, o in zip(arrays(cg), was):
        assert np.array_equal(a, o)


def start(cfg):
    pk.load_library()
    pk.finalize()
    pk.init(cfg)


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("fail", sorted(FAILS))
def test_run_leaves_refreshed_ghosts(fail, mag, order):
    cfg = pk.Config(magnetized=mag, limiter="vanleer", integration_order=order, smalld=1e-6, smallei=1e-6)
    print(f"run fails at the {fail}, magnetized {mag}, order {order}", flush=True)
    start(cfg)
    cg = block(cfg)
    before = cg.u.copy()
    cg.upload()
    pk.set_time_control(**FAILS[fail])
    with pytest.raises(pk.PiernikError, match="below dt_min"):
        pk.run(cg, 3)
    cg.download()
    inner = (slice(None), slice(4, -4), slice(4, -4), slice(4, -4))
    assert np.array_equal(cg.u[inner], before[inner]) == (fail == "first step")
    assert_periodic(cg)
    # what reads the ghosts next computes from those: as from the same state uploaded
    left = [a.copy() for a in arrays(cg)]
    out = []
    for again in (False, True):
        if again:
            for a, o in zip(arrays(cg), left):
                a[...] = o
            cg.upload()
        pk.fluid_update(cg, 1e-4)
        cg.download()
        out.append([a.copy() for a in arrays(cg)])
    for a, o in zip(*out):
        assert np.array_equal(a, o)
    pk.finalize()


def test_redone_too_often_leaves_refreshed_ghosts():
    from floors_setup import floor_block

    cg, cfg = floor_block(magnetized=True)
    start(cfg)
    pk.set_cfl_control("redo", cfl_max=0.95, max_redostep_attempts=2, disallow_negatives=True)
    cg.upload()
    print("redone too often", flush=True)
    with pytest.raises(pk.PiernikError, match="max_redostep_attempts"):
        pk.run(cg, 2)
    cg.download()
    was = [a.copy(order="F") for a in arrays(cg)]
    setups.fill_ghosts_periodic(cg)
    for a, o in zip(arrays(cg), was):
        assert np.array_equal(a, o, equal_nan=True)
    pk.finalize()


@pytest.mark.parametrize("linked", [False, True])
@pytest.mark.parametrize("fail", sorted(FAILS))
def test_list_run_leaves_refreshed_ghosts(fail, linked):
    """Two blocks, each periodic on itself or side by side along x."""
    cfg = pk.Config(limiter="vanleer", smalld=1e-6, smallei=1e-6)
    print(f"list run fails at the {fail}, linked {linked}", flush=True)
    start(cfg)
    cgs = [block(cfg, seed=s) for s in (3, 4)]
    for cg in cgs:
        cg.upload()
    if linked:
        for cg, o in zip(cgs, cgs[::-1]):
            for side in (0, 1):
                pk.set_neighbour(cg, 0, side, o)
    pk.set_time_control(**FAILS[fail])
    with pytest.raises(pk.PiernikError, match="below dt_min"):
        pk.run_all(3)
    for cg in cgs:
        cg.download()
    if not linked:
        for cg in cgs:
            assert_periodic(cg)
    else:
        for cg, o in zip(cgs, cgs[::-1]):
            inner = (slice(None), slice(None), slice(4, -4), slice(4, -4))
            assert np.array_equal(cg.u[inner][:, :4], o.u[inner][:, -8:-4])
            assert np.array_equal(cg.u[inner][:, -4:], o.u[inner][:, 4:8])
    pk.finalize()
