"""Which ghosts are old is tracked by the block list, by single blocks and by
saved states; these calls hand a state from one to another.  Every route ends
in a download, whose ghosts have to be the periodic images of its interior, and
in the state that the single-block calls give, bit for bit."""
import ctypes

import numpy as np
import pytest

import piernik_amd as pk
from piernik_amd import setups

pytestmark = pytest.mark.gpu

SHAPES = [(12, 9, 10), (8, 16, 4)]
DTS = [2e-3, 1e-3]
NSW = 6


def start(mag):
    cfg = pk.Config(magnetized=mag, limiter="vanleer", smalld=1e-6, smallei=1e-6)
    pk.load_library()
    pk.finalize()
    pk.init(cfg)
    cgs = [setups.smooth_random(n, nb=4, seed=sum(n), magnetized=mag, gamma=cfg.gamma) for n in SHAPES]
    for cg in cgs:
        cg.upload()
        pk.update_boundaries(cg)
        pk._call("pk_adjoint_setup", cg.cg_id, NSW + 1)
    return cgs


def arrays(cg):
    return [a for a in (cg.u, cg.b, cg.psi) if a is not None]


def got(cg):
    cg.download()
    was = [a.copy(order="F") for a in arrays(cg)]
    setups.fill_ghosts_periodic(cg)
    for a, o in zip(arrays(cg), was):
        assert np.array_equal(a, o), "ghosts are not the images of the interior"
    return was


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def dts():
    return (ctypes.c_double * len(DTS))(*DTS)


def block_states(mag):
    """Per block: the states before sweeps 0..5 of a recorded step, and after it."""
    out = []
    cgs = start(mag)
    for cg, dt in zip(cgs, DTS):
        pk._call("pk_fluid_update_record", cg.cg_id, 0, dt)
        end = got(cg)
        states = []
        for k in range(NSW):
            pk._call("pk_state_load", cg.cg_id, k)
            states.append(got(cg))
        out.append(states + [end])
    pk.finalize()
    return out


@pytest.mark.parametrize("mag", [False, True])
def test_recorded_slots_through_every_load(mag):
    print(f"recorded slots, magnetized {mag}", flush=True)
    ref = block_states(mag)
    cgs = start(mag)
    # the ensemble's record: its final state, then each slot loaded block by block
    pk._call("pk_ensemble_record_step", dts(), 0)
    pk._call("pk_ensemble_state_save", NSW)
    for i, cg in enumerate(cgs):
        assert same(got(cg), ref[i][NSW])
        for k in range(NSW):
            pk._call("pk_state_load", cg.cg_id, k)
            assert same(got(cg), ref[i][k])
    # ... and by the ensemble, slot NSW saved while the ghosts were old
    for k in (3, 0, NSW, 5):
        pk._call("pk_ensemble_state_load", k)
        for i, cg in enumerate(cgs):
            assert same(got(cg), ref[i][k])
    # a block's own record loaded by the ensemble
    pk._call("pk_ensemble_state_load", 0)
    for cg, dt in zip(cgs, DTS):
        pk._call("pk_fluid_update_record", cg.cg_id, 0, dt)
    pk._call("pk_ensemble_state_load", 4)
    for i, cg in enumerate(cgs):
        assert same(got(cg), ref[i][4])
    pk.finalize()


@pytest.mark.parametrize("mag", [False, True])
def test_steps_after_loads(mag):
    """Single-block calls, which read ghosts, after list calls and loads that
    leave them old: each equals the same call on a freshly uploaded copy."""
    print(f"steps after loads, magnetized {mag}", flush=True)

    def routes(cgs):
        cg = cgs[0]
        pk._call("pk_ensemble_record_step", dts(), 0)
        yield "record", cg
        pk._call("pk_state_load", cg.cg_id, 3)
        yield "state_load", cg
        pk._call("pk_ensemble_state_load", 5)
        yield "ensemble_state_load", cgs[1]
        pk.run_all(1)
        yield "run_all", cg
        pk._call("pk_ensemble_run", pk.BATCH_GRAPH, 2, None, None)
        yield "ensemble_run", cgs[1]
        pk.run(cg, 1)
        pk.fluid_update_all(1e-3)
        yield "fluid_update_all", cg

    def sweep_of(k, reupload):
        cgs = start(mag)
        for i, (name, cg) in enumerate(routes(cgs)):
            if i < k:
                continue
            if reupload:
                cg.download()
                setups.fill_ghosts_periodic(cg)
                cg.upload()
            pk.sweep(cg, 1, 5e-4, 1.3)
            cg.download()
            out = [np.array(cg.interior(a)) for a in arrays(cg)]
            pk.finalize()
            return name, out

    for k in range(6):
        name, a = sweep_of(k, False)
        _, b = sweep_of(k, True)
        assert same(a, b), name


def test_failed_record_step_leaves_the_next_steps_right():
    """A record that runs out of slots is refused before its first sweep: the
    states and their ghosts are as they were, and later steps unaffected."""
    ref = start(False)
    t_ref, dt_ref = (ctypes.c_double * 2)(), (ctypes.c_double * 2)()
    pk._call("pk_ensemble_run", pk.BATCH_GRAPH, 2, t_ref, dt_ref)
    want = [got(cg) for cg in ref]
    cgs = start(False)
    for slot0 in (3, NSW + 1, -1):
        with pytest.raises(pk.PiernikError, match="slot"):
            pk._call("pk_ensemble_record_step", dts(), slot0)
    t, dt = (ctypes.c_double * 2)(), (ctypes.c_double * 2)()
    pk._call("pk_ensemble_run", pk.BATCH_GRAPH, 2, t, dt)
    assert list(t) == list(t_ref) and list(dt) == list(dt_ref)
    for cg, w in zip(cgs, want):
        assert same(got(cg), w)
    pk.finalize()


@pytest.mark.parametrize("mag", [False, True])
def test_record_step_reads_the_ghosts_it_is_given(mag):
    """Recorded steps linearise about the state as it is: the first sweep of an
    ensemble's record reads the ghosts a caller has set, as the block's does."""
    print(f"record from given ghosts, magnetized {mag}", flush=True)
    out = []
    for ens in (False, True):
        cgs = start(mag)
        for cg in cgs:
            for a in arrays(cg)[:2]:
                a[:, :4] *= 1.25
            cg.upload()
        if ens:
            pk._call("pk_ensemble_record_step", dts(), 0)
        else:
            for cg, dt in zip(cgs, DTS):
                pk._call("pk_fluid_update_record", cg.cg_id, 0, dt)
        out.append([got(cg) for cg in cgs])
        # later steps read the interior again
        pk._call("pk_ensemble_run", pk.BATCH_GRAPH, 1, None, None)
        out[-1] += [got(cg) for cg in cgs]
        pk.finalize()
    for a, b in zip(*out):
        assert same(a, b)
