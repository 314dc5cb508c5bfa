"""Unsplit tiles at their edges: pencils shorter than the halo needs, lengths
either side of a chunk (28 cells along y and z), pencils that leave the last
tile partly empty, ghosts read from their pre-images, and the timestep and psi
factors folded into the passes.  Bit for bit against the oracle, through
whole runs and through single steps from ghosts that are not periodic images
(a step reads the ghosts it is given)."""
import numpy as np
import pytest

import piernik_amd as pk
from piernik_amd import setups

pytestmark = pytest.mark.gpu

CASES = [((4, 4, 4), (True, True, True)), ((5, 29, 7), (True, True, True)), ((61, 6, 28), (True, True, True)),
         ((9, 57, 1), (True, True, False)), ((253, 1, 1), (True, False, False))]


def assert_same(cg, ob, where):
    for name in ("u", "b", "psi"):
        a, o = getattr(cg, name), getattr(ob, name)
        if a is None:
            continue
        bad = np.argwhere(~(a == o))
        assert bad.size == 0, f"{where} {name}: {len(bad)} differ, first at {tuple(bad[0])}"


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("n,has_dir", CASES)
def test_run_bit_exact(oracle, n, has_dir, mag):
    cfg = pk.Config(magnetized=mag, limiter="vanleer", cfl=0.3, smalld=1e-10, smallei=1e-10, has_dir=has_dir)
    cg = setups.smooth_random(n, seed=sum(n), magnetized=mag, has_dir=has_dir)
    if mag:
        cg.psi[...] = np.random.default_rng(4).normal(0, 0.01, cg.psi.shape)
    setups.fill_ghosts_periodic(cg)
    print(f"unsplit {n} magnetized {mag}", flush=True)
    pk.load_library()
    pk.finalize()
    pk.init(cfg)
    ob = oracle.OBlock.from_cg(cg)
    p = oracle.params_from_config(cfg)
    cg.upload()
    t_g, n_g = pk.run_unsplit(cg, 1.0, nmax=3)
    t_o, n_o = oracle.run_unsplit(p, ob, 1.0, nmax=3)
    cg.download()
    assert (t_g, n_g) == (t_o, n_o)
    assert_same(cg, ob, f"{n}")
    # the timestep the last pass reduced is that of the state it left
    pending = pk.timestep_fluid(cg)
    cg.upload()
    assert pk.timestep_fluid(cg) == pending
    pk.finalize()


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("n,has_dir", CASES)
def test_relaxed_steps_take_the_exact_timestep(n, has_dir, mag):
    """The timestep after relaxed steps is the exact formula of the state they
    left: what the exact build gives for that state."""
    print(f"unsplit timestep {n} magnetized {mag}", flush=True)
    cg = setups.smooth_random(n, seed=sum(n), magnetized=mag, has_dir=has_dir)
    got = []
    for fast in (True, False):
        cfg = pk.Config(magnetized=mag, limiter="vanleer", cfl=0.3, has_dir=has_dir, fast_math=fast)
        pk.load_library()
        pk.finalize()
        pk.init(cfg)
        if not fast:
            cg = copy_of(cg)
        cg.upload()
        if fast:
            pk.run_unsplit(cg, 1.0, nmax=2)
        got.append(pk.timestep_fluid(cg))
        cg.download()
        pk.finalize()
    assert got[0] == got[1]


def copy_of(cg):
    """The block's arrays in a block that is not registered."""
    out = pk.GridContainer(cg.n, nb=cg.nb, dl=cg.dl, magnetized=cg.b is not None, has_dir=cg.has_dir)
    for a, o in zip((out.u, out.b, out.psi), (cg.u, cg.b, cg.psi)):
        if a is not None:
            a[...] = o
    return out


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("n", [(12, 9, 8), (5, 33, 4)])
def test_step_reads_the_ghosts_it_is_given(oracle, n, mag):
    """One step from ghosts that are not the periodic images of the interior,
    on every face and in every variable: the first stage reads them as they
    are, psi damped with the rest, and the step leaves refreshed ones -- every
    cell of the oracle's step, which refreshes after each stage only."""
    cfg = pk.Config(magnetized=mag, limiter="vanleer", smalld=1e-10, smallei=1e-10)
    print(f"unsplit step from given ghosts {n} magnetized {mag}", flush=True)
    cg = setups.smooth_random(n, seed=3, magnetized=mag)
    rng = np.random.default_rng(8)
    if mag:
        cg.psi[...] = rng.normal(0, 0.01, cg.psi.shape)
    setups.fill_ghosts_periodic(cg)
    for a in (cg.u, cg.b, cg.psi):
        if a is not None:
            inner = np.array(cg.interior(a))
            a *= rng.uniform(1.0, 1.1, a.shape)
            cg.interior(a)[...] = inner
    pk.load_library()
    pk.finalize()
    pk.init(cfg)
    ob = oracle.OBlock.from_cg(cg)
    cg.upload()
    pk.fluid_update_unsplit(cg, 1e-3)
    oracle.fluid_update_unsplit(oracle.params_from_config(cfg), ob, 1e-3)
    cg.download()
    assert_same(cg, ob, f"{n}")
    pk.finalize()
