"""Layout conversion, ghost refresh and ghost copies at their edges: block
sizes that leave partial workgroups, blocks as short as their ghosts, 1D and
2D, and every number of values a cell has (5, 9, 10 and 14).  All of it moves
or adds values without rounding choices, so results are compared for equality."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import piernik_amd as pk  # noqa: E402
from piernik_amd import setups  # noqa: E402

pytestmark = pytest.mark.gpu

SHAPES = [((4, 4, 4), (True, True, True)), ((33, 5, 7), (True, True, True)), ((6, 61, 4), (True, True, True)),
          ((37, 23, 1), (True, True, False)), ((129, 1, 1), (True, False, False))]
ION, NEU = (5.0 / 3.0, True), (1.4, False)


def block(cfg, shape, has_dir):
    cg = pk.GridContainer(shape, nb=4, dl=tuple(1.0 / s for s in shape), magnetized=cfg.magnetized, has_dir=has_dir,
                          nfluids=cfg.nfluids)
    rng = np.random.default_rng(sum(shape))
    for a in (cg.u, cg.b, cg.psi):
        if a is not None:
            a[...] = rng.uniform(1.0, 2.0, a.shape)
    return cg


@pytest.mark.parametrize("fluids", [(ION,), (NEU,), (ION, NEU), (NEU, NEU)])
@pytest.mark.parametrize("shape,has_dir", SHAPES)
def test_round_trip_and_ghosts(shape, has_dir, fluids):
    cfg = setups.batch_config(fluids=fluids, has_dir=has_dir)
    print(f"layout {shape} fluids {fluids}", flush=True)
    pk.load_library()
    pk.finalize()
    pk.init(cfg)
    cg = block(cfg, shape, has_dir)
    was = [None if a is None else a.copy(order="F") for a in (cg.u, cg.b, cg.psi)]
    cg.upload()
    for a in (cg.u, cg.b, cg.psi):
        if a is not None:
            a[...] = 0.0
    cg.download()
    for a, o in zip((cg.u, cg.b, cg.psi), was):
        assert a is None or np.array_equal(a, o)
    pk.update_boundaries(cg)
    cg.download()
    got = [None if a is None else a.copy(order="F") for a in (cg.u, cg.b, cg.psi)]
    setups.fill_ghosts_periodic(cg)
    for a, o in zip((cg.u, cg.b, cg.psi), got):
        assert a is None or np.array_equal(a, o)
    pk.finalize()


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("shape,has_dir", SHAPES)
def test_adjoint_arrays_fold(shape, has_dir, mag):
    """Ghost values go to the cells they copy: z, then y, then x, the cell's
    own value first, the low ghost before the high one."""
    cfg = pk.Config(magnetized=mag, has_dir=has_dir)
    print(f"fold {shape} magnetized {mag}", flush=True)
    pk.load_library()
    pk.finalize()
    pk.init(cfg)
    cg = setups._DeviceBlock(shape, 4, cfg, 1)
    cg.register()
    pk._call("pk_adjoint_setup", 1, 1)
    ng = cg.ng
    gen = torch.Generator().manual_seed(sum(shape))
    rand = lambda *tail: torch.rand((ng[2], ng[1], ng[0]) + tail, dtype=torch.float64, generator=gen).cuda()
    lam = [rand(5)] + ([rand(3), rand()] if mag else [])
    pk._call("pk_adjoint_set", 1, *(pk._device_ptrs(*lam) + [None] * (3 - len(lam))))
    out = [torch.full_like(t, -1.0) for t in lam]
    pk._call("pk_adjoint_get", 1, *(pk._device_ptrs(*out) + [None] * (3 - len(out))))
    for t, o in zip(lam, out):
        ref = t.cpu().numpy().copy()
        for axis, d in ((0, 2), (1, 1), (2, 0)):
            if not has_dir[d]:
                continue
            a = np.moveaxis(ref, axis, 0)
            n = shape[d]
            inner = a[4:4 + n].copy()
            inner[n - 4:] = inner[n - 4:] + a[:4]
            inner[:4] = inner[:4] + a[4 + n:]
            a[...] = 0.0
            a[4:4 + n] = inner
        assert np.array_equal(o.cpu().numpy(), ref)
    pk.finalize()


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("shape,has_dir", SHAPES)
def test_stage_keeps_the_other_cells(oracle, shape, has_dir, mag):
    """One stage along each direction, ghosts refreshed in between, from a
    state whose ghosts are not periodic images: every cell against the oracle."""
    cfg = pk.Config(magnetized=mag, limiter="vanleer", smalld=1e-3, smallei=1e-4, has_dir=has_dir)
    print(f"stage {shape} magnetized {mag}", flush=True)
    pk.load_library()
    pk.finalize()
    pk.init(cfg)
    cg = setups.smooth_random(shape, nb=4, seed=9, magnetized=mag, gamma=cfg.gamma, has_dir=has_dir)
    cg.u[0] *= np.random.default_rng(2).uniform(1.0, 1.1, cg.u[0].shape)
    ob = oracle.OBlock.from_cg(cg)
    p = oracle.params_from_config(cfg)
    cg.upload()
    for d in range(3):
        if not has_dir[d]:
            continue
        for istep in (pk.RK2_1, pk.RK2_2):
            pk.solve_cg(cg, d, istep, 1e-4, 1.7)
            oracle.solve_cg(p, ob, d, istep, 1e-4, 1.7)
            cg.download()
            for name in ("u", "b", "psi"):
                a, o = getattr(cg, name), getattr(ob, name)
                assert a is None or (a == o).all(), f"direction {d} stage {istep} {name}"
            if d != 1:
                pk.update_boundaries(cg)
                oracle.fill_ghosts(p, ob)
    pk.finalize()
