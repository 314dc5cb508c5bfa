"""Sweep tiles at their edges: lengths either side of where the default shape
changes (whole pencil, two chunks, three pencils a tile, few pencils), blocks
as short as their ghosts (every halo is read from its pre-image in the
interior, which wraps more than once), pencils that leave the last tile
partly empty, and lists whose launches have fewer items than CUs.

Bit for bit against the oracle, as the rest of the exact build.  A pinned
tile runs beside the default: a tile changes who computes a cell, never how.
"""
import ctypes

import numpy as np
import pytest

import piernik_amd as pk
from piernik_amd import setups

pytestmark = pytest.mark.gpu

# (shape, active directions)
BLOCKS = [((4, 4, 4), (True, True, True)), ((5, 4, 9), (True, True, True)), ((77, 6, 5), (True, True, True)),
          ((6, 78, 5), (True, True, True)), ((249, 4, 4), (True, True, True)), ((7, 5, 57), (True, True, True)),
          ((40, 36, 33), (True, True, True)), ((124, 5, 1), (True, True, False)), ((9, 65, 1), (True, True, False)),
          ((300, 1, 1), (True, False, False))]


def assert_same(cg, ob, where):
    for name in ("u", "b", "psi"):
        a, o = getattr(cg, name), getattr(ob, name)
        if a is None:
            continue
        bad = np.argwhere(~(a == o))
        assert bad.size == 0, f"{where} {name}: {len(bad)} differ, first at {tuple(bad[0])}"


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("shape,has_dir", BLOCKS)
def test_block_tiles_bit_exact(oracle, shape, has_dir, mag):
    out = None
    # default; tiles of one and several pencils; (1D: no y, z); whole pencils (march); streams
    for tile in [(0, 0), (1, 9), (7, 23), (64, -1), (2, -3)]:
        cfg = pk.Config(magnetized=mag, limiter="vanleer", smalld=1e-3, smallei=1e-4, has_dir=has_dir,
                        tile_x=tile, tile_yz=tile)
        print(f"block {shape} magnetized {mag} tile {tile}", flush=True)
        pk.load_library()
        pk.finalize()
        pk.init(cfg)
        cg = setups.smooth_random(shape, nb=4, seed=sum(shape), magnetized=mag, gamma=cfg.gamma, has_dir=has_dir)
        if out is None:
            out = oracle.OBlock.from_cg(cg)
            t_o = oracle.run(oracle.params_from_config(cfg), out, 2)
        cg.upload()
        t_g, _ = pk.run(cg, 2)
        cg.download()
        assert t_g == t_o
        assert_same(cg, out, f"{shape} {tile}")
        pk.finalize()


@pytest.mark.parametrize("lanes,ts", [(0, 0), (64, -2), (128, 0), (256, 9), (512, 0)])
@pytest.mark.parametrize("shapes", [[(4, 4, 4)], [(5, 6, 4), (33, 30, 34), (4, 77, 5)]])
def test_list_items_bit_exact(oracle, shapes, lanes, ts):
    cfg = setups.batch_config(fluids=((5.0 / 3.0, True), (1.4, False)))
    cgs = setups.batch_blocks(shapes, cfg, seed=5)
    obs = [oracle.OBlock.from_cg(c) for c in cgs]
    print(f"list {shapes} lanes {lanes} ts {ts}", flush=True)
    pk.load_library()
    pk.finalize()
    pk.init(cfg)
    for cg in cgs:
        cg.registered = False
        cg.upload()
    if lanes:
        for d in range(3):
            for f in range(2):
                pk.set_list_tiles(d, f, lanes, ts)
    t_g, _ = pk.run_all(2)
    assert t_g == oracle.run_list(oracle.params_from_config(cfg), obs, 2)
    for cg, ob in zip(cgs, obs):
        cg.download()
        assert_same(cg, ob, f"list {cg.n}")
    pk.finalize()


# Pencils of two blocks, in stream items of one pencil group each: a group is a
# pencil along x and eight along y and z.
STREAM_LISTS = {2900: ((44, 41), (33, 33)), 4300: ((60, 45), (40, 40)), 5700: ((75, 48), (50, 42))}


@pytest.mark.parametrize("items", sorted(STREAM_LISTS))
@pytest.mark.parametrize("d", [0, 1, 2])
def test_stream_ranges_of_several_items_bit_exact(oracle, d, items):
    """More items than workgroups the device holds (2048 at two waves per SIMD,
    3072 at three, 4096 at four), by less than half: the launch has one round of
    workgroups, whose ranges hold one or two items, join items of a block, and
    cross from one block to the next."""
    cfg = setups.batch_config(fluids=((5.0 / 3.0, True), (1.4, False)))
    shapes = []
    for (a, b), length in zip(STREAM_LISTS[items], (125, 121) if d == 0 else (5, 7)):
        n = [a, b] if d == 0 else [4 * a, 2 * b]
        n.insert(d, length)
        shapes.append(tuple(n))
    shapes.append((4, 4, 4))
    print(f"stream list of {items} items along {'xyz'[d]}: {shapes}", flush=True)
    cgs = setups.batch_blocks(shapes, cfg, seed=5)
    obs = [oracle.OBlock.from_cg(c) for c in cgs]
    pk.load_library()
    pk.finalize()
    pk.init(cfg)
    for cg in cgs:
        cg.registered = False
        cg.upload()
    for f in range(2):
        pk.set_list_tiles(d, f, 64, -2)
    t_g, _ = pk.run_all(1)
    assert t_g == oracle.run_list(oracle.params_from_config(cfg), obs, 1)
    for cg, ob in zip(cgs, obs):
        cg.download()
        assert_same(cg, ob, f"list {cg.n}")
    pk.finalize()


def test_list_of_several_launches():
    """More tiles than one launch takes (2^22): one cell and 14 pencils a tile
    against the default tiles, the same bits."""
    torch = pytest.importorskip("torch")
    n = 400
    print(f"list of {n}^3 cells in tiles of 14", flush=True)
    cfg = pk.Config(limiter="vanleer", gamma=1.4)
    gen = torch.Generator(device="cuda").manual_seed(1)
    u = torch.empty((n + 8, n + 8, n + 8, 5), dtype=torch.float64, device="cuda")
    u.uniform_(-0.3, 0.3, generator=gen)
    u[..., 0] += 1.0
    u[..., 4] += 3.0
    out = []
    for ts in (0, 9):
        pk.load_library()
        pk.finalize()
        pk.init(cfg)
        cg = setups._DeviceBlock((n, n, n), 4, cfg, 1)
        cg.upload_device(u)
        if ts:
            for d in range(3):
                pk.set_list_tiles(d, 0, 128, ts)
        pk.run_all(1)
        out.append(torch.empty_like(u))
        cg.download_device(out[-1])
        pk.finalize()
    assert torch.equal(out[0], out[1]) and bool(torch.isfinite(out[0]).all())


@pytest.mark.parametrize("n", [(12, 9, 8), (5, 4, 33)])
def test_step_reads_the_ghosts_it_is_given(n):
    """A single step from ghosts that are not periodic images: its first sweep
    reads them as they are, the later ones see refreshed ghosts; sweep by
    sweep with refreshes in between gives the same bits."""
    cfg = pk.Config(limiter="vanleer", smalld=1e-3, smallei=1e-4)
    out = []
    for whole in (True, False):
        pk.load_library()
        pk.finalize()
        pk.init(cfg)
        cg = setups.smooth_random(n, nb=4, seed=7, gamma=cfg.gamma)
        cg.u[:, :4] *= 1.25
        cg.upload()
        if whole:
            pk.fluid_update(cg, 1e-3)
        else:
            for d in (0, 1, 2, 2, 1, 0):
                pk.sweep(cg, d, 1e-3)
                pk.update_boundaries(cg)
        cg.download()
        out.append(cg.u.copy())
        pk.finalize()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("mode", [pk.BATCH_GRAPH, pk.BATCH_PERSISTENT, pk.BATCH_PER_BLOCK])
def test_ensemble_steps_refresh_the_ghosts(mode):
    """An ensemble's steps take each block as periodic, whatever its ghosts
    hold: an ensemble of one from ghosts that are not periodic images equals
    fluid_update with the same dt from refreshed ones, at the first step and
    after it."""
    cfg = pk.Config(limiter="vanleer", smalld=1e-3, smallei=1e-4)
    out, dts = [], []
    for ens in (True, False):
        pk.load_library()
        pk.finalize()
        pk.init(cfg)
        cg = setups.smooth_random((12, 9, 8), nb=4, seed=7, gamma=cfg.gamma)
        cg.u[:, :4] *= 1.25
        cg.upload()
        if not ens:
            pk.update_boundaries(cg)
        for s in range(2):
            if ens:
                dt, cap = (ctypes.c_double * 1)(), (ctypes.c_int32 * 1)()
                pk._call("pk_ensemble_step", int(mode), int(s == 0), dt, cap)
                dts.append(dt[0])
            else:
                pk.fluid_update(cg, dts[s])
        cg.download()
        out.append(cg.u.copy())
        pk.finalize()
    assert np.array_equal(out[0], out[1])
