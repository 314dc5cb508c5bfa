"""Timed cases: what a program using this library has it do, end to end.

Every case goes through the Python binding, from the caller's device tensors
in the reference layout to tensors (or, for the output fields, host arrays)
of the results:

  run       one periodic block stepped by pk.run: upload, main loop, download
  stages    the per-block operator as sweep() calls it: both RK2 stages of
            every direction through pk.solve_cg, ghosts refreshed in between
  list      a list of independent uneven two-fluid blocks with one dt (run_all)
  linked    a periodic domain cut into blocks that exchange ghosts (run_all)
  unsplit   the unsplit solver (run_unsplit)
  rollout   value and gradient of a checkpointed rollout (adjoint.rollout)
  ensemble  the same for many independent 2D instances (adjoint.EnsemblePlan)
  fields    the output fields of a snapshot, as 32-bit host arrays

A case is a dict of plain values.  The library holds one configuration and
one block list per process, so the states of one case share its registered
blocks (as a program's successive problems would) and differ in their input
tensors; another case configures the library anew.
"""
import math

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

import piernik_amd as pk
from piernik_amd import adjoint, setups

NB = 4          # ghost layers, as every configuration of this repository
GAMMA = 5.0 / 3.0
LIST_SIZES = (16, 24, 32, 48, 64)    # block edges of the batched list
ENSEMBLE_SIZES = (64, 96, 128, 192, 256)
FIELDS_MHD = ("deni", "vlxi", "vlyi", "vlzi", "enei", "prei", "ethi", "magx", "magy", "magz", "magB", "psi")
FIELDS_HD = ("denn", "vlxn", "vlyn", "vlzn", "enen", "pren", "ethn")


# ---- the cases --------------------------------------------------------------


def listed():
    return [
        # the smallest call: one step of a 16^3 hydro block, where launches and host latency count
        dict(name="step_hd_16", kind="run", field="smooth", nx=16, ny=16, nz=16, mag=False, fast=False, tuned=False,
             limiter="vanleer", steps=1),
        # the 64^3 Sedov blast of the reference's benchmark, default configuration
        dict(name="sedov_hd_64", kind="run", field="sedov", nx=64, ny=64, nz=64, mag=False, fast=False, tuned=False,
             limiter="vanleer", steps=5),
        # a ragged MHD block with the bit-exact arithmetic, shapes left to the library
        dict(name="mhd_ragged_exact", kind="run", field="turbulence", nx=131, ny=98, nz=77, mag=True, fast=False,
             tuned=False, limiter="vanleer", steps=4),
        # the headline workload: 256^3 MHD turbulence, contracted arithmetic, autotuned once
        dict(name="turbulence_256", kind="run", field="turbulence", nx=256, ny=256, nz=256, mag=True, fast=True,
             tuned=True, limiter="minmod", steps=4),
        # the drop-in operator, stage by stage, on an ordinary block
        dict(name="stages_mhd_96", kind="stages", field="turbulence", nx=96, ny=96, nz=96, mag=True, fast=False,
             tuned=False, limiter="vanleer", steps=1),
        # an AMR-like list of uneven two-fluid blocks, autotuned once
        dict(name="list_two_fluid", kind="list", nblocks=144, sizes_seed=0, fast=True, tuned=True, limiter="vanleer",
             steps=4),
        # a periodic domain cut unevenly into linked blocks, bit-exact
        dict(name="linked_mhd_blocks", kind="linked", nx=120, ny=96, nz=80, cx=3, cy=2, cz=2, mag=True, fast=False,
             tuned=False, limiter="minmod", steps=3),
        # the unsplit solver on a 3D block
        dict(name="unsplit_mhd_128", kind="unsplit", field="turbulence", nx=128, ny=128, nz=128, mag=True, fast=True,
             limiter="vanleer", steps=3),
        # gradient of a 3D hydro rollout, checkpointed
        dict(name="rollout_hd_96", kind="rollout", nx=96, ny=96, nz=96, mag=False, limiter="vanleer", steps=4, every=2),
        # gradient of a small 3D MHD rollout of odd sizes
        dict(name="rollout_mhd_45x40x34", kind="rollout", nx=45, ny=40, nz=34, mag=True, limiter="vanleer", steps=3,
             every=3),
        # gradients of many independent 2D MHD problems at once
        dict(name="ensemble_mhd_2d", kind="ensemble", ninst=20, sizes_seed=3, limiter="vanleer", steps=4, every=2),
        # a snapshot's output fields
        dict(name="fields_mhd_112", kind="fields", field="turbulence", nx=112, ny=112, nz=112, mag=True, fast=False,
             limiter="vanleer", steps=1),
    ]


def _edge(rng, lo, hi):
    """An edge length spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "run", "stages", "stages", "list", "linked", "unsplit", "unsplit",
                       "rollout", "rollout", "ensemble", "fields"])
    c = {"kind": kind, "limiter": rng.choice(["vanleer", "vanleer", "minmod", "moncen", "superbee"])}
    mag = rng.random() < 0.6
    if kind in ("run", "stages", "unsplit", "fields"):
        c.update(nx=_edge(rng, 12, 200), ny=_edge(rng, 12, 200), nz=_edge(rng, 12, 200), mag=mag,
                 field=rng.choice(["smooth", "turbulence"]) if mag else rng.choice(["smooth", "sedov"]),
                 fast=rng.random() < 0.5, steps=rng.randint(1, 4))
        if kind in ("run", "stages"):
            c["tuned"] = kind == "run" and rng.random() < 0.4
        if kind == "stages":
            c["fast"] = False
            c["field"] = "smooth" if c["field"] == "sedov" else c["field"]  # their dt is fixed
        if kind in ("unsplit", "run") and rng.random() < 0.2:  # a 2D block
            c.update(nz=1, nx=_edge(rng, 24, 512), ny=_edge(rng, 24, 512), field="smooth")
        if kind == "fields":
            c["steps"] = 1
    elif kind == "list":
        c.update(nblocks=_edge(rng, 4, 144), sizes_seed=rng.randint(0, 999), fast=rng.random() < 0.5,
                 tuned=rng.random() < 0.5, steps=rng.randint(1, 4))
    elif kind == "linked":
        c.update(nx=_edge(rng, 32, 140), ny=_edge(rng, 32, 140), nz=_edge(rng, 32, 140), cx=rng.randint(1, 3),
                 cy=rng.randint(1, 3), cz=rng.randint(2, 3), mag=mag, fast=rng.random() < 0.5, tuned=False,
                 steps=rng.randint(1, 3))
    elif kind == "rollout":
        top = 48 if mag else 96
        steps = rng.randint(2, 5)
        c.update(nx=_edge(rng, 12, top), ny=_edge(rng, 12, top), nz=_edge(rng, 12, top), mag=mag, steps=steps,
                 every=rng.randint(1, steps))
    else:
        steps = rng.randint(2, 4)
        c.update(ninst=_edge(rng, 2, 20), sizes_seed=rng.randint(0, 999), steps=steps, every=rng.randint(1, steps))
    return c


# ---- configuration and blocks, kept for the states of one case ----------------


def _shape(c):
    return (c["nx"], c["ny"], c["nz"])


def _has_dir(c):
    if c["kind"] == "ensemble":
        return (True, True, False)
    return (True, True, c.get("nz", 2) > 1)


def _config(c):
    lim = c["limiter"]
    if c["kind"] == "list":
        cfg = setups.batch_config(limiter=lim)
    else:
        cfl = 0.3 if c["kind"] == "unsplit" else (0.7 if c.get("field") == "sedov" else 0.5)
        mag = c["kind"] == "ensemble" or bool(c["mag"])
        cfg = pk.Config(gamma=GAMMA, magnetized=mag, limiter=lim, limiter_b=lim, cfl=cfl, cfl_glm=cfl, glm_alpha=0.1,
                        smalld=1e-10 if c.get("field") == "sedov" else 1e-4,
                        smallei=1e-10 if c.get("field") == "sedov" else 1e-6, has_dir=_has_dir(c))
    cfg.fast_math = bool(c.get("fast", False))
    return cfg


def _cuts(n, k, nb=NB):
    """k uneven pieces of n cells: cut positions, each piece at least nb wide."""
    w = [2 + (i % 3) for i in range(k)]
    at = [n * sum(w[: i + 1]) // sum(w) for i in range(k - 1)]
    return [max(nb * (i + 1), min(n - nb * (k - 1 - i), a)) for i, a in enumerate(at)]


def _list_sizes(c):
    return setups.batch_sizes(c["nblocks"], seed=c["sizes_seed"], sizes=LIST_SIZES)


def _ensemble_sizes(c):
    rng = np.random.default_rng([c["sizes_seed"], 5555])
    return [int(n) for n in rng.choice(np.asarray(ENSEMBLE_SIZES), size=c["ninst"])]


class _Session:
    """The library configured for one case and its registered blocks."""

    def __init__(self, c):
        self.cfg = cfg = _config(c)
        pk.init(cfg)
        kind = c["kind"]
        self.plan = None
        self.tuned = not c.get("tuned", False)
        if kind == "rollout":
            self.plan = adjoint.RolloutPlan(cfg, _shape(c), c["steps"], checkpoint_every=c["every"])
            self.blocks = [self.plan.cg]
        elif kind == "ensemble":
            self.plan = adjoint.EnsemblePlan(cfg, [(n, n, 1) for n in _ensemble_sizes(c)], c["steps"],
                                             checkpoint_every=c["every"])
            self.blocks = self.plan.blocks
        elif kind == "list":
            self.blocks = [setups._DeviceBlock((n, n, n), NB, cfg, 1 + i) for i, n in enumerate(_list_sizes(c))]
            for b in self.blocks:
                b.register()
        elif kind == "linked":
            n = _shape(c)
            whole = pk.GridContainer(n, nb=NB, dl=tuple(1.0 / max(n) for _ in n), magnetized=cfg.magnetized)
            cuts = [_cuts(n[d], k) for d, k in enumerate((c["cx"], c["cy"], c["cz"]))]
            self.blocks, nbr, self.boxes = setups.decompose(whole, cuts, first_id=1)
            pk.connect(self.blocks, nbr)
        else:
            self.blocks = [setups._DeviceBlock(_shape(c), NB, cfg, 1)]
            self.blocks[0].register()


_open = {"key": None, "session": None}


def _session(c):
    key = tuple(sorted((k, v) for k, v in c.items() if k != "name"))
    if _open["key"] != key:
        _open.update(key=None, session=None)
        _open.update(session=_Session(c), key=key)
    return _open["session"]


# ---- initial states ------------------------------------------------------------


def _waves(shape, gen, n=1):
    """n smooth periodic fields of a few low modes, within [-1, 1]."""
    ax = [2.0 * math.pi * (torch.arange(s, device="cuda", dtype=torch.float64) + 0.5) / s for s in shape]
    out = []
    for _ in range(n):
        f = torch.zeros(shape, device="cuda", dtype=torch.float64)
        k = torch.randint(1, 3, (3, 3), generator=gen).tolist()
        ph = (2.0 * math.pi * torch.rand(3, generator=gen)).tolist()
        for m in range(3):
            kv = [k[m][d] if shape[d] > 1 else 0 for d in range(3)]
            f += torch.sin(kv[0] * ax[0].view(-1, 1, 1) + kv[1] * ax[1].view(1, -1, 1) + kv[2] * ax[2].view(1, 1, -1)
                           + ph[m])
        out.append(f / 3.0)
    return out


def _gaussian(shape, gen, n):
    """n Gaussian random fields, E(k) ~ k^-2 on 1 <= k <= 8, and their spectra."""
    k = [torch.fft.fftfreq(s, d=1.0 / s, device="cuda", dtype=torch.float64) for s in shape]
    kx, ky, kz = torch.meshgrid(*k, indexing="ij")
    k2 = kx * kx + ky * ky + kz * kz
    amp = torch.where((k2 >= 1.0) & (k2 <= 64.0), 1.0 / k2.clamp(min=1.0), torch.zeros_like(k2))
    dev = torch.Generator(device="cuda").manual_seed(int(torch.randint(0, 1 << 31, (1,), generator=gen)))
    out = []
    for _ in range(n):
        white = torch.randn(shape, generator=dev, device="cuda", dtype=torch.float64)
        out.append(torch.fft.fftn(white) * amp)
    return out, (kx, ky, kz)


def _conserved(rho, v, p, b=None):
    e = p / (GAMMA - 1.0) + 0.5 * rho * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2])
    if b is None:
        return [rho, rho * v[0], rho * v[1], rho * v[2], e]
    e = e + 0.5 * (b[0] * b[0] + b[1] * b[1] + b[2] * b[2])
    return [rho, rho * v[0], rho * v[1], rho * v[2], e, b[0], b[1], b[2], torch.zeros_like(rho)]


def _smooth(shape, gen, mag, b0=0.7):
    f = _waves(shape, gen, 8 if mag else 5)
    v = [0.5 * x for x in f[2:5]]
    return _conserved(1.0 + 0.2 * f[0], v, 1.0 + 0.2 * f[1], [b0 * x for x in f[5:8]] if mag else None)


def _initial(c, shape, gen):
    """Interior state of one fluid, a list of 5 or 9 (nx, ny, nz) tensors."""
    mag = c["kind"] == "ensemble" or bool(c["mag"])
    field = c.get("field", "smooth")
    if field == "sedov":
        # a blast of unit energy within three cells of a centre, cold uniform surroundings
        off = (torch.rand(4, generator=gen) - 0.5).tolist()
        ax = [torch.arange(s, device="cuda", dtype=torch.float64) - 0.5 * (s - 1) - off[d] for d, s in enumerate(shape)]
        r2 = ax[0].view(-1, 1, 1) ** 2 + ax[1].view(1, -1, 1) ** 2 + ax[2].view(1, 1, -1) ** 2
        inside = (r2 <= 9.0).to(torch.float64)
        one, zero = torch.ones_like(r2), torch.zeros_like(r2)
        u = _conserved(one, [zero, zero, zero], 1e-5 * one)
        u[4] = u[4] + inside * ((1.0 + 0.2 * off[3]) * r2.numel() / inside.sum())
        return u
    if field == "turbulence":
        vk, (kx, ky, kz) = _gaussian(shape, gen, 6)
        v = [torch.fft.ifftn(x).real for x in vk[:3]]
        s = 1.0 / torch.sqrt(sum((x * x).mean() for x in v))
        a = vk[3:]
        b = [torch.fft.ifftn(1j * x).real for x in (ky * a[2] - kz * a[1], kz * a[0] - kx * a[2], kx * a[1] - ky * a[0])]
        sb = torch.sqrt(1.2 / sum((x * x).mean() for x in b))  # plasma beta 1 at p = 0.6
        one = torch.ones(shape, device="cuda", dtype=torch.float64)
        return _conserved(one, [s * x for x in v], 0.6 * one, [sb * x for x in b])
    if c["kind"] == "ensemble":
        # the Orszag-Tang vortex of this instance's amplitude with smooth perturbations
        amp = 1.0 + 0.2 * (float(torch.rand(1, generator=gen)) - 0.5)
        f = [0.1 * x for x in _waves(shape, gen, 9)]
        x = ((torch.arange(shape[0], device="cuda", dtype=torch.float64) + 0.5) / shape[0]).view(-1, 1, 1)
        y = ((torch.arange(shape[1], device="cuda", dtype=torch.float64) + 0.5) / shape[1]).view(1, -1, 1)
        b0 = 1.0 / math.sqrt(4.0 * math.pi)
        two_pi = 2.0 * math.pi
        v = [f[0] - amp * torch.sin(two_pi * y), f[1] + amp * torch.sin(two_pi * x), f[2]]
        b = [b0 * (f[3] - amp * torch.sin(two_pi * y)), b0 * (f[4] + amp * torch.sin(2 * two_pi * x)), b0 * f[5]]
        u = _conserved(25.0 / (36.0 * math.pi) * (1.0 + f[6]), v, 5.0 / (12.0 * math.pi) * (1.0 + f[7]), b)
        u[8] = b0 * f[8]
        return u
    return _smooth(shape, gen, mag)


def _pad(x, has_dir):
    """Periodic ghost layers on the last three axes."""
    for d in range(3):
        if has_dir[d]:
            ax = x.dim() - 3 + d
            x = torch.cat([x.narrow(ax, x.shape[ax] - NB, NB), x, x.narrow(ax, 0, NB)], dim=ax)
    return x


def _arrays(fluids, has_dir):
    """Interior fluids (lists of 5 or 9 tensors) -> u, b, psi tensors in the
    reference layout, ghosts included: (nzg, nyg, nxg, nvar), (nzg, nyg, nxg, 3), (nzg, nyg, nxg)."""
    u = torch.stack([_pad(x, has_dir) for f in fluids for x in f[:5]]).permute(3, 2, 1, 0).contiguous()
    mag = next((f for f in fluids if len(f) == 9), None)
    if mag is None:
        return (u,)
    b = torch.stack([_pad(x, has_dir) for x in mag[5:8]]).permute(3, 2, 1, 0).contiguous()
    return u, b, _pad(mag[8], has_dir).permute(2, 1, 0).contiguous()


def _fluids(c, shape, gen):
    if c["kind"] == "list":
        return [_smooth(shape, gen, True, 0.3), _smooth(shape, gen, False)]
    return [_initial(c, shape, gen)]


def _block_shapes(c):
    if c["kind"] == "list":
        return [(n, n, n) for n in _list_sizes(c)]
    if c["kind"] == "ensemble":
        return [(n, n, 1) for n in _ensemble_sizes(c)]
    return [_shape(c)]


def _interiors(c, seed):
    gen = torch.Generator().manual_seed(int(seed) * 7919 + 17)
    return [_fluids(c, s, gen) for s in _block_shapes(c)]


def _cotangents(arrays, seed):
    """dL/d(final state) of a linear loss, for every value of the state."""
    dev = torch.Generator(device="cuda").manual_seed(int(seed) * 31 + 5)
    return [tuple(torch.randn(t.shape, generator=dev, device="cuda", dtype=torch.float64) for t in a) for a in arrays]


def _box(whole, off, size):
    """The ghost-padded box of a block of a periodic domain, reference layout."""
    idx = [torch.remainder(torch.arange(-NB, size[d] + NB, device="cuda") + off[d], whole.shape[2 - d]) for d in range(3)]
    return whole[idx[2]][:, idx[1]][:, :, idx[0]].contiguous()


class _Flat:
    """Result tensors of every block, as views of one buffer per array."""

    def __init__(self, shapes):
        self.whole, self.parts = [], []
        for k in range(len(shapes[0])):
            n = [int(np.prod(s[k])) for s in shapes]
            buf = torch.empty(sum(n), device="cuda", dtype=torch.float64)
            self.whole.append(buf)
            self.parts.append([p.view(s[k]) for p, s in zip(torch.split(buf, n), shapes)])

    def block(self, i):
        return [p[i] for p in self.parts]


def prepare(c, seed):
    s = _session(c)
    has_dir = _has_dir(c)
    if c["kind"] == "linked":
        whole = _arrays(_interiors(c, seed)[0], (False, False, False))
        arrays = [tuple(_box(t, off, size) for t in whole) for off, size in s.boxes]
    else:
        arrays = [_arrays(f, has_dir) for f in _interiors(c, seed)]
    st = {"case": c, "session": s, "in": arrays, "out": _Flat([[t.shape for t in a] for a in arrays])}
    if c["kind"] in ("rollout", "ensemble"):
        st["g"] = _cotangents(arrays, seed)
    if not s.tuned:
        for b, a in zip(s.blocks, arrays):
            b.upload_device(*a)
        if c["kind"] == "list":
            pk.autotune_all()
        else:
            pk.update_boundaries(s.blocks[0])
            pk.autotune(s.blocks[0])
        s.tuned = True
    return st


# ---- one pass ----------------------------------------------------------------------


def run(st):
    c, s = st["case"], st["session"]
    kind = c["kind"]
    if kind == "rollout":
        x = tuple(t.requires_grad_(True) for t in st["in"][0])
        y = adjoint.rollout(x if c["mag"] else x[0], s.plan)
        y = y if c["mag"] else (y,)
        return {"state": list(y), "grad": list(torch.autograd.grad(y, x, st["g"][0]))}
    if kind == "ensemble":
        final = s.plan.run(st["in"])
        grad = s.plan.backward(st["g"])
        cat = lambda v: [torch.cat([t[k].reshape(-1) for t in v]) for k in range(3)]  # noqa: E731
        return {"state": cat(final), "grad": cat(grad)}
    for b, a in zip(s.blocks, st["in"]):
        b.upload_device(*a)
    cg = s.blocks[0]
    if kind == "fields":
        return [pk.datafield_f32(cg, n) for n in (FIELDS_MHD if c["mag"] else FIELDS_HD)]
    if kind == "run":
        told = pk.run(cg, c["steps"])
    elif kind in ("list", "linked"):
        told = pk.run_all(c["steps"])
    elif kind == "unsplit":
        told = pk.run_unsplit(cg, 1e30, c["steps"])[:1]
    else:
        dt, ch = _stage_scalars(c)
        for _ in range(c["steps"]):
            for d in range(3):
                for istep in (pk.RK2_1, pk.RK2_2):
                    pk.solve_cg(cg, d, istep, dt, ch)
                    pk.update_boundaries(cg)
        told = ()
    out = st["out"]
    for i, b in enumerate(s.blocks):
        b.download_device(*out.block(i))
    return {"state": out.whole, "told": list(told)}


def _stage_scalars(c):
    """A dt and GLM speed a stage is called with (well inside the CFL limit)."""
    return 0.05 / max(_shape(c)), 1.0


def work(c):
    kind = c["kind"]
    cells = [float(np.prod(s)) for s in _block_shapes(c)]
    ndir = sum(_has_dir(c))
    nv = 14 if kind == "list" else (9 if kind == "ensemble" or c["mag"] else 5)
    flops = {5: 500.0, 9: 1300.0, 14: 1800.0}[nv]  # of one sweep (two RK2 stages) of one cell
    n = sum(cells)
    if kind == "fields":
        names = FIELDS_MHD if c["mag"] else FIELDS_HD
        return {"bytes": n * (8.0 * nv + 4.0 * len(names)), "flops": n * 30.0}
    if kind == "stages":
        sweeps = c["steps"] * ndir
        return {"bytes": n * sweeps * (2 * 16.0 + 8.0) * nv, "flops": n * sweeps * flops}
    if kind == "unsplit":
        # two stages: the state read (the second also reads the base) and written; every direction's fluxes
        return {"bytes": n * c["steps"] * 40.0 * nv, "flops": n * c["steps"] * ndir * flops}
    sweeps = c["steps"] * 2 * ndir
    if kind in ("rollout", "ensemble"):
        # forward sweeps, and backward ones that read the state and the adjoint and write the adjoint
        return {"bytes": n * sweeps * (16.0 + 24.0) * nv, "flops": n * sweeps * 4.0 * flops}
    return {"bytes": n * sweeps * 16.0 * nv, "flops": n * sweeps * flops}


# ---- the same in plain 64-bit torch ---------------------------------------------------
#
# The scheme of the library on periodic interiors: torch.roll is the boundary,
# every branch a torch.where, so autograd differentiates the branch taken.
# A fluid is a list of 5 or 9 tensors whose last three axes are x, y, z.


def _limited(lim, a, b):
    """Slope from backward (a) and forward (b) differences."""
    if lim == "vanleer":
        ok = a * b > 0.0
        return torch.where(ok, 2.0 * a * b / torch.where(ok, a + b, torch.ones_like(a)), torch.zeros_like(a))
    s = 0.5 * (torch.copysign(torch.ones_like(a), a) + torch.copysign(torch.ones_like(b), b))
    x, y = a.abs(), b.abs()
    if lim == "minmod":
        return s * torch.minimum(x, y)
    if lim == "moncen":
        return s * torch.minimum(2.0 * torch.minimum(x, y), 0.5 * (a + b).abs())
    return s * torch.where(x > y, torch.minimum(x, 2.0 * y), torch.minimum(2.0 * x, y))


def _side(q, gam):
    """Conserved state and flux along the normal of a face state
    [rho, vn, vt1, vt2, p, bn, bt1, bt2]; B entries absent for hydro."""
    rho, u, v, w, p = q[:5]
    en = p / (gam - 1.0) + 0.5 * rho * (u * u + v * v + w * w)
    if len(q) == 5:
        return [rho, rho * u, rho * v, rho * w, en], [rho * u, rho * u * u + p, rho * v * u, rho * w * u, (en + p) * u]
    bx, by, bz = q[5:8]
    b2 = bx * bx + by * by + bz * bz
    en = en + 0.5 * b2
    pt = p + 0.5 * b2
    f = [rho * u, rho * u * u + pt - bx * bx, rho * v * u - bx * by, rho * w * u - bx * bz,
         (en + pt) * u - bx * (u * bx + v * by + w * bz), by * u - bx * v, bz * u - bx * w]
    return [rho, rho * u, rho * v, rho * w, en, by, bz], f


def _safe(x, ok):
    return torch.where(ok, x, torch.ones_like(x))


def _pick(sup_l, sup_r, left, both, fl, fr, a, b):
    """Per variable: the upwind flux, or the left, right or averaged star flux."""
    out = []
    for x, y, s, t in zip(fl, fr, a, b):
        star = torch.where(both, 0.5 * (s + t), torch.where(left, s, t))
        out.append(torch.where(sup_l, x, torch.where(sup_r, y, star)))
    return out


def _hllc(l, r, gam):
    ul, fl = _side(l, gam)
    ur, fr = _side(r, gam)
    c = torch.sqrt(torch.maximum(gam * l[4] / l[0], gam * r[4] / r[0]))
    sl, sr = torch.minimum(l[1], r[1]) - c, torch.maximum(l[1], r[1]) + c
    al, ar = (sl - l[1]) * l[0], (sr - r[1]) * r[0]
    sm = ((ar * r[1] - r[4]) - (al * l[1] - l[4])) / (ar - al)
    ps = 0.5 * ((l[4] + al * (sm - l[1])) + (r[4] + ar * (sm - r[1])))

    def star(q, s, a, u, f):
        d = s - sm
        d = _safe(d, d != 0.0)
        n = a / d
        us = [n, n * sm, n * q[2], n * q[3], ((s - q[1]) * u[4] - q[4] * q[1] + ps * sm) / d]
        return [x + s * (y - z) for x, y, z in zip(f, us, u)]

    return _pick(sl >= 0.0, sr <= 0.0, sm > 0.0, sm == 0.0, fl, fr, star(l, sl, al, ul, fl), star(r, sr, ar, ur, fr))


def _hlld(l, r, gam, ch):
    f_psi = 0.5 * ch * ch * ((r[5] + l[5]) - (r[8] - l[8]) / ch)
    f_bn = 0.5 * ((r[8] + l[8]) - ch * (r[5] - l[5]))
    ul, fl = _side(l[:8], gam)
    ur, fr = _side(r[:8], gam)

    def speed(q):
        b2 = q[5] * q[5] + q[6] * q[6] + q[7] * q[7]
        gp = gam * q[4]
        t = gp + b2
        return (t + torch.sqrt(t * t - 4.0 * gp * (q[5] * q[5]))) / q[0], q[4] + 0.5 * b2

    cl, pl = speed(l)
    cr, pr = speed(r)
    c = torch.sqrt(0.5 * torch.maximum(cl, cr))
    sl, sr = torch.minimum(l[1], r[1]) - c, torch.maximum(l[1], r[1]) + c
    xl, xr = sl - l[1], sr - r[1]
    al, ar = xl * l[0], xr * r[0]
    sm = ((ar * r[1] - pr) - (al * l[1] - pl)) / (ar - al)
    ps = 0.5 * ((pl + al * (sm - l[1])) + (pr + ar * (sm - r[1])))
    bb = l[5] * r[5]
    hy = ((sr * r[6] - sl * l[6]) - (fr[5] - fl[5])) / (sr - sl)
    hz = ((sr * r[7] - sl * l[7]) - (fr[6] - fl[6])) / (sr - sl)

    def outer(q, s, x, a):
        d = s - sm
        d = _safe(d, d != 0.0)
        e = a * d - bb
        ok = (e.abs() > 2.220446049250313e-16 * bb.abs()) & (bb / gam <= q[4])
        k = (a * x - bb) / _safe(e, ok)
        by, bz = torch.where(ok, q[6] * k, hy), torch.where(ok, q[7] * k, hz)
        return d, a / d, by, bz, q[2] + q[5] / a * (q[6] - by), q[3] + q[5] / a * (q[7] - bz)

    dl, nl, bly, blz, vly, vlz = outer(l, sl, xl, al)
    dr, nr, bry, brz, vry, vrz = outer(r, sr, xr, ar)
    hasb = l[5].abs() > 0.0
    ql, qr = torch.sqrt(_safe(nl, nl > 0.0)), torch.sqrt(_safe(nr, nr > 0.0))
    all_, alr = sm - l[5].abs() / ql, sm + r[5].abs() / qr
    inner = hasb & ~(all_ > 0.0) & ~(alr < 0.0)
    sg = torch.where(l[5] >= 0.0, torch.ones_like(c), -torch.ones_like(c))
    add = ql + qr
    v2y = (ql * vly + qr * vry + sg * (bry - bly)) / add
    v2z = (ql * vlz + qr * vrz + sg * (brz - blz)) / add
    b2y = (ql * bry + qr * bly + sg * ql * qr * (vry - vly)) / add
    b2z = (ql * brz + qr * blz + sg * ql * qr * (vrz - vlz)) / add
    vb2 = sm * (0.5 * (l[5] + r[5])) + v2y * b2y + v2z * b2z

    def star(q, s, x, d, n, by, bz, vy, vz, pt, u, f, alf, sq, sign):
        vb = q[1] * q[5] + q[2] * q[6] + q[3] * q[7]
        vbs = sm * q[5] + vy * by + vz * bz
        e = (x * u[4] - pt * q[1] + ps * sm + q[5] * (vb - vbs)) / d
        us = [n, n * sm, n * vy, n * vz, e, by, bz]
        u2 = [n, n * sm, n * v2y, n * v2z, e + sign * sg * sq * (vbs - vb2), b2y, b2z]
        out = []
        for k in range(7):
            one = f[k] + s * (us[k] - u[k])
            two = f[k] + alf * u2[k] - (alf - s) * us[k] - s * u[k]
            out.append(torch.where(inner, two, one))
        return out

    a = star(l, sl, xl, dl, nl, bly, blz, vly, vlz, pl, ul, fl, all_, ql, -1.0)
    b = star(r, sr, xr, dr, nr, bry, brz, vry, vrz, pr, ur, fr, alr, qr, 1.0)
    left = torch.where(inner | ~hasb, sm > 0.0, all_ > 0.0)
    both = (sm == 0.0) & (inner | ~hasb)
    f = _pick(sl >= 0.0, sr <= 0.0, left, both, fl, fr, a, b)
    return f[:5] + [f_bn, f[5], f[6], f_psi]


def _order(d, nv):
    """Variables with the normal components first along direction d (an involution)."""
    p = {0: [0, 1, 2, 3, 4, 5, 6, 7, 8], 1: [0, 2, 1, 3, 4, 6, 5, 7, 8], 2: [0, 3, 2, 1, 4, 7, 6, 5, 8]}[d]
    return p[:nv]


def _prims(u):
    rho = u[0]
    p = (GAMMA - 1.0) * (u[4] - 0.5 * (u[1] * u[1] + u[2] * u[2] + u[3] * u[3]) / rho)
    if len(u) == 9:
        p = p - 0.5 * (GAMMA - 1.0) * (u[5] * u[5] + u[6] * u[6] + u[7] * u[7])
    return [rho, u[1] / rho, u[2] / rho, u[3] / rho, p] + list(u[5:])


def _flux_difference(w, ax, lim, ch):
    """F(i-1/2) - F(i+1/2) of a state in sweep order along tensor axis ax."""
    l, r = [], []
    for q in _prims(w):
        h = 0.5 * _limited(lim, q - torch.roll(q, 1, ax), torch.roll(q, -1, ax) - q)
        l.append(q + h)
        r.append(torch.roll(q - h, -1, ax))
    f = _hlld(l, r, GAMMA, ch) if len(w) == 9 else _hllc(l, r, GAMMA)
    return [torch.roll(x, 1, ax) - x for x in f]


def _floored(w, cfg):
    rho = torch.clamp(w[0], min=cfg.smalld)
    k = 0.5 * (w[1] * w[1] + w[2] * w[2] + w[3] * w[3]) / rho
    if len(w) == 9:
        k = k + 0.5 * (w[5] * w[5] + w[6] * w[6] + w[7] * w[7])
    return [rho, w[1], w[2], w[3], torch.clamp(w[4] - k, min=cfg.smallei) + k] + list(w[5:])


def _swept(u, d, dt, dl, ch, fac, lim, cfg):
    """Both RK2 stages along d, psi damped by fac."""
    nv = len(u)
    p = _order(d, nv)
    w = [u[k] for k in p]
    ax = w[0].dim() - 3 + d
    half = _floored([x + 0.5 * dt / dl * y for x, y in zip(w, _flux_difference(w, ax, lim, ch))], cfg)
    w = _floored([x + dt / dl * y for x, y in zip(w, _flux_difference(half, ax, lim, ch))], cfg)
    w = [w[k] for k in p]
    if nv == 9:
        w[8] = w[8] * fac
    return w


def _cfl_dt(u, dls, has_dir, cfg):
    rho = u[0]
    ek = 0.5 * (u[1] * u[1] + u[2] * u[2] + u[3] * u[3]) / rho
    pmag = 0.5 * (u[5] * u[5] + u[6] * u[6] + u[7] * u[7]) if len(u) == 9 else 0.0
    p = (u[4] - ek) * (GAMMA - 1.0) + (1.0 - GAMMA) * pmag
    cs = torch.sqrt(((2.0 * pmag + GAMMA * p) / rho).abs())
    return cfg.cfl * torch.stack([(dls[d] / ((u[1 + d] / rho).abs() + cs)).min() for d in range(3) if has_dir[d]]).min()


def _stepped(groups, steps, lim, cfg, has_dir, each=False):
    """The main loop over groups of blocks [(fluids, dls)], one dt for all;
    each: remember what a rollout's backward pass needs sweep by sweep.
    Returns the groups, the simulated time and the last dt."""
    old, t, dt = None, 0.0, None
    for k in range(steps):
        dt = torch.stack([_cfl_dt(u, dls, has_dir, cfg) for fl, dls in groups for u in fl]).min()
        if k:
            dt = torch.minimum(dt, 2.0 * old)
        mdl = [min(dls[d] for d in range(3) if has_dir[d]) for _, dls in groups]
        ch = cfg.cfl_glm * min(mdl) / dt
        fac = math.exp(-cfg.glm_alpha * cfg.cfl_glm * min(mdl) / min(mdl))
        for half in ((0, 1, 2), (2, 1, 0)):
            dirs = [d for d in half if has_dir[d]]
            for d in dirs:
                f = fac if d == dirs[-1] else 1.0

                def sweep(fl, dls, dt, ch, d=d, f=f):
                    return [_swept(u, d, dt, dls[d], ch, f, lim, cfg) for u in fl]

                groups = [(checkpoint(sweep, fl, dls, dt, ch, use_reentrant=False) if each else sweep(fl, dls, dt, ch),
                           dls) for fl, dls in groups]
        old = dt
        t = t + 2.0 * dt
    return groups, t, dt


def _dls(c, shape):
    if c["kind"] == "linked":
        return (1.0 / max(shape),) * 3
    return tuple(1.0 / s for s in shape)


def _unsplit(u, steps, lim, cfg, dls, has_dir):
    t, old = 0.0, None
    mdl = min(dls[d] for d in range(3) if has_dir[d])
    for k in range(steps):
        dt = _cfl_dt(u, dls, has_dir, cfg)
        if k:
            dt = torch.minimum(dt, 2.0 * old)
        ch = cfg.cfl_glm * mdl / dt
        fac = math.exp(-0.5 * cfg.glm_alpha * cfg.cfl_glm)

        def add(base, w, coef):
            out = list(base)
            for d in range(3):
                if has_dir[d]:
                    p = _order(d, len(w))
                    df = _flux_difference([w[i] for i in p], w[0].dim() - 3 + d, lim, ch)
                    for i, x in zip(p, df):
                        out[i] = out[i] + coef * dt / dls[d] * x
            return out

        if len(u) == 9:
            u = list(u[:8]) + [u[8] * fac]
        u = add(u, add(u, u, 0.5), 1.0)
        for d in range(3):
            if has_dir[d]:
                u = _floored(u, cfg)
        if len(u) == 9:
            u = list(u[:8]) + [u[8] * fac]
        t, old = t + dt, dt
    return u, t


def exact(c, seed):
    cfg, kind, lim, has_dir = _config(c), c["kind"], c["limiter"], _has_dir(c)
    blocks, shapes = _interiors(c, seed), _block_shapes(c)
    if kind == "rollout":
        x = _arrays(blocks[0], has_dir)
        g = _cotangents([x], seed)[0]
        u = [t.clone().requires_grad_(True) for t in blocks[0][0]]
        groups, _, _ = _stepped([([u], _dls(c, shapes[0]))], c["steps"], lim, cfg, has_dir, True)
        y = _arrays(groups[0][0], has_dir)
        return {"state": [t.detach() for t in y], "grad": _scattered(torch.autograd.grad(y, u, g), has_dir)}
    if kind == "ensemble":
        state, grad = [], []
        g = _cotangents([_arrays(f, has_dir) for f in blocks], seed)
        for f, s, gi in zip(blocks, shapes, g):
            u = [t.clone().requires_grad_(True) for t in f[0]]
            groups, _, _ = _stepped([([u], _dls(c, s))], c["steps"], lim, cfg, has_dir, True)
            y = _arrays(groups[0][0], has_dir)
            state.append([t.detach() for t in y])
            grad.append(_scattered(torch.autograd.grad(y, u, gi), has_dir))
        cat = lambda v: [torch.cat([t[k].reshape(-1) for t in v]) for k in range(3)]  # noqa: E731
        return {"state": cat(state), "grad": cat(grad)}
    if kind == "list":
        # blocks of one shape advance together along a leading axis
        order = sorted(set(shapes))
        groups = []
        for s in order:
            members = [b for b, sh in zip(blocks, shapes) if sh == s]
            fl = [[torch.stack([m[f][k] for m in members]) for k in range(len(members[0][f]))] for f in range(2)]
            groups.append((fl, _dls(c, s)))
        groups, t, dt = _stepped(groups, c["steps"], lim, cfg, has_dir)
        at = {s: 0 for s in order}
        arrays = []
        for s in shapes:
            fl, i = groups[order.index(s)][0], at[s]
            at[s] += 1
            arrays.append(_arrays([[x[i] for x in f] for f in fl], has_dir))
        return {"state": _joined(arrays), "told": [float(t), float(dt)]}
    dls = _dls(c, shapes[0])
    if kind == "fields":
        return _fields(blocks[0][0])
    if kind == "unsplit":
        u, t = _unsplit(blocks[0][0], c["steps"], lim, cfg, dls, has_dir)
        return {"state": _joined([_arrays([u], has_dir)]), "told": [float(t)]}
    if kind == "stages":
        dt, ch = _stage_scalars(c)
        u = blocks[0][0]
        for _ in range(c["steps"]):
            for d in range(3):
                u = _swept(u, d, dt, dls[d], ch, 1.0, lim, cfg)
        return {"state": _joined([_arrays([u], has_dir)]), "told": []}
    groups, t, dt = _stepped([(blocks[0], dls)], c["steps"], lim, cfg, has_dir)
    if kind == "linked":
        whole = _arrays(groups[0][0], (False, False, False))
        n = shapes[0]
        edges = [[0] + _cuts(n[d], k) + [n[d]] for d, k in enumerate((c["cx"], c["cy"], c["cz"]))]
        arrays = []
        for z0, z1 in zip(edges[2], edges[2][1:]):
            for y0, y1 in zip(edges[1], edges[1][1:]):
                for x0, x1 in zip(edges[0], edges[0][1:]):
                    arrays.append(tuple(_box(w, (x0, y0, z0), (x1 - x0, y1 - y0, z1 - z0)) for w in whole))
    else:
        arrays = [_arrays(groups[0][0], has_dir)]
    return {"state": _joined(arrays), "told": [float(t), float(dt)]}


def _joined(arrays):
    return [torch.cat([a[k].reshape(-1) for a in arrays]) for k in range(len(arrays[0]))]


def _scattered(grad, has_dir):
    """Gradients of the interior values in the reference layout, ghosts zero."""
    pad = [x for d in (2, 1, 0) for x in ((NB, NB) if has_dir[d] else (0, 0))]
    g = [torch.nn.functional.pad(t, pad) for t in grad]
    u = torch.stack(g[:5]).permute(3, 2, 1, 0).contiguous()
    if len(g) == 5:
        return [u]
    return [u, torch.stack(g[5:8]).permute(3, 2, 1, 0).contiguous(), g[8].permute(2, 1, 0).contiguous()]


def _fields(u):
    mag = len(u) == 9
    m2 = u[1] * u[1] + u[2] * u[2] + u[3] * u[3]
    b2 = u[5] * u[5] + u[6] * u[6] + u[7] * u[7] if mag else torch.zeros_like(m2)
    eth = u[4] - 0.5 * m2 / u[0] - 0.5 * b2
    out = [u[0], u[1] / u[0], u[2] / u[0], u[3] / u[0], u[4], (GAMMA - 1.0) * eth, eth / u[0]]
    if mag:
        out += [u[5], u[6], u[7], torch.sqrt(b2), u[8]]
    return [x.cpu().numpy() for x in out]
