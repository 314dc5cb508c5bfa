"""The adjoint sweep away from ordinary numbers: slopes whose squares underflow,
and states whose forward sweep is not a number."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import piernik_amd as pk  # noqa: E402
from piernik_amd import setups  # noqa: E402

pytestmark = pytest.mark.gpu

N = (12, 10, 9)


def gradient(cfg, fields, lam, d):
    pk.load_library()
    pk.finalize()
    pk.init(cfg)
    cg = setups._DeviceBlock(N, 4, cfg, 1)
    to = setups.to_device_layout
    cg.upload_device(*[to(f) for f in fields])
    pk.update_boundaries(cg)
    pk._call("pk_adjoint_setup", 1, 1)
    pk._call("pk_state_save", 1, 0)
    dev = []
    for x in lam:
        t = torch.zeros_like(to(x))
        setups.interior_of(t).copy_(torch.as_tensor(x))
        dev.append(t)
    ptrs = lambda ts: pk._device_ptrs(*ts) + [None] * (3 - len(ts))
    pk._call("pk_adjoint_set", 1, *ptrs(dev))
    dtb, chb = ctypes.c_double(0.0), ctypes.c_double(0.0)
    pk._call("pk_sweep_adjoint", 1, 0, d, 1e-3, 1.3, 0.9, ctypes.byref(dtb), ctypes.byref(chb))
    out = [torch.empty_like(t) for t in dev]
    pk._call("pk_adjoint_get", 1, *ptrs(out))
    res = [setups.interior_of(t).cpu().numpy() for t in out]
    pk.finalize()
    return res, dtb.value


def state(mag, scale, rho=1.0, p=1.0, vn=0.0):
    """Noise of the given size on velocities, transverse B and psi."""
    rng = np.random.default_rng(5)
    gam1 = 5.0 / 3.0 - 1.0
    r = rho * (1.0 + 0.1 * rng.uniform(-1, 1, N))
    v = [vn + scale * rng.normal(0, 1, N) for _ in range(3)]
    b = [scale * rng.normal(0, 1, N) for _ in range(3)]
    b[0] = b[0] * 0.0 + 0.5
    e = p / gam1 * (1.0 + 0.1 * rng.uniform(-1, 1, N)) + 0.5 * r * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
    if not mag:
        return [np.stack([r, r * v[0], r * v[1], r * v[2], e])]
    e = e + 0.5 * (b[0] ** 2 + b[1] ** 2 + b[2] ** 2)
    return [np.stack([r, r * v[0], r * v[1], r * v[2], e]), np.stack(b), scale * rng.normal(0, 1, N)]


def smallest_product(fields, d):
    """The smallest positive product of neighbouring differences along d of the
    tiny variables."""
    u = fields[0]
    q = [u[k] / u[0] for k in (1, 2, 3)] + ([fields[1][1], fields[1][2], fields[2]] if len(fields) > 1 else [])
    p = np.stack([(a - np.roll(a, 1, d)) * (np.roll(a, -1, d) - a) for a in q])
    return p[p > 0.0].min()


def adjoints(fields):
    rng = np.random.default_rng(6)
    return [rng.uniform(0.5, 1.5, f.shape) for f in fields]


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("d", [0, 1, 2])
def test_tiny_slopes(d, mag):
    """The van Leer slope's derivative depends on the ratio of the differences
    only, and noise of 1e-100 or 1e-156 changes rho and p by nothing: the
    gradients differ by roundings of values of order 1, a few hundred
    operations deep (1e-12), and by what the forward slope 2*dl*dr/(dl+dr)
    itself loses where dl*dr is subnormal, which stage 2 is linearised about:
    half of the smallest number over the product, with sensitivities of order 1."""
    cfg = pk.Config(magnetized=mag, limiter="vanleer", limiter_b="vanleer", smalld=1e-6, smallei=1e-6)
    print(f"tiny slopes, direction {d}, magnetized {mag}", flush=True)
    ref = small = None
    for scale in (1e-100, 1e-156, 1e-158):
        f = state(mag, scale)
        got, dtb = gradient(cfg, f, adjoints(f), d)
        assert np.isfinite(dtb) and all(np.all(np.isfinite(g)) for g in got), scale
        if ref is None:
            ref, small = got, dtb
        tol = 1e-12 + 0.5 * (2.0 ** -1074 / smallest_product(f, d)) if scale < 1e-150 else 1e-12
        assert tol < 1e-2 and abs(dtb - small) <= tol * max(1.0, abs(small))
        for a, b in zip(got, ref):
            assert np.all(np.abs(a - b) <= tol * np.maximum(1.0, np.abs(b))), scale


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("d", [0, 1, 2])
def test_not_a_number_stays_one(d, mag):
    """A negative sound speed squared makes the forward flux NaN, in supersonic
    flow too; without floors that is the step's result, and the gradient's."""
    cfg = pk.Config(magnetized=mag, limiter="vanleer", use_smalld=False, use_smallei=False)
    print(f"not a number, direction {d}, magnetized {mag}", flush=True)
    f = state(mag, 0.01, rho=-1.0 if mag else 1.0, p=1.0 if mag else -1.0, vn=10.0)
    got, dtb = gradient(cfg, f, adjoints(f), d)
    assert np.isnan(got[0]).any(axis=0).all()
    assert np.isnan(dtb)
