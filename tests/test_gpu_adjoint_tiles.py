"""The adjoint sweep's tiles at their edges: a periodic sweep commutes with a
shift of the state along its direction, cell by cell with the same
operations, so the adjoint of a shifted state is the shifted adjoint bit for
bit wherever the tiles' edges fall.  Lengths: the shortest (nb cells, every
halo wraps several times), one tile with and without idle lanes, two and
three chunks with a remainder, and pencils that do not fill the last tile.
dL/d(dt) and dL/d(ch) are sums over the same cells in another order: at most
500*35 terms of order 1, each sum within 500*35 roundings of its magnitude
(2e4 * 1e-16 = 2e-12, times the cancellation of the terms' signs, up to 50).
"""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import piernik_amd as pk  # noqa: E402
from piernik_amd import setups  # noqa: E402

pytestmark = pytest.mark.gpu


def adjoint_of(cfg, shape, fields, lam, d):
    """lam through the adjoint of one sweep along d at the given state."""
    pk.finalize()
    pk.init(cfg)
    cg = setups._DeviceBlock(shape, 4, cfg, 1)
    to = lambda a: setups.to_device_layout(a, 4, cfg.has_dir)
    cg.upload_device(*[to(f) for f in fields])
    pk.update_boundaries(cg)
    pk._call("pk_adjoint_setup", 1, 1)
    pk._call("pk_state_save", 1, 0)
    dev = [to(x).clone() for x in lam]
    for t in dev:  # ghost entries would be folded into the interior
        inner = setups.interior_of(t, 4, cfg.has_dir).clone()
        t.zero_()
        setups.interior_of(t, 4, cfg.has_dir).copy_(inner)
    ptr = lambda ts: [ctypes.c_void_p(pk._device_ptr(t)) for t in ts] + [None] * (3 - len(ts))
    pk._call("pk_adjoint_set", 1, *ptr(dev))
    dtb, chb = ctypes.c_double(0.0), ctypes.c_double(0.0)
    pk._call("pk_sweep_adjoint", 1, 0, d, 2e-4, 1.3, 0.9, ctypes.byref(dtb), ctypes.byref(chb))
    out = [torch.empty_like(t) for t in dev]
    pk._call("pk_adjoint_get", 1, *ptr(out))
    res = [setups.interior_of(t, 4, cfg.has_dir).cpu().numpy() for t in out]
    pk.finalize()
    return res, dtb.value, chb.value


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("d", [0, 1, 2])
@pytest.mark.parametrize("n", [4, 47, 240, 241, 500])
def test_adjoint_commutes_with_shifts(n, d, mag):
    shape = [5, 5, 5]
    shape[d] = n
    shape[(d + 1) % 3] = 7
    print(f"adjoint tiles: shape {shape}, direction {d}, magnetized {mag}", flush=True)
    cfg = pk.Config(magnetized=mag, limiter="vanleer", limiter_b="vanleer", smalld=1e-6, smallei=1e-6)
    cg = setups.smooth_random(tuple(shape), seed=n + d, magnetized=mag)
    rng = np.random.default_rng(n)
    noise = lambda a: a * (1.0 + 0.01 * rng.uniform(-1, 1, a.shape))
    fields = [noise(np.array(cg.interior(a))) for a in ((cg.u, cg.b) if mag else (cg.u,))]
    if mag:
        fields.append(rng.normal(0.0, 0.01, shape))
    lam = [1.0 + 0.5 * rng.uniform(-1, 1, f.shape) for f in fields]
    base, dtb, chb = adjoint_of(cfg, tuple(shape), fields, lam, d)
    assert all(np.all(np.isfinite(b)) for b in base) and any(np.any(b != 0.0) for b in base)
    for k in sorted({1, n // 2, n - 1}):
        roll = lambda a: np.roll(a, k, axis=a.ndim - 3 + d)
        got, dtk, chk = adjoint_of(cfg, tuple(shape), [roll(f) for f in fields], [roll(x) for x in lam], d)
        for b, g in zip(base, got):
            assert np.array_equal(roll(b), g), (k, float(np.abs(roll(b) - g).max()))
        assert abs(dtk - dtb) <= 1e-10 * max(1.0, abs(dtb)) and abs(chk - chb) <= 1e-10 * max(1.0, abs(chb))
