"""The y- and x-passes of a RHS in one launch (planes that fit in LDS) and with
a wavefront per field (larger ones) against the separate passes, over plane
shapes, precisions and solver options.

The two differ in rounding only: the bars are those the steps have against the
oracle elsewhere (FP64 1e-11, FP32 1e-5 of the largest entry)."""
import numpy as np
import pytest

import speccodelib_amd as scl

pytestmark = pytest.mark.gpu

BAR = {scl.SP: 1e-5, scl.DP: 1e-11}
PLANES = [(16, 16), (16, 64), (16, 128), (16, 256), (32, 32), (32, 128), (64, 16), (64, 64), (128, 32), (256, 16)]


def state(nx, ny, nz, ncomp, seed=1):
    """Entries on both sides of every cut, the kx = nx/2 column among them."""
    rng = np.random.default_rng(seed)
    k2 = (np.arange(nx // 2 + 1)[None, None, :] ** 2 + (np.fft.fftfreq(ny, 1.0 / ny) ** 2)[None, :, None]
          + (np.fft.fftfreq(nz, 1.0 / nz) ** 2)[:, None, None])
    s = 0.1 / (1.0 + k2)
    return [s * (rng.standard_normal(k2.shape) + 1j * rng.standard_normal(k2.shape)) for _ in range(ncomp)]


def run(monkeypatch, plane, shape, prec, steps=3, zblock=None, **kw):
    monkeypatch.setenv("SCL_PLANE", "1" if plane else "0")
    if zblock:
        monkeypatch.setenv("SCL_ZBLOCK", str(zblock))
    ct = np.complex64 if prec == scl.SP else np.complex128
    v = [a.astype(ct) for a in state(*shape, 4 if kw.get("scalar") else 3)]
    plan = scl.Plan3D(*shape, prec)
    d = scl.DNS(plan, nu=0.02, dt=1e-3, fkmax=2.5, eps=0.1, eta=0.2, **kw)
    d.set_velocity(*v[:3])
    if kw.get("scalar"):
        d.set_scalar(v[3])
    d.step(1)
    d.step(steps - 1)
    out = list(d.get_velocity())
    if kw.get("scalar"):
        out.append(d.get_scalar())
    d.close()
    plan.close()
    return out


def compare(monkeypatch, shape, prec, **kw):
    a = run(monkeypatch, False, shape, prec, **kw)
    b = run(monkeypatch, True, shape, prec, **kw)
    for x, y in zip(a, b):
        assert np.isfinite(x).all()
        assert np.abs(x - y).max() < BAR[prec] * np.abs(x).max()


@pytest.mark.parametrize("prec", [scl.SP, scl.DP])
@pytest.mark.parametrize("plane", PLANES)
@pytest.mark.parametrize("forced", [0, 1, 2])
def test_dns_planes(monkeypatch, plane, prec, forced):
    compare(monkeypatch, (*plane, 32), prec, forced=forced)


@pytest.mark.parametrize("prec", [scl.SP, scl.DP])
@pytest.mark.parametrize("plane", PLANES)
@pytest.mark.parametrize("sgs,scalar", [(1, False), (0, True), (1, True)])
def test_les_and_scalar_planes(monkeypatch, plane, prec, sgs, scalar):
    compare(monkeypatch, (*plane, 16), prec, forced=1, sgs=sgs, cs2=0.03 if sgs else 0.0, scalar=scalar,
            grad=1.0 if scalar else 0.0, schmidt=0.7)


LINES = [(64, 128, 16), (32, 256, 16), (16, 512, 16), (32, 512, 16), (128, 64, 16), (512, 16, 16), (1024, 16, 16),
         (128, 128, 32)]


@pytest.mark.parametrize("prec", [scl.SP, scl.DP])
@pytest.mark.parametrize("shape", LINES)
@pytest.mark.parametrize("sgs,scalar", [(0, False), (1, False), (0, True), (1, True)])
def test_wavefront_per_field(monkeypatch, shape, prec, sgs, scalar):
    compare(monkeypatch, shape, prec, forced=2 if not (sgs or scalar) else 1, sgs=sgs, cs2=0.03 if sgs else 0.0,
            scalar=scalar, grad=1.0 if scalar else 0.0, schmidt=0.7)


# (32, 64, 512) and (32, 512, 64) with a radius above nx/2: every kx is kept, not every column
@pytest.mark.parametrize("shape", [(64, 128, 16), (64, 128, 128), (256, 64, 64), (32, 64, 512), (32, 512, 64)])
@pytest.mark.parametrize("prec", [scl.SP, scl.DP])
@pytest.mark.parametrize("kw", [dict(), dict(dealias_rhs=True), dict(stepper=1, kcut=31.0), dict(kcut=20.5)])
def test_truncated_lines(monkeypatch, shape, prec, kw):
    compare(monkeypatch, shape, prec, steps=5, forced=1, **kw)


@pytest.mark.parametrize("kw", [dict(), dict(dealias_rhs=True), dict(stepper=1, kcut=31.0), dict(stepper=2)])
def test_truncated_and_ab2_steps(monkeypatch, kw):
    compare(monkeypatch, (64, 64, 128), scl.SP, steps=5, forced=1, **kw)


def test_radius_above_half_nx(monkeypatch):
    """Every kx is kept, and still not every column."""
    compare(monkeypatch, (32, 64, 512), scl.SP, steps=5, forced=1, kcut=20.5)


@pytest.mark.parametrize("sgs", [0, 1])
@pytest.mark.parametrize("shape", [(32, 32, 32), (64, 128, 16)])
def test_blocked_row_order(monkeypatch, shape, sgs):
    compare(monkeypatch, shape, scl.DP, zblock=8, forced=1, sgs=sgs, cs2=0.03 if sgs else 0.0)


@pytest.mark.parametrize("prec", [scl.SP, scl.DP])
def test_rates_of_host_arrays(monkeypatch, prec):
    ct = np.complex64 if prec == scl.SP else np.complex128
    v = [a.astype(ct) for a in state(32, 64, 16, 3)]
    out = []
    for plane in ("0", "1"):
        monkeypatch.setenv("SCL_PLANE", plane)
        p = scl.Plan3D(32, 64, 16, prec)
        out.append(p.ratesdudt(*v, forced=2, fkmax=2.5, eps=0.1, eta=0.2))
        p.close()
    for x, y in zip(*out):
        assert np.abs(x - y).max() < BAR[prec] * np.abs(x).max()


@pytest.mark.parametrize("sgs", [0, 1])
@pytest.mark.parametrize("shape", [(32, 32, 16), (64, 128, 16)])
def test_adjoint_tape(monkeypatch, shape, sgs):
    """Gradients with the physical tape written by either kernel (FP64)."""
    v = state(*shape, 3)
    g = state(*shape, 3, seed=2)
    out = []
    for plane in ("0", "1"):
        monkeypatch.setenv("SCL_PLANE", plane)
        p = scl.Plan3D(*shape, scl.DP)
        a = scl.Adjoint(p, 4, 2, nu=0.02, dt=1e-3, sgs=sgs)
        a.forward(v, 0.03 if sgs else 0.0)
        out.append(a.backward(g))
        a.close()
        p.close()
    (ga, ca), (gb, cb) = out
    for x, y in zip(ga, gb):
        assert np.abs(x - y).max() < 1e-10 * np.abs(x).max()
    assert abs(ca - cb) <= 1e-10 * abs(ca)
