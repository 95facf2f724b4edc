"""LES and scalar steps that leave out what lies beyond the truncation.

A run whose state was set again from a dump takes its first step over all modes,
a run that went on leaves them out: both give the same bits.  Beyond the
truncation the state is zero, and a state that was not truncated when it was set
is taken as it is (FP64 against the oracle at the bar of the other LES steps,
1e-10)."""
import numpy as np
import pytest

import speccodelib_amd as scl
from oracle import les_scalar as les
from oracle import spectral3d as orc

pytestmark = pytest.mark.gpu

GRIDS = [((128, 64, 64), scl.SP), ((64, 64, 128), scl.SP), ((256, 128, 64), scl.SP), ((512, 64, 32), scl.SP),
         ((64, 64, 64), scl.DP), ((128, 256, 16), scl.DP), ((32, 32, 256), scl.DP), ((16, 64, 512), scl.DP)]
KINDS = [dict(sgs=1, cs2=0.03), dict(sgs=1, cs2=0.03, scalar=True, grad=1.0), dict(scalar=True, grad=1.0),
         dict(sgs=2, iupdate=3)]


def _k2(dims):
    nx, ny, nz = dims
    kx, ky, kz = np.arange(nx // 2 + 1), np.fft.fftfreq(ny, 1.0 / ny), np.fft.fftfreq(nz, 1.0 / nz)
    return kx[None, None, :] ** 2 + ky[None, :, None] ** 2 + kz[:, None, None] ** 2


def _state(d):
    return [*d.get_velocity()] + ([d.get_scalar()] if d.params.scalar else [])


@pytest.mark.parametrize("i", range(len(GRIDS)))
@pytest.mark.parametrize("j", range(len(KINDS)))
@pytest.mark.parametrize("kw", [dict(), dict(stepper=2), dict(dealias_rhs=True, kcut=14.5)])
def test_restart_is_bit_identical(i, j, kw):
    dims, prec = GRIDS[i]
    if kw.get("stepper") and KINDS[j].get("sgs") == 2:
        pytest.skip("the history of an AB2 run restarts with the state")
    p = scl.Plan3D(*dims, prec)
    v0 = scl.initialize(*dims, 1, 4.0, 1.0, prec)

    def start(state):
        d = scl.DNS(p, nu=0.01, dt=1e-3, forced=1, schmidt=0.7, **KINDS[j], **kw)
        d.set_velocity(*state[:3])
        if d.params.scalar:
            d.set_scalar(state[3])
        return d

    a = start([*v0, v0[1]])
    if kw.get("stepper"):
        # no restart of an AB2 run continues its history: graph steps against eager ones
        b = start([*v0, v0[1]])
        a.step(6)
        for _ in range(6):
            b.step(1)
        whole, again = _state(a), _state(b)
        b.close()
    else:
        a.step(6)
        whole = _state(a)
        b = start([*v0, v0[1]])
        b.step(2)
        b.step(1)
        c = start(_state(b))
        c.step(3)
        again = _state(c)
        b.close()
        c.close()
    out = _k2(dims) >= np.float32(kw.get("kcut") or 2.0 * (dims[0] // 2) / 3.0) ** 2 * (1 + 1e-6)
    for x, y in zip(whole, again):
        np.testing.assert_array_equal(x, y)
        assert not x[out].any()
    a.close()
    p.close()


@pytest.mark.parametrize("steps", [1, 3])
def test_untruncated_start_fp64(steps):
    n = 64
    rng = np.random.default_rng(5)
    v = [a + 1e-4 * (rng.standard_normal(a.shape) + 1j * rng.standard_normal(a.shape))
         for a in orc.initialize(n, n, n, -3, 4.0, 1.0)]
    phi = orc.initialize(n, n, n, -4, 3.0, 1.0)[0] + 1e-4 * rng.standard_normal(v[0].shape)
    for a in (*v, phi):
        orc.symmetrize3d(a)
    p = scl.Plan3D(n, n, n, scl.DP)
    delta = 2 * np.pi / n
    d = scl.DNS(p, nu=0.01, dt=1e-3, forced=1, fkmax=2.0, eps=0.1, sgs=1, cs2=0.03, delta=delta, scalar=True, grad=1.0,
                schmidt=0.7)
    d.set_velocity(*v)
    d.set_scalar(phi)
    d.step(steps)
    o = les.LESScalar(les.LESParams(nx=n, nu=0.01, dt=1e-3, forced=True, fkmax=2.0, eps=0.1, cs2=0.03, delta=delta,
                                    scalar=True, G=1.0, Sc=0.7))
    w = (*v, phi)
    for _ in range(steps):
        w = o.rk4_step(*w)
    for x, y in zip(_state(d), w):
        assert np.abs(x - y).max() < 1e-10 * np.abs(y).max()
