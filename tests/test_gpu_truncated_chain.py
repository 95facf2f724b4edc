"""The steps that leave out what lies beyond the truncation (GPU).

From its second step on a run knows that its state is zero for k^2 >= kc2 and
leaves those modes out of its passes.  A run whose state was set again from a
dump takes its first step over all modes: both have to give the same bits, at
line lengths on both sides of the size where modes are left out.  The state
beyond the truncation has to come back as zeros, and a state that was not
truncated when it was set has to be taken as it is.
"""
import numpy as np
import pytest

import speccodelib_amd as scl

from oracle import spectral3d as orc

pytestmark = pytest.mark.gpu

GRIDS = [
    ((32, 32, 32), scl.SP), ((64, 64, 64), scl.SP), ((128, 64, 64), scl.SP), ((64, 128, 64), scl.DP),
    ((512, 64, 16), scl.SP), ((512, 32, 32), scl.DP), ((64, 32, 512), scl.SP), ((32, 64, 1024), scl.SP),
    ((64, 16, 1024), scl.DP), ((1024, 16, 32), scl.SP), ((16, 512, 64), scl.SP), ((32, 1024, 64), scl.SP),
]
KINDS = [dict(), dict(dealias_rhs=True), dict(forced=2, eta=0.1), dict(forced=0, kcut=20.5)]


def _k2(dims):
    nx, ny, nz = dims
    kx, ky, kz = np.arange(nx // 2 + 1), np.fft.fftfreq(ny, 1.0 / ny), np.fft.fftfreq(nz, 1.0 / nz)
    return kx[None, None, :] ** 2 + ky[None, :, None] ** 2 + kz[:, None, None] ** 2


@pytest.mark.parametrize("i", range(len(GRIDS)))
def test_restart_is_bit_identical(i):
    dims, prec = GRIDS[i]
    kw = KINDS[i % len(KINDS)]
    p = scl.Plan3D(*dims, prec)
    v0 = scl.initialize(*dims, 1, 4.0, 1.0, prec)
    for graph in (True, False):
        a = scl.DNS(p, use_graph=graph, **kw)
        a.set_velocity(*v0)
        a.step(4)
        a.sync()
        whole = a.get_velocity()
        a.set_velocity(*v0)
        a.step(1)
        a.step(1)
        a.sync()
        mid = a.get_velocity()
        a.set_velocity(*mid)
        a.step(2)
        a.sync()
        for x, y in zip(whole, a.get_velocity()):
            np.testing.assert_array_equal(x, y)
        a.close()
    kc = kw.get("kcut", 0.0) or 2.0 * (dims[0] // 2) / 3.0
    out = _k2(dims) >= np.float32(kc) ** 2 * (1 + 1e-6)
    assert all(not x[out].any() for x in whole)
    p.close()


@pytest.mark.parametrize("dealias", [False, True])
def test_untruncated_start_matches_oracle(dealias):
    # white-noise modes up to the corners: the first step has to use those
    # beyond the cut, the next ones to drop them (FP64: 1e-11, the solver's
    # step bar)
    n = 64
    p = scl.Plan3D(n, 2 * n, n, scl.DP)
    rng = np.random.default_rng(3)
    shape = (n, 2 * n, n // 2 + 1)
    kx, ky, kz, k2 = orc.wavenumber(n, 2 * n, n, "dp")
    v = [rng.standard_normal(shape) + 1j * rng.standard_normal(shape) for _ in range(3)]
    v = [np.ascontiguousarray(a / (1.0 + k2)) for a in v]
    for a in v:
        orc.symmetrize3d(a)
    orc.projection(*v, kx, ky, kz)
    d = scl.DNS(p, nu=0.01, dt=0.002, forced=1, fkmax=2.0, eps=0.1, dealias_rhs=dealias)
    d.set_velocity(*v)
    d.step(3)
    d.sync()
    got = d.get_velocity()
    o = orc.DNS(orc.DNSParams(nx=n, ny=2 * n, nz=n, dealias_rhs=dealias))
    w = v
    for _ in range(3):
        w = o.rk4_step(*w)
    for a, b in zip(got, w):
        assert np.abs(a - b).max() <= 1e-11 * np.abs(b).max()
    d.close()
    p.close()


@pytest.mark.parametrize("kcut", [0.0, 63.0, 20.5, 200.0])
def test_ab2_truncation_radii_match_small_grid_path(kcut):
    # IF-AB2 drops the modes beyond kcut in every step; eager and graph runs
    # give the same bits, and nothing is left beyond the radius
    dims = (128, 64, 64)
    p = scl.Plan3D(*dims, scl.SP)
    v0 = scl.initialize(*dims, 1, 4.0, 1.0, scl.SP)
    got = []
    for graph in (True, False):
        d = scl.DNS(p, stepper=1, kcut=kcut, use_graph=graph)
        d.set_velocity(*v0)
        d.step(7)
        d.sync()
        got.append(d.get_velocity())
        d.close()
    for x, y in zip(*got):
        np.testing.assert_array_equal(x, y)
    kc = kcut or 2.0 * 64 / 3.0
    out = _k2(dims) >= np.float32(kc) ** 2 * (1 + 1e-6)
    assert all(not x[out].any() and np.isfinite(x).all() and x.any() for x in got[0])
    p.close()
