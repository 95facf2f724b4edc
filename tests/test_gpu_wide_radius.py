"""Truncation radii up to and beyond the corner of the box (GPU): steps that leave
out what lies beyond the radius, and steps that leave nothing out because the
radius keeps nearly all modes, against the FP64 oracle at the bars of the solvers'
other tests (two steps: DNS 1e-11, LES and scalar 1e-10), from a state with
energy in every mode."""
import numpy as np
import pytest

import speccodelib_amd as scl
from oracle import les_scalar as les
from oracle import spectral3d as orc

pytestmark = pytest.mark.gpu

# FP64 fields of 2 MB, where modes are left out at every radius, and of 17 MB,
# where they are left out as long as enough are
GRIDS = [(64, 64, 64), (512, 64, 64)]
# radii as parts of nx/2 that keep from a quarter of the modes to all of them, on
# both sides of each rule; the last is beyond the corner
RADII = {GRIDS[0]: [0.8, 0.97, 1.25, 1.74], GRIDS[1]: [0.7, 0.92, 1.1]}
CASES = [(g, r * g[0] / 2) for g in GRIDS for r in RADII[g]]


def start(grid, nc):
    rng = np.random.default_rng(11)
    kx, ky, kz, k2 = orc.wavenumber(*grid, "dp")
    v = [0.02 * (rng.standard_normal(k2.shape) + 1j * rng.standard_normal(k2.shape)) / (1.0 + k2) for _ in range(nc)]
    v = [np.ascontiguousarray(a) for a in v]
    for a in v:
        orc.symmetrize3d(a)
    orc.projection(*v[:3], kx, ky, kz)
    return v


@pytest.mark.parametrize("grid,kcut", CASES)
def test_dns(grid, kcut):
    dealias = kcut > grid[0] / 2
    class Params(orc.DNSParams):
        kcut2 = kcut * kcut

    v = start(grid, 3)
    p = scl.Plan3D(*grid, scl.DP)
    d = scl.DNS(p, nu=0.01, dt=0.002, forced=1, fkmax=2.0, eps=0.1, kcut=kcut, dealias_rhs=dealias)
    d.set_velocity(*v)
    d.step(1)
    d.step(1)
    o = orc.DNS(Params(nx=grid[0], ny=grid[1], nz=grid[2], nu=0.01, dt=0.002, forced=True, fkmax=2.0, eps=0.1,
                       dealias_rhs=dealias))
    for _ in range(2):
        v = o.rk4_step(*v)
    for a, b in zip(d.get_velocity(), v):
        assert np.abs(a - b).max() < 1e-11 * np.abs(b).max()
    d.close()
    p.close()


@pytest.mark.parametrize("grid,kcut", CASES)
@pytest.mark.parametrize("sgs,scalar", [(0, True), (1, True)])
def test_les_and_scalar(grid, kcut, sgs, scalar):
    v = start(grid, 4)
    p = scl.Plan3D(*grid, scl.DP)
    delta = 2 * np.pi / grid[0]
    d = scl.DNS(p, nu=0.01, dt=0.001, forced=1, fkmax=2.0, eps=0.1, kcut=kcut, sgs=sgs, cs2=0.03 if sgs else 0.0,
                delta=delta, scalar=scalar, grad=1.0 if scalar else 0.0, schmidt=0.7)
    d.set_velocity(*v[:3])
    if scalar:
        d.set_scalar(v[3])
    d.step(1)
    d.step(1)
    o = les.LESScalar(les.LESParams(nx=grid[0], ny=grid[1], nz=grid[2], nu=0.01, dt=0.001, forced=True, fkmax=2.0,
                                    eps=0.1, cs2=0.03 if sgs else 0.0, delta=delta, scalar=scalar,
                                    G=1.0 if scalar else 0.0, Sc=0.7))
    o.kcut2 = kcut * kcut
    w = v if scalar else (*v[:3], np.zeros_like(v[3]))
    for _ in range(2):
        w = o.rk4_step(*w)
    got = [*d.get_velocity()] + ([d.get_scalar()] if scalar else [])
    for a, b in zip(got, w):
        assert np.abs(a - b).max() < 1e-10 * np.abs(b).max()
    d.close()
    p.close()
