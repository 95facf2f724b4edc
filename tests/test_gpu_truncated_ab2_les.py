"""IF-AB2 steps of the LES and scalar solvers that leave out what lies beyond the
truncation (GPU; fields of 2 MB and more).

Against the FP64 oracle at the bar of the stepper's other tests (1e-10; time steps
1e-13), from a state with energy beyond the radius; against the passes that leave
nothing out (SCL_EXT_UNFUSED=1) over grids, precisions and kinds, at the bars that
two forms of the passes have elsewhere (FP64 1e-11, FP32 1e-5 of the largest
entry); captured steps equal to direct launches to the bit."""
import numpy as np
import pytest

import speccodelib_amd as scl
from oracle import ab2
from oracle import les_scalar as les
from oracle import spectral3d as orc

pytestmark = pytest.mark.gpu

GRIDS = [((128, 64, 64), scl.SP), ((64, 64, 128), scl.SP), ((512, 64, 32), scl.SP), ((64, 64, 64), scl.DP),
         ((32, 256, 32), scl.DP), ((16, 64, 512), scl.DP)]
KINDS = [dict(sgs=1, cs2=0.03), dict(sgs=1, cs2=0.03, scalar=True, grad=1.0, schmidt=0.7),
         dict(scalar=True, grad=1.0, schmidt=0.7), dict(sgs=2, iupdate=2)]
BAR = {scl.SP: 1e-5, scl.DP: 1e-11}


def fields(grid, prec, nc=4):
    """Energy in every mode, beyond each radius too."""
    rng = np.random.default_rng(7)
    kx, ky, kz, k2 = orc.wavenumber(*grid, "dp")
    v = [np.ascontiguousarray(0.05 * (rng.standard_normal(k2.shape) + 1j * rng.standard_normal(k2.shape)) / (1.0 + k2))
         for _ in range(nc)]
    for a in v:
        orc.symmetrize3d(a)
    orc.projection(*v[:3], kx, ky, kz)
    return [a.astype(np.complex64 if prec == scl.SP else np.complex128) for a in v]


def run(grid, prec, calls, **kw):
    p = scl.Plan3D(*grid, prec)
    d = scl.DNS(p, nu=0.02, dt=1e-3, forced=1, fkmax=2.5, eps=0.1, **kw)
    v = fields(grid, prec)
    d.set_velocity(*v[:3])
    if kw.get("scalar"):
        d.set_scalar(v[3])
    for n in calls:
        d.step(n)
    out = [*d.get_velocity()] + ([d.get_scalar()] if kw.get("scalar") else [])
    d.close()
    p.close()
    return out


@pytest.mark.parametrize("i", range(len(GRIDS)))
@pytest.mark.parametrize("kind", range(len(KINDS)))
@pytest.mark.parametrize("kw", [dict(stepper=2), dict(stepper=1, beta=0.1, umax=3.0, kcut=14.5), dict(stepper=0)])
def test_against_passes_over_all_modes(monkeypatch, i, kind, kw):
    grid, prec = GRIDS[i]
    got = run(grid, prec, (1, 2, 2), **KINDS[kind], **kw)
    monkeypatch.setenv("SCL_EXT_UNFUSED", "1")
    want = run(grid, prec, (1, 2, 2), **KINDS[kind], **kw)
    for a, b in zip(got, want):
        assert np.isfinite(a).all() and b.any()
        assert np.abs(a - b).max() < BAR[prec] * np.abs(b).max()


@pytest.mark.parametrize("i", range(len(GRIDS)))
@pytest.mark.parametrize("kind", range(len(KINDS)))
def test_captured_steps_are_the_direct_ones(i, kind):
    grid, prec = GRIDS[i]
    got = [run(grid, prec, calls, stepper=2, use_graph=graph, **KINDS[kind])
           for graph, calls in ((True, (6,)), (True, (1, 1, 1, 3)), (False, (6,)))]
    for other in got[1:]:
        for a, b in zip(got[0], other):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("dynamic", [False, True])
@pytest.mark.parametrize("kcut", [64.0 / 3.0, 30.5])
def test_oracle_fp64(dynamic, kcut):
    n, steps, nu, sc = 64, 5, 5e-3, 0.7
    cfl = dict(beta=0.5, dtw=0.03, ieout=3, umax=3.0 * np.sqrt(3.0))
    delta = 2 * np.pi / n
    v = fields((n, n, n), scl.DP)
    lo = les.LESScalar(les.LESParams(nx=n, nu=nu, dt=0.0, forced=True, fkmax=2.5, eps=0.1, cs2=0.0289, delta=delta,
                                     dynamic=dynamic, iupdate=3, scalar=True, G=1.0, Sc=sc))
    lo.rhs_per_step = 1
    o = ab2.AB2(ab2.AB2Params(nx=n, nu=nu, forced=True, fkmax=2.5, eps=0.1, kcut=kcut, **cfl), v, rhs=lo.rhs,
                nus=[nu, nu, nu, nu / sc])
    p = scl.Plan3D(n, n, n, scl.DP)
    s = scl.DNS(p, nu=nu, forced=1, fkmax=2.5, eps=0.1, sgs=2 if dynamic else 1, cs2=0.0289, delta=delta,
                delta_test=2 * delta, k_test=(2 * (n // 2) / 3) / 2, iupdate=3, scalar=True, grad=1.0, schmidt=sc,
                stepper=1, kcut=kcut, **cfl)
    s.set_velocity(*v[:3])
    s.set_scalar(v[3])
    dts = []
    for _ in range(steps):
        s.step(1)
        o.step()
        dts.append(s.step_info()[1])
    assert np.abs(np.array(dts) - np.array(o.dts)).max() < 1e-13 * max(o.dts)
    for a, b in zip([*s.get_velocity(), s.get_scalar()], o.v):
        assert np.abs(a - b).max() < 1e-10 * np.abs(b).max()
    s.close()
    p.close()
