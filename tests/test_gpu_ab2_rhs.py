"""A right-hand side evaluated between two steps of an IF-AB2 run (GPU): the run
continues as if it had not been, to the bit, by scl_dns_rhs on host arrays and by
the device callback, and both still give the oracle-tested values of an IF-RK4
solver."""
import numpy as np
import pytest

import speccodelib_amd as scl

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

KINDS = [dict(), dict(sgs=1, cs2=0.03), dict(scalar=True, grad=1.0, schmidt=0.7)]


@pytest.mark.parametrize("grid,prec", [((32, 32, 32), scl.SP), ((64, 64, 64), scl.DP)])
@pytest.mark.parametrize("kind", range(len(KINDS)))
@pytest.mark.parametrize("steps", [1, 4])
def test_rhs_between_steps(grid, prec, kind, steps):
    if not torch.cuda.is_available():
        pytest.skip("no GPU visible to torch")
    p = scl.Plan3D(*grid, prec)
    v = [*scl.initialize(*grid, 1, 4.0, 1.0, prec)]
    v.append(v[1])
    nc = 4 if KINDS[kind].get("scalar") else 3

    def solver(stepper):
        d = scl.DNS(p, nu=0.02, dt=1e-3, forced=1, fkmax=2.5, eps=0.1, stepper=stepper, **KINDS[kind])
        d.set_velocity(*v[:3])
        if nc == 4:
            d.set_scalar(v[3])
        return d

    got, rhs = [], []
    for evaluate in (False, True):
        d = solver(2)
        d.step(steps)
        if evaluate:
            rhs.append(d.rhs(*v[:nc]))
            other = solver(0)
            ptr, n = other.state()
            y = torch.empty(n, dtype=torch.complex64 if prec == scl.SP else torch.complex128, device="cuda")
            torch.cuda.synchronize()
            scl._check(scl.lib().scl_dns_derivs_cb(d.h, 0.0, ptr, y.data_ptr()))
            other.close()
        d.step(3)
        got.append([*d.get_velocity()] + ([d.get_scalar()] if nc == 4 else []))
        d.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
    d = solver(0)
    for a, b in zip(rhs[0], d.rhs(*v[:nc])):
        np.testing.assert_array_equal(a, b)
    d.close()
    p.close()
