"""A plan closed before the solvers and adjoints made on it (GPU): they go on with
the bits they have otherwise, and closing them afterwards is in order, which is
what the garbage collector may do with objects that refer to each other."""
import numpy as np
import pytest

import speccodelib_amd as scl

pytestmark = pytest.mark.gpu

N = 32


def run(kind, prec, plan_first):
    p = scl.Plan3D(N, N, N, prec)
    u = scl.initialize(N, N, N, 1, 4.0, 1.0, prec)
    if kind == "adjoint":
        o = scl.Adjoint(p, 2, 1, nu=0.02, dt=1e-3, sgs=1)
    else:
        o = scl.DNS(p, nu=0.02, dt=1e-3, sgs=int(kind == "les"), cs2=0.03)
        o.set_velocity(*u)
        o.step(2)
    if plan_first:
        p.close()
        scl.Plan3D(N, N, N, prec).close()  # would take a freed plan's memory
    if kind == "adjoint":
        out = [*o.forward(u, 0.03)]
        g, c = o.backward(u)
        out += [*g, c]
    else:
        o.step(3)
        out = [*o.get_velocity(), o.diagnostics()["energy"]]
    o.close()
    p.close()
    return out


@pytest.mark.parametrize("kind", ["dns", "les", "adjoint"])
@pytest.mark.parametrize("prec", [scl.SP, scl.DP])
def test_the_plan_is_closed_first(kind, prec):
    for a, b in zip(run(kind, prec, True), run(kind, prec, False)):
        np.testing.assert_array_equal(a, b)
