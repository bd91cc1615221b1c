"""The FP64 stage kernel of the Gauss-Lobatto split form (one lane per line of nodes) against the
oracle at every degree, solver and kind of metric terms: the line and node phases have a remainder
of their own at each N. Bound: the library's parity target of 1e-12 relative, at Mach 1, where the
right-hand side is not a small difference of large pressure terms."""
import numpy as np
import pytest

import oracle as orc
from flexi_amd import testcase
from flexi_amd.mesh import periodic_box, sine_deform

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel())


@pytest.mark.parametrize("riemann", ["lf", "roe", "roeentropyfix"])
@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7])
def test_stage_curved_host_metrics_against_oracle(N, riemann):
    from flexi_amd.solver import DGSolver
    mesh = periodic_box(3, 2, 4, NGeo=2, deform=sine_deform(0.1))
    m = orc.calc_metrics(N, orc.NODE_GL, mesh)
    U = testcase.tgv_density_perturbed(m["Elem_xGP"], amplitude=1e-2, Ma=1.0)
    ref = orc.Solver(orc.params(N, orc.NODE_GL, 1, {"lf": 1, "roe": 3, "roeentropyfix": 33}[riemann]), mesh, m)
    gpu = DGSolver(mesh, N, node_type="gauss-lobatto", split_dg="pi", riemann=riemann, metrics=m)
    try:
        assert rel(gpu.rhs(U), ref.rhs(U)) <= 1e-12
        # a step, and the time step of its last stage's spectral radii against the time-step kernel's
        gpu.set_state(U)
        gpu.dt, err = gpu.CalcTimeStep()
        assert err == 0
        gpu.TimeStepByLSERKW2(0.0)
        dt_stage = gpu.CalcTimeStep()
        U1 = gpu.get_state()
        gpu.set_state(U1)
        assert gpu.CalcTimeStep() == dt_stage
        Uo, R = U.copy(order="F"), 0.0
        for a, b in zip(np.concatenate([[0.0], gpu.scheme.RKA]), gpu.scheme.RKb):
            R = ref.rhs(Uo) - a * R
            Uo = Uo + b * gpu.dt * R
        assert rel(U1, Uo) <= 1e-13
    finally:
        gpu.close()
