"""The two line kernels of the weak form (FP64, no boundary sides) against the oracle at every degree, on
Gauss and Gauss-Lobatto nodes, for each solver and kind of metric terms, and against the four-kernel
path (FXG_PIPELINE=classic). Bound: the parity target of 1e-12 relative, at Mach 1."""
import numpy as np
import pytest

import oracle as orc
from flexi_amd import testcase
from flexi_amd.mesh import periodic_box, sine_deform

pytestmark = pytest.mark.gpu
NODES = {"gauss": orc.NODE_G, "gauss-lobatto": orc.NODE_GL}


def rel(a, b):
    return np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel())


@pytest.mark.parametrize("node", list(NODES))
@pytest.mark.parametrize("how", ["host", "own", "straight"])
@pytest.mark.parametrize("N,riemann", [(2, "roe"), (3, "lf"), (4, "roeentropyfix"), (5, "roe"), (6, "lf"), (7, "roe")])
def test_weak_stage_against_oracle(N, riemann, how, node, monkeypatch):
    from flexi_amd.solver import DGSolver
    mesh = periodic_box(3, 2, 4) if how == "straight" else periodic_box(3, 2, 4, NGeo=2, deform=sine_deform(0.1))
    m = orc.calc_metrics(N, NODES[node], mesh)
    U = testcase.tgv_density_perturbed(m["Elem_xGP"], amplitude=1e-2, Ma=1.0)
    ref = orc.Solver(orc.params(N, NODES[node], 0, {"lf": 1, "roe": 3, "roeentropyfix": 33}[riemann]), mesh, m)
    kw = dict(node_type=node, split_dg=None, riemann=riemann, metrics=m if how == "host" else None)
    gpu = DGSolver(mesh, N, **kw)
    monkeypatch.setenv("FXG_PIPELINE", "classic")
    four = DGSolver(mesh, N, **kw)
    try:
        Ut = gpu.rhs(U)
        assert rel(Ut, ref.rhs(U)) <= 1e-12
        assert rel(Ut, four.rhs(U)) <= 1e-12
        for a, b in zip(gpu.gradients(), four.gradients()):
            assert rel(a, b) <= 1e-12
        out = []
        for s in (gpu, four):  # two steps: the second on the face states the first one left
            s.set_state(U)
            s.run(2)
            out.append((s.get_state(), s.t))
        assert rel(out[0][0], out[1][0]) <= 1e-13 and abs(out[0][1] - out[1][1]) <= 1e-13 * out[1][1]
    finally:
        gpu.close()
        four.close()
