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


@pytest.mark.parametrize("node,split", [("gauss", None), ("gauss-lobatto", None), ("gauss-lobatto", "pi")])
@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("shape,straight", [((3, 2, 4), False), ((3, 2, 4), True), ((11, 10, 10), True)])
def test_time_step_of_last_stage(N, node, split, shape, straight):
    """The time step from the sums that a step's last stage leaves (with and without the elements' values, on
    meshes smaller and larger than its workgroup) equals, bit for bit, the one formed from the state."""
    from flexi_amd.solver import DGSolver
    if N > 4 and shape[0] > 3:
        shape = (11, 10, 10) if N == 5 else (3, 3, 3)
    mesh = periodic_box(*shape) if straight else periodic_box(*shape, NGeo=2, deform=sine_deform(0.1))
    gpu = DGSolver(mesh, N, node_type=node, split_dg=split, riemann="roe")
    try:
        U = testcase.tgv_density_perturbed(gpu.metrics()["Elem_xGP"], amplitude=1e-2, Ma=1.0)
        gpu.set_state(U)
        gpu.dt, err = gpu.CalcTimeStep()
        gpu.TimeStepByLSERKW2(0.0)
        dt, err = gpu.CalcTimeStep()
        dte, erre, elem = gpu.CalcTimeStep(with_elements=True)
        U1 = gpu.get_state()
        gpu.set_state(U1)
        dt0, err0, elem0 = gpu.CalcTimeStep(with_elements=True)
        assert (dt, err) == (dte, erre) == (dt0, err0) and err == 0
        assert np.array_equal(elem, elem0) and dt == elem.min()
        gpu.dt = dt
        U1[0, 0, 0, 0, 1] = np.nan  # a NaN density is reported from the sums as from the state
        gpu.set_state(U1)
        gpu.TimeStepByLSERKW2(0.0)
        assert gpu.CalcTimeStep()[1] == 1
    finally:
        gpu.close()
