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


def sheared(pts):
    """A linear map: every element of the box stays a parallelepiped."""
    x, y, z = pts[..., 0], pts[..., 1], pts[..., 2]
    return np.stack([x + 0.3 * y, y - 0.2 * z, 0.8 * z + 0.1 * x], axis=-1)


@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("how", ["own", "host", "bent"])
def test_stage_constant_metrics_against_oracle(N, how):
    """Parallelepipeds: the library's metric terms are the same at all nodes of an element, and the
    kernels that read them once per element agree with the oracle, with the library's own face
    metrics and with host-supplied ones (the side's normals). bent: one geometry node moved by
    1e-6 of the box, far above the coordinates' rounding: the general route."""
    from flexi_amd.solver import DGSolver
    mesh = periodic_box(3, 2, 4, NGeo=2, deform=sheared)
    if how == "bent":
        mesh.NodeCoords[0, 1, 1, 1, 5] += 1e-6 * 2 * np.pi
    m = orc.calc_metrics(N, orc.NODE_GL, mesh)
    U = testcase.tgv_density_perturbed(m["Elem_xGP"], amplitude=1e-2, Ma=1.0)
    gpu = DGSolver(mesh, N, node_type="gauss-lobatto", split_dg="pi", riemann="roe")
    try:
        g = gpu.metrics()
        for k in ("Metrics_fTilde", "Metrics_gTilde", "Metrics_hTilde", "sJ"):
            assert rel(g[k], m[k]) <= 1e-12
            first = g[k][..., :1, :1, :1, :]
            assert np.array_equal(np.broadcast_to(first, g[k].shape), g[k]) == (how != "bent")
        if how == "host":
            gpu.close()
            gpu = DGSolver(mesh, N, node_type="gauss-lobatto", split_dg="pi", riemann="roe", metrics=g)
        ref = orc.Solver(orc.params(N, orc.NODE_GL, 1, orc.RIEMANN_ROE), mesh, g if how == "host" else m)
        assert rel(gpu.rhs(U), ref.rhs(U)) <= 1e-12
        gpu.set_state(U)
        gpu.dt, _ = gpu.CalcTimeStep()
        gpu.TimeStepByLSERKW2(0.0)
        dt_stage = gpu.CalcTimeStep()
        U1 = gpu.get_state()
        gpu.set_state(U1)
        assert gpu.CalcTimeStep() == dt_stage
    finally:
        gpu.close()


@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("how", ["own", "host", "reference"])
def test_bulk_stage_against_oracle(N, how):
    """FP32-bulk: packed metric terms of the nodes and the face points, from either side's own face
    metric or the side's normals. Bound: sums of up to 48 products rounded to 2^-24 whose terms are up to
    16 times the sum, 48 * 2^-24 * 16 = 4.6e-5."""
    from flexi_amd.solver import DGSolver
    mesh = periodic_box(3, 2, 4, NGeo=2, deform=sine_deform(0.1))
    m = orc.calc_metrics(N, orc.NODE_GL, mesh)
    U = testcase.tgv_density_perturbed(m["Elem_xGP"], amplitude=1e-2, Ma=1.0)
    ref = orc.Solver(orc.params(N, orc.NODE_GL, 1, orc.RIEMANN_ROE), mesh, m)
    kw = dict(metrics=m) if how == "host" else dict(metric_order=how)
    gpu = DGSolver(mesh, N, node_type="gauss-lobatto", split_dg="pi", riemann="roe", precision="fp32-bulk", **kw)
    try:
        assert rel(gpu.rhs(U), ref.rhs(U)) <= 4.6e-5
    finally:
        gpu.close()
