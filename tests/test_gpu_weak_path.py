"""The weak form's two line kernels are the ones that run where they should, and, with constant metric terms that the
host supplies (the side's normals on both sides of a face), they agree with the oracle. Bound: the parity
target of 1e-12 relative."""
import numpy as np
import pytest

import oracle as orc
from flexi_amd import testcase
from flexi_amd.mesh import periodic_box, walled_box

pytestmark = pytest.mark.gpu
NODES = {"gauss": orc.NODE_G, "gauss-lobatto": orc.NODE_GL}
FOUR = ("prolong_u", "lift", "flux", "volint")


@pytest.mark.parametrize("node", list(NODES))
@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7])
def test_which_kernels_run(N, node, monkeypatch):
    from flexi_amd.solver import DGSolver
    mesh = periodic_box(2, 2, 2)
    kw = dict(node_type=node, split_dg=None, riemann="lf")

    def path(s):
        try:
            s.set_state(testcase.tgv(s.metrics()["Elem_xGP"], Ma=1.0))
            s.profile()
            s.run(1)
            ran = {k for k, v in s.kernel_times().items() if v[1]}
            return s.kernel_pipeline(), ran & set(FOUR), ran & {"weak_faces", "weak_visc", "weak_stage"}
        finally:
            s.close()
    four = ("classic", set(FOUR), set())
    want = ("weak", set(), {"weak_faces", "weak_visc", "weak_stage"}) if N >= 2 else four
    assert path(DGSolver(mesh, N, **kw)) == want
    assert path(DGSolver(mesh, N, precision="fp32-bulk", **kw)) == four
    walls = DGSolver(walled_box(2, 2, 2), N, R=1.0, mu0=0.01, ref_state_prim=np.array([[1.0, 0, 0, 0, 71.0, 71.0]]).T, **kw)
    assert path(walls)[0] == "classic"
    monkeypatch.setenv("FXG_PIPELINE", "classic")
    assert path(DGSolver(mesh, N, **kw)) == four


@pytest.mark.parametrize("node", list(NODES))
@pytest.mark.parametrize("shear", [0.0, 0.25])
@pytest.mark.parametrize("N,riemann", [(2, "roe"), (3, "lf"), (5, "roeentropyfix"), (7, "roe")])
def test_constant_terms_from_the_host(N, riemann, shear, node):
    from flexi_amd.solver import DGSolver
    # unit cells, and a shear without rounding: the library's own terms are exactly constant
    mesh = periodic_box(3, 2, 4, lo=(0, 0, 0), length=(3, 2, 4),
                        deform=lambda x: x + shear * x[..., [1, 2, 0]])
    own = DGSolver(mesh, N, node_type=node, split_dg=None)
    m = own.metrics()
    own.close()
    assert all(np.all(m[k] == m[k][:, :1, :1, :1]) for k in ("Metrics_fTilde", "Metrics_gTilde", "Metrics_hTilde"))
    U = testcase.tgv_density_perturbed(m["Elem_xGP"], amplitude=1e-2, Ma=1.0)
    s = DGSolver(mesh, N, node_type=node, split_dg=None, riemann=riemann, metrics=m)
    ref = orc.Solver(orc.params(N, NODES[node], 0, {"lf": 1, "roe": 3, "roeentropyfix": 33}[riemann]), mesh, m).rhs(U)
    try:
        assert s.kernel_pipeline() == "weak"
        Ut = s.rhs(U)
        assert np.linalg.norm((Ut - ref).ravel()) <= 1e-12 * np.linalg.norm(ref.ravel())
    finally:
        s.close()
