"""Ut, gradients and the analysis of the context's own state after steps on a caller's state in between: bit for bit
what a context without those steps returns."""
import numpy as np
import pytest

from flexi_amd import testcase
from flexi_amd.mesh import periodic_box, sine_deform

pytestmark = pytest.mark.gpu

PATHS = {"split": dict(node_type="gauss-lobatto", split_dg="pi"),
         "split FP32-bulk": dict(node_type="gauss-lobatto", split_dg="pi", precision="fp32-bulk"),
         "weak lines": dict(node_type="gauss", split_dg=None),
         "four kernels": dict(node_type="gauss", split_dg=None, precision="fp32-bulk")}


@pytest.mark.parametrize("path,trajectory", [(p, False) for p in PATHS] + [("split", True)])  # (FP64 split form only)
@pytest.mark.parametrize("last", ["step", "rhs"])
@pytest.mark.parametrize("read", ["after", "between"])  # 'between': the context's values were already read once
def test_context_keeps_its_last_right_hand_side(path, trajectory, last, read):
    import torch
    from flexi_amd.solver import DGSolver
    mesh = periodic_box(3, 2, 4, NGeo=2, deform=sine_deform(0.1))
    got = {}
    for mixed in (False, True):
        s = DGSolver(mesh, 3, riemann="roe", **PATHS[path])
        try:
            U = testcase.tgv_density_perturbed(s.metrics()["Elem_xGP"], amplitude=1e-2, Ma=1.0)
            s.set_state(U)
            if last == "step":
                s.run(2)
            else:
                s.DGTimeDerivative_weakForm(0.0)
            if read == "between":
                s.gradients(5)
            if mixed:
                other = torch.from_numpy(np.ascontiguousarray((1.1 * U).ravel(order="K"))).cuda()
                ckpt = torch.empty(s.adjoint_storage(2, 0), dtype=torch.float64, device="cuda") if trajectory else None
                torch.cuda.synchronize()
                s.forward_n_steps_dev(other.data_ptr(), [1e-3, 1e-3], ckpt.data_ptr() if trajectory else 0, 0)
                s.sync()
            got[mixed] = [*s.gradients(4), *s.gradients(5), s.get_ut(), s.tgv_analyze(5), s.get_state()]
        finally:
            s.close()
    assert np.any(got[False][6] != 0.0)
    for a, b in zip(got[True], got[False]):
        assert np.array_equal(a, b)
