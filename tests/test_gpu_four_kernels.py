"""The four-kernel path (weak form in FP32-bulk, N = 1): a stage leaves the face states of its new state
for the next one. Steps on them equal, bit for bit, steps that begin from a state set by the caller."""
import numpy as np
import pytest

from flexi_amd import testcase
from flexi_amd.mesh import periodic_box, sine_deform

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,node,split,precision", [(1, "gauss-lobatto", "pi", "fp64"), (1, "gauss", None, "fp64")] +
                         [(N, "gauss", None, "fp32-bulk") for N in (1, 2, 3, 4, 5, 6, 7)])
def test_steps_on_kept_face_states(N, node, split, precision):
    from flexi_amd.solver import DGSolver
    mesh = periodic_box(3, 2, 4, NGeo=2, deform=sine_deform(0.1))
    gpu = DGSolver(mesh, N, node_type=node, split_dg=split, riemann="roe", precision=precision)
    try:
        U = testcase.tgv_density_perturbed(gpu.metrics()["Elem_xGP"], amplitude=1e-2, Ma=1.0)
        states = {}
        for how in ("kept", "set"):
            gpu.set_state(U)
            gpu.dt, err = gpu.CalcTimeStep()
            assert err == 0
            for step in range(4):
                gpu.TimeStepByLSERKW2(0.0)
                if step == 1:  # gradients with the density's: they prolong another state into the face arrays
                    gpu.gradients(5)
                if how == "set":
                    gpu.set_state(gpu.get_state())
            states[how] = gpu.get_state()
        assert np.all(np.isfinite(states["kept"])) and np.array_equal(states["kept"], states["set"])
    finally:
        gpu.close()
