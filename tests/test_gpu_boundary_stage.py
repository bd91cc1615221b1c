"""Boundary sides on the FP64 stage kernels: a stage leaves the boundary states of its new state, and the viscous
kernel forms the boundary fluxes. Steps on them equal, bit for bit, steps that begin from a state set by the caller,
also where the conditions change between two steps."""
import numpy as np
import pytest

from flexi_amd import _lib
from flexi_amd.mesh import walled_box

pytestmark = pytest.mark.gpu
RP = np.asfortranarray(np.array([[1.0, 0.3, 0.1, 0.0, 1.4, 1.4], [1.1, 0.2, 0.0, 0.1, 1.5, 1.5 / 1.1]]).T)


@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("first,then", [((4, 1), (3, 0)), ((2, 1), (2, 2)), ((9, 0), (91, 0)), ((24, 1), (4, 2))])
def test_steps_on_kept_boundary_states(N, first, then):
    from flexi_amd.solver import DGSolver
    mesh = walled_box(3, 2, 2, boundary_types={"BC_yplus": first, "BC_xminus": first})
    gpu = DGSolver(mesh, N, node_type="gauss-lobatto", split_dg="pi", riemann="roe", R=1.0, mu0=1e-2, ref_state_prim=RP)
    try:
        L = _lib.lib()
        bc = np.ascontiguousarray(mesh.BC[:mesh.nBCSides], dtype=np.int32)
        types = [np.asfortranarray(mesh.BoundaryType.astype(np.int32)) for _ in range(2)]
        types[1][(types[0][:, :2] == first).all(axis=1), :2] = then

        def conditions(bt):
            _lib.check(L.fxg_set_boundaries(gpu.ctx, bt.shape[0], bc.ctypes.data, bt.ctypes.data, RP.shape[1],
                                            RP.ctypes.data))

        x = gpu.metrics()["Elem_xGP"]
        rho, p = 1.0 + 0.05 * np.sin(3 * x[0]), 1.4 + 0.05 * np.cos(2 * x[1])
        v = np.stack([0.2 * np.sin(x[1]), 0.1 * np.cos(x[2]), 0.1 * np.sin(x[0])])
        U = np.asfortranarray(np.concatenate([rho[None], rho * v, (2.5 * p + 0.5 * rho * (v ** 2).sum(0))[None]]))
        gpu.dt = 1e-3
        out = {}
        for how in ("kept", "set"):
            conditions(types[0])
            gpu.set_state(U)
            for step in range(4):
                if step == 2:
                    conditions(types[1])
                gpu.TimeStepByLSERKW2(0.0)
                if how == "set":
                    gpu.set_state(gpu.get_state())
            out[how] = gpu.get_state()
        assert np.all(np.isfinite(out["kept"])) and np.array_equal(out["kept"], out["set"])
        assert not np.array_equal(out["kept"], U)
    finally:
        gpu.close()
