"""Calls on a caller's state captured into a HIP graph and replayed between the context's own calls: replays write
the context's work arrays without the library's knowledge, so nothing kept there may be taken for the context's
own. Bit for bit what a context without replays returns, and every replay what the eager call gives."""
import numpy as np
import pytest

from flexi_amd import testcase
from flexi_amd.mesh import periodic_box, sine_deform, walled_box

pytestmark = pytest.mark.gpu

PATHS = {"split": dict(node_type="gauss-lobatto", split_dg="pi"),
         "split FP32-bulk": dict(node_type="gauss-lobatto", split_dg="pi", precision="fp32-bulk"),
         "split, walls": dict(node_type="gauss-lobatto", split_dg="pi", R=1.0, mu0=1e-2,
                              ref_state_prim=np.array([[1.0, 0, 0, 0, 1.4, 1.4]]).T),
         "weak lines": dict(node_type="gauss", split_dg=None),
         "four kernels": dict(node_type="gauss", split_dg=None, precision="fp32-bulk")}


@pytest.mark.parametrize("path", list(PATHS))
@pytest.mark.parametrize("call", ["rhs", "step", "steps"])
def test_replays_between_the_contexts_own_calls(path, call):
    import torch
    from flexi_amd.solver import DGSolver
    mesh = walled_box(3, 2, 4) if "walls" in path else periodic_box(3, 2, 4, NGeo=2, deform=sine_deform(0.1))

    def own_calls(replay):
        out = []
        for _ in range(4):  # (a step leaves its face states in either of two buffers)
            s.TimeStepByLSERKW2(0.0)
            replay()
        out.append(s.get_state())
        for _ in range(3):
            s.TimeStepByLSERKW2(0.0)
            replay()
            out.append(s.get_ut())
            replay()
            out += s.gradients(4)
            replay()
            out += s.gradients(5)
            replay()
            out += [s.tgv_analyze(5), s.get_state()]
            replay()
        s.DGTimeDerivative_weakForm(0.0)
        replay()
        return out + s.gradients(5) + [s.get_ut()]

    s = DGSolver(mesh, 3, riemann="roe", **PATHS[path])
    try:
        U = testcase.tgv_density_perturbed(s.metrics()["Elem_xGP"], amplitude=1e-2, Ma=1.0)
        s.dt = 1e-3
        s.set_state(U)
        want = own_calls(lambda: None)
        start = torch.from_numpy(np.ascontiguousarray((1.1 * U).ravel(order="K"))).cuda()
        V, W = start.clone(), torch.zeros_like(start)

        def eager(stream):
            if call == "rhs":
                s.rhs_dev(V.data_ptr(), W.data_ptr(), stream=stream)
            elif call == "step":
                s.step_dev(V.data_ptr(), W.data_ptr(), 1e-3, stream=stream)
            else:
                s.forward_n_steps_dev(V.data_ptr(), [1e-3, 1e-3], stream=stream)
        torch.cuda.synchronize()
        eager(0)
        s.sync()
        ref = V.clone(), W.clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            eager(torch.cuda.current_stream().cuda_stream)

        def replay():
            V.copy_(start)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(V, ref[0]) and torch.equal(W, ref[1])
        s.set_state(U)
        got = own_calls(replay)
        for a, b in zip(got, want):
            assert np.array_equal(a, b)
    finally:
        s.close()
