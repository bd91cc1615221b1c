"""The device memory an adjoint run leaves with its context: given back on request, and the next run as before."""
import numpy as np
import pytest

from flexi_amd.mesh import periodic_box

pytestmark = pytest.mark.gpu


def test_release_workspace():
    import torch
    from flexi_amd.solver import DGSolver
    from test_gpu_adjoint import perturbed_tgv
    s = DGSolver(periodic_box(12, 12, 12), 5)
    try:
        s.release_workspace()  # nothing kept yet
        U = torch.from_numpy(np.ascontiguousarray(perturbed_tgv(s, 1).ravel(order="K"))).cuda()

        def grad(every, steps=4):
            ub = torch.ones_like(U)
            torch.cuda.synchronize()
            s.adjoint_n_steps_dev(U.data_ptr(), ub.data_ptr(), [1e-4] * steps, every)
            return ub
        first = grad(1, 1)  # the scratch that the context needs for any adjoint
        s.release_workspace()

        def taken():  # device memory in use beside torch's own
            free, total = torch.cuda.mem_get_info()
            return total - free - torch.cuda.memory_reserved()
        before = taken()
        want = grad(4)
        kept = taken() - before
        states = 4 * 5 * U.numel() * 8  # the stage states of the four steps, without their face states
        assert states < kept <= 4 << 30
        s.release_workspace()
        assert taken() <= before
        assert torch.equal(grad(4), want) and torch.equal(grad(1, 1), first)
    finally:
        s.close()
