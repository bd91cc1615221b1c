"""The adjoint kernels (one lane per line of nodes) at every degree, with constant metric terms per
element and with general ones: <lam, J d> from central differences of the GPU right-hand side against
<J^T lam, d>. Bound 1e-7 of sum |lam J d|: the differences' rounding (1e-16 / 1e-6) and truncation."""
import numpy as np
import pytest

from flexi_amd.mesh import sine_deform
from test_gpu_adjoint import make, perturbed_tgv, vjp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("riemann", ["lf", "roe", "roeentropyfix"])
@pytest.mark.parametrize("curved", [False, True])
def test_vjp_is_the_transpose(N, riemann, curved):
    _, s = make(N, riemann, shape=(2, 3, 2), deform=sine_deform(0.1) if curved else None, NGeo=2 if curved else 1)
    try:
        U = perturbed_tgv(s, 1)
        rng = np.random.default_rng(2)
        lam = np.asfortranarray(rng.normal(size=U.shape))
        d = np.asfortranarray(rng.normal(size=U.shape) * np.abs(U))
        jd = (s.rhs(U + 1e-6 * d) - s.rhs(U - 1e-6 * d)) / 2e-6
        assert abs(np.sum(lam * jd) - np.sum(vjp(s, U, lam) * d)) <= 1e-7 * np.sum(np.abs(lam * jd))
    finally:
        s.close()


@pytest.mark.parametrize("N", [2, 5, 7])
def test_runs_of_different_sizes_share_a_context(N):
    """The workspace of an adjoint run stays with its context: runs that need less of it or more give, bit for
    bit, what a context of their own gives."""
    import torch

    def grad(s, U, steps, every):
        x = torch.from_numpy(np.ascontiguousarray(U.ravel(order="K"))).cuda()
        ubar = torch.ones_like(x)
        torch.cuda.synchronize()
        s.adjoint_n_steps_dev(x.data_ptr(), ubar.data_ptr(), [1e-3] * steps, checkpoint_every=every)
        return ubar.cpu().numpy()

    _, s = make(N, "roe", shape=(2, 3, 2))
    try:
        U = perturbed_tgv(s, 1)
        for steps, every in ((4, 2), (6, 6), (3, 1), (5, 3), (4, 2)):
            _, own = make(N, "roe", shape=(2, 3, 2))
            try:
                assert np.array_equal(grad(s, U, steps, every), grad(own, U, steps, every))
            finally:
                own.close()
    finally:
        s.close()
