"""Device memory of a context. The weak form's two kernels take no more than the four kernels, so that every mesh that
fits those still fits. The split form's contexts hold, beside the four kernels' arrays, at most the face states
(20 doubles a face point), viscous face fluxes (8 in the working precision), the side slots and the boundary nodes'
metric terms in FP64; with the library's own metric terms the four kernels have 8 doubles of their own."""
import pytest

from flexi_amd.mesh import periodic_box, sine_deform

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,node,split,precision", [
    (2, "gauss", None, "fp64"), (5, "gauss", None, "fp64"), (7, "gauss-lobatto", None, "fp64"),
    (2, "gauss-lobatto", "pi", "fp64"), (7, "gauss-lobatto", "pi", "fp64"),
    (2, "gauss-lobatto", "pi", "fp32-bulk"), (7, "gauss-lobatto", "pi", "fp32-bulk")])
def test_memory_beside_the_four_kernels(N, node, split, precision, monkeypatch):
    import torch
    from flexi_amd.solver import DGSolver
    K = {2: 32, 5: 16, 7: 12}[N]
    mesh = periodic_box(K, K, K, NGeo=2, deform=sine_deform(0.1))

    def taken():
        def used():
            torch.cuda.synchronize()
            free, total = torch.cuda.mem_get_info()
            return total - free
        before = used()
        s = DGSolver(mesh, N, node_type=node, split_dg=split, precision=precision)
        try:
            return s.kernel_pipeline(), used() - before
        finally:
            s.close()
    taken()  # loads the library's kernels
    path, mine = taken()
    monkeypatch.setenv("FXG_PIPELINE", "classic")
    classic, four = taken()
    assert path == ("fused" if split else "weak") and classic == "classic"
    points, boundary = 3 * (N + 1) ** 2 * mesh.nElems, ((N + 1) ** 3 - (N - 1) ** 3) * mesh.nElems
    more = points * (160 + 8 * (8 if precision == "fp64" else 4) + 8 - 64) + 80 * boundary
    assert 0 < mine <= four + (more if split else 0)
