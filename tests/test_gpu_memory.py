"""Device memory of a context: the two-kernel paths take no more than the four kernels, whose face arrays they do not use,
so that every mesh that fits those still fits."""
import pytest

from flexi_amd.mesh import periodic_box, sine_deform

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,node,split", [(2, "gauss", None), (5, "gauss", None), (7, "gauss-lobatto", None),
                                          (2, "gauss-lobatto", "pi"), (7, "gauss-lobatto", "pi")])
def test_two_kernels_take_no_more_than_four(N, node, split, monkeypatch):
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
        s = DGSolver(mesh, N, node_type=node, split_dg=split)
        try:
            return s.kernel_pipeline(), used() - before
        finally:
            s.close()
    taken()  # loads the library's kernels
    path, mine = taken()
    monkeypatch.setenv("FXG_PIPELINE", "classic")
    classic, four = taken()
    assert path in ("weak", "fused") and classic == "classic"
    assert 0 < mine <= four
