"""Metric terms of meshes of parallelepipeds, which the library forms from the edges of each element: one value per face
for both of its elements wherever the mesh lies, no flattening of what is no rounding, constant terms where the
box is axis-aligned, and conservation on sheared boxes in both forms."""
import numpy as np
import pytest

import oracle as orc
from flexi_amd import testcase
from flexi_amd.basis import nodes_weights
from flexi_amd.mesh import periodic_box

pytestmark = pytest.mark.gpu

SHEAR = np.array([[1.0, 0.3, 0.1], [0.2, 1.0, 0.15], [0.05, 0.25, 1.0]])
TERMS = ("Metrics_fTilde", "Metrics_gTilde", "Metrics_hTilde")


def box(offset=0.0, h=1.0, shear=True, NGeo=1):
    return periodic_box(4, 3, 5, NGeo=NGeo, deform=lambda x: offset + h * (x @ SHEAR.T if shear else x))


def solver(mesh, N, node="gauss-lobatto", split="pi"):
    from flexi_amd.solver import DGSolver
    return DGSolver(mesh, N, node_type=node, split_dg=split, riemann="roe")


def metrics(mesh, N):
    s = solver(mesh, N)
    try:
        return s.metrics()
    finally:
        s.close()


@pytest.mark.parametrize("N", [3, 7])
@pytest.mark.parametrize("offset,h", [(0.0, 1.0), (0.0, 0.2), (100.0, 1e-3), (1000.0, 1e-4)])
def test_both_elements_of_a_face_have_its_metric(N, offset, h):
    m = metrics(box(offset, h), N)
    # two derivatives of degree N, each at most 2 N^2 times the rounding of its values
    bound = (2.0 * N * N) ** 2 * 1.2e-16
    dims = (4, 3, 5)
    for d, name in enumerate(TERMS):
        M = m[name].reshape((3,) + (N + 1,) * 3 + dims, order="F")
        plus = np.take(np.take(M, N, 1 + d), range(dims[d] - 1), 3 + d)
        minus = np.take(np.take(M, 0, 1 + d), range(1, dims[d]), 3 + d)
        assert np.abs(plus - minus).max() <= bound * np.abs(plus).max()


@pytest.mark.parametrize("offset,h,NGeo", [(0.0, 1.0, 1), (0.0, 1.0, 2), (1000.0, 1e-4, 1)])
def test_axis_aligned_boxes_have_constant_terms(offset, h, NGeo):
    m = metrics(box(offset, h, shear=False, NGeo=NGeo), 4)
    for name in TERMS:
        assert np.all(m[name] == m[name][:, :1, :1, :1])
    assert np.all(m["sJ"] == m["sJ"][:1, :1, :1])


def test_small_curved_elements_beside_a_large_one():
    # two layers of elements of 1e-6 with faces curved by 3e-12, far less than the rounding of the third
    # layer's coordinates (1e3)
    def deform(x):
        t = (x[..., 0] + np.pi) * 3.0 / (2.0 * np.pi)
        frac = t - np.floor(t + 1e-9)
        y = x.copy()
        y[..., 0] = np.where(t <= 2.0 + 1e-9, 1e-6 * t, 2e-6 + (t - 2.0) * 1e3)
        for d in (1, 2):
            y[..., d] = (x[..., d] + np.pi) * 1e-6
        y[..., 1] += 3e-12 * 4.0 * frac * (1.0 - frac)
        return y
    mesh = periodic_box(3, 2, 2, NGeo=2, deform=deform)
    got, want = metrics(mesh, 4), orc.calc_metrics(4, orc.NODE_GL, mesh)
    small = np.arange(mesh.nElems) % 3 < 2
    for name in TERMS + ("sJ",):
        a, b = got[name][..., small], want[name][..., small]
        assert np.abs(a - b).max() <= 1e-10 * np.abs(b).max()


@pytest.mark.parametrize("node,split", [("gauss-lobatto", "pi"), ("gauss-lobatto", None), ("gauss", None)])
@pytest.mark.parametrize("h", [1.0, 0.2])
def test_conservation_on_sheared_boxes(node, split, h):
    s = solver(box(0.0, h), 5, node, split)
    try:
        m = s.metrics()
        U = testcase.tgv_density_perturbed(m["Elem_xGP"] / h, amplitude=1e-2, Ma=1.0)
        Ut = s.rhs(U)
    finally:
        s.close()
    w = nodes_weights(5, s.node_type)[1]
    W = (w[:, None, None] * w[None, :, None] * w[None, None, :])[..., None] / m["sJ"]
    for v in range(5):
        assert abs(np.sum(W * Ut[v])) <= 1e-13 * np.sum(W * np.abs(Ut[v]))
