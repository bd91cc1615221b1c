"""Elements in every orientation: each element of a box turned by one of the 24 rotations of its axes and the master of
each inner side drawn, so that all four flips and every pair of local sides occur. Right-hand sides and steps
against the oracle on the same mesh, the adjoint against central differences. Bounds, relative: 1e-11, since the
rounding of the metric terms alone moves the oracle by up to 8e-13 between a mesh and its turned copy; FP32-bulk 1e-3 (a
point of a face taken for another one moves these by more than a tenth); the adjoint's as in test_gpu_adjoint_lines."""
import itertools

import numpy as np
import pytest

import oracle as orc
from flexi_amd import testcase
from flexi_amd.mesh import Mesh, periodic_box, side_to_vol, sine_deform, walled_box

pytestmark = pytest.mark.gpu
ROTATIONS = [(p, f) for p in itertools.permutations(range(3)) for f in itertools.product((0, 1), repeat=3)
             if np.linalg.det(np.eye(3)[list(p)] * (1 - 2 * np.array(f))[:, None]) > 0]
SIDE = {(2, 0): 1, (1, 0): 2, (0, 1): 3, (1, 1): 4, (0, 0): 5, (2, 1): 6}


def turn(a, rot):
    """Nodal array (n,n,n,...) along the turned axes: axis d is axis p[d] of before, reversed where f[d]."""
    p, f = rot
    a = np.transpose(a, list(p) + list(range(3, a.ndim)))
    return a[tuple(slice(None, None, -1) if x else slice(None) for x in f)]


def turn_elements(a, rots):
    """turn() on the node axes of a (vars,n,n,n,K)."""
    out = np.empty_like(a)
    for e, rot in enumerate(rots):
        out[..., e] = np.moveaxis(turn(np.moveaxis(a[..., e], 0, -1), rot), -1, 0)
    return np.asfortranarray(out)


def corners(e, ls, flip, ids):
    return [ids[e][side_to_vol(1, 0, p, q, flip, ls)] for p in (0, 1) for q in (0, 1)]


def reorient(mesh, seed):
    """The mesh with turned elements. Needs three elements in each periodic direction."""
    rng = np.random.default_rng(seed)
    K, nx, ny = mesh.nElems, *mesh.shape[:2]
    rots = [ROTATIONS[i] for i in np.concatenate([np.arange(24), rng.integers(0, 24, K)])[:K]]
    vertex = lambda v: tuple(v % np.array(mesh.shape)) if mesh.nBCSides == 0 else tuple(v)
    ids = []
    for e in range(K):
        at = np.array([e % nx, e // nx % ny, e // (nx * ny)])
        a = np.empty((2, 2, 2), dtype=object)
        for c in itertools.product((0, 1), repeat=3):
            a[c] = vertex(at + c)
        ids.append(turn(a, rots[e]))
    new_side = np.zeros((K, 7), dtype=int)
    old = {ls: d for d, ls in SIDE.items()}
    for e, (p, f) in enumerate(rots):
        for ls, (d, plus) in old.items():
            nd = p.index(d)
            new_side[e, ls] = SIDE[nd, plus ^ f[nd]]
    S2E, E2S = mesh.SideToElem.copy(order="F"), np.zeros_like(mesh.ElemToSide)
    for s in range(mesh.nSides):
        m, sl = S2E[0, s] - 1, S2E[1, s] - 1
        mls, sls = new_side[m, S2E[2, s]], new_side[sl, S2E[3, s]] if s >= mesh.nBCSides else 0
        if s >= mesh.nBCSides:
            if rng.random() < 0.5:
                m, sl, mls, sls = sl, m, sls, mls
            want = corners(m, mls, 0, ids)
            flip = [f for f in range(1, 5) if corners(sl, sls, f, ids) == want]
            assert len(flip) == 1
            S2E[:, s] = (m + 1, sl + 1, mls, sls, flip[0])
            E2S[:, sls - 1, sl] = (s + 1, flip[0])
        else:
            S2E[2, s] = mls
        E2S[:, mls - 1, m] = (s + 1, 0)
    return Mesh(nElems=K, nSides=mesh.nSides, NGeo=mesh.NGeo, NodeCoords=turn_elements(mesh.NodeCoords, rots),
                ElemToSide=E2S, SideToElem=S2E, nBCSides=mesh.nBCSides, BC=mesh.BC, BoundaryType=mesh.BoundaryType)


def box(kind):
    if kind == "walls":
        return walled_box(4, 3, 5, boundary_types={"BC_yplus": (2, 1), "BC_xminus": (3, 0), "BC_zplus": (9, 0)})
    return periodic_box(4, 3, 5, NGeo=2 if kind == "curved" else 1, deform=sine_deform(0.1) if kind == "curved" else None)


def state(x):
    # (the noise makes the right-hand side large beside its rounding)
    rho = 1.0 + 0.05 * np.sin(x[0] + 2 * x[1]) + 0.02 * np.random.default_rng(1).uniform(-1, 1, x[0].shape)
    p = 1.4 + 0.05 * np.cos(2 * x[1] - x[2])
    v = np.stack([0.4 * np.sin(x[1]), 0.3 * np.cos(x[2] + x[0]), 0.5 * np.sin(x[0])])
    return np.asfortranarray(np.concatenate([rho[None], rho * v, (2.5 * p + 0.5 * rho * (v ** 2).sum(0))[None]]))


PATHS = {"split": dict(node_type="gauss-lobatto", split_dg="pi"), "weak": dict(node_type="gauss", split_dg=None),
         "weak GL": dict(node_type="gauss-lobatto", split_dg=None)}
RP = np.asfortranarray(np.array([[1.0, 0.3, 0.0, 0.1, 1.4, 1.4]]).T)


@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("path", list(PATHS))
@pytest.mark.parametrize("kind", ["straight", "curved", "walls"])
def test_right_hand_side_and_steps(N, path, kind):
    from flexi_amd.solver import DGSolver
    mesh = reorient(box(kind), N)
    inner = mesh.SideToElem[:, mesh.nBCSides:]
    assert set(inner[4]) == {1, 2, 3, 4} and len(set(zip(inner[2], inner[3]))) >= 35
    kw = dict(PATHS[path], riemann="roe", R=1.0, mu0=1e-2)
    if kind == "walls":
        kw["ref_state_prim"] = RP
    node, split = (orc.NODE_G if path == "weak" else orc.NODE_GL), int(path == "split")
    m = orc.calc_metrics(N, node, mesh)
    ref = orc.Solver(orc.params(N, node, split, 3, R=1.0, mu0=1e-2), mesh, m, ref_state_prim=kw.get("ref_state_prim"))
    U = state(m["Elem_xGP"])
    for precision, metrics, bound in (("fp64", None, 1e-11), ("fp64", m, 1e-11), ("fp32-bulk", None, 1e-3)):
        s = DGSolver(mesh, N, precision=precision, metrics=metrics, **kw)
        try:
            s.dt = dt = 1e-3
            want = ref.rhs(U)
            assert np.linalg.norm((s.rhs(U) - want).ravel()) <= bound * np.linalg.norm(want.ravel())
            s.set_state(U)
            V = U.copy(order="F")
            for _ in range(2):  # the second on kept face states
                s.TimeStepByLSERKW2(0.0)
                ref.step(V, 0.0, dt)
            assert np.linalg.norm((s.get_state() - V).ravel()) <= bound * np.linalg.norm((V - U).ravel())
        finally:
            s.close()


@pytest.mark.parametrize("N", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("kind", ["straight", "curved"])
def test_adjoint(N, kind):
    from flexi_amd.solver import DGSolver
    from test_gpu_adjoint import perturbed_tgv, vjp
    s = DGSolver(reorient(box(kind), N), N, riemann="roe", **PATHS["split"])
    try:
        U = perturbed_tgv(s, 1)
        rng = np.random.default_rng(2)
        lam = np.asfortranarray(rng.normal(size=U.shape))
        d = np.asfortranarray(rng.normal(size=U.shape) * np.abs(U))
        jd = (s.rhs(U + 1e-6 * d) - s.rhs(U - 1e-6 * d)) / 2e-6
        assert abs(np.sum(lam * jd) - np.sum(vjp(s, U, lam) * d)) <= 1e-7 * np.sum(np.abs(lam * jd))
    finally:
        s.close()
