"""The FP64 fused kernels form Jacobians and gradients by exchanges between the
lanes of an element's points; the staged path integrates each point from the
basis tables.  Same pattern, values to 1e-13 of the norm (sums of at most 10
terms in each Jacobian entry, 5 points, 24 elements an entry), for general node
positions, every form, one element up to several tiles, elements far from the
origin, inverted elements and elements that list a node twice."""
import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

import oracle as O

pytestmark = pytest.mark.gpu

A = np.random.default_rng(5).uniform(-1.0, 1.0, (6, 6))
FORMS = [(L.LIN_ELASTIC, 3, O.iso_D(200.0, 0.3)), (L.LIN_ELASTIC, 3, A @ A.T + 6.0 * np.eye(6)),
         (L.DIFFUSION_ISO, 1, [1.7]), (L.DIFFUSION_MAT, 1, A[:3, :3] @ A[:3, :3].T + np.eye(3)),
         (L.DOT, 1, [2.5]), (L.DOT, 2, [[2.0, 0.5], [0.5, 1.0]]), (L.DOT, 3, np.diag([1.0, 2.0, 3.0]))]


def block(etype, n, seed=0):
    gen = core.gen_h8block if etype == L.H8 else core.gen_t10block
    conn, xyz = gen(1.0, 2.0, 0.5, *n)
    rng = np.random.default_rng(seed)
    return conn, xyz + rng.uniform(-0.08, 0.08, xyz.shape) * np.array([1.0, 2.0, 0.5]) / np.array(n)


def check(ctx, etype, conn, xyz, tol=1e-13):
    rule = (L.RULE_GAUSS, 2) if etype == L.H8 else (L.RULE_TET, 4)
    for form, ndn, coeff in FORMS:
        out = []
        for path in ("fused", "staged"):
            mesh = core.DeviceMesh(ctx, etype, conn, xyz)
            mesh.set_dofs(ndn)
            mesh.set_numeric_path(path)
            out.append(mesh.bilform(form, *rule, np.ravel(coeff)).csc_arrays(1))
            mesh.close()
        (cp, rv, nz), (scp, srv, snz) = out
        assert np.array_equal(cp, scp) and np.array_equal(rv, srv)
        assert np.linalg.norm(nz - snz) <= tol * np.linalg.norm(snz), (form, ndn)


@pytest.mark.parametrize("etype", [L.H8, L.T10])
@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 1), (5, 3, 4), (9, 8, 7)])
def test_blocks(ctx, etype, n):
    check(ctx, etype, *block(etype, n, n[0]))


@pytest.mark.parametrize("etype", [L.H8, L.T10])
def test_far_from_the_origin(ctx, etype):
    conn, xyz = block(etype, (4, 3, 5))
    # coordinates carry 1e3 in front of differences of 0.05: 1e-12 of them
    check(ctx, etype, conn, xyz + np.array([1e3, -2e3, 3e3]), tol=1e-10)


@pytest.mark.parametrize("etype", [L.H8, L.T10])
def test_inverted_and_repeated(ctx, etype):
    conn, xyz = block(etype, (4, 3, 2))
    conn = conn.copy()
    if etype == L.H8:
        conn[5] = conn[5][[4, 5, 6, 7, 0, 1, 2, 3]]  # det J < 0
        conn[7, 3] = conn[7, 2]  # a collapsed edge
    else:
        conn[5] = conn[5][[1, 0, 2, 3, 4, 6, 5, 8, 7, 9]]  # det J < 0
        conn[7, 4] = conn[7, 0]  # an edge node on its corner
    check(ctx, etype, conn, xyz)
