"""H8 FP64 diffusion (packed element matrices, summed over the points direction
by direction) against the staged path, which integrates point by point: the
same pattern, values to 1e-13 of the norm (products of at most 64 terms an
element, 8 elements an entry); general node positions and coefficients, one
element up to several tiles, elements far from the origin, inverted elements
and elements that list a node twice."""
import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

pytestmark = pytest.mark.gpu

KAPPA = np.array([[2.0, 0.3, -0.2], [0.3, 1.5, 0.1], [-0.2, 0.1, 0.9]])


def values(ctx, conn, xyz, form, coeff, path):
    mesh = core.DeviceMesh(ctx, L.H8, conn, xyz)
    mesh.set_dofs(1)
    mesh.set_numeric_path(path)
    M = mesh.bilform(form, L.RULE_GAUSS, 2, np.ravel(coeff))
    out = M.csc_arrays(1)
    mesh.bilform_into(M, form, L.RULE_GAUSS, 2, 2.0 * np.ravel(coeff))
    twice = M.csc_arrays(1)
    M.close()
    mesh.close()
    return out, twice


def check(ctx, conn, xyz, tol=1e-13):
    for form, coeff in ((L.DIFFUSION_ISO, [1.7]), (L.DIFFUSION_MAT, KAPPA)):
        (cp, rv, nz), twice = values(ctx, conn, xyz, form, coeff, "fused")
        (scp, srv, snz), _ = values(ctx, conn, xyz, form, coeff, "staged")
        assert np.array_equal(cp, scp) and np.array_equal(rv, srv)
        assert np.linalg.norm(nz - snz) <= tol * np.linalg.norm(snz)
        assert np.array_equal(twice[2], 2.0 * nz)  # a power of two scales exactly


@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 1), (3, 3, 3), (4, 4, 4), (13, 5, 9), (17, 16, 15)])
def test_blocks(ctx, n):
    conn, xyz = core.gen_h8block(1.0, 2.0, 0.5, *n)
    rng = np.random.default_rng(n[0])
    check(ctx, conn, xyz + rng.uniform(-0.1, 0.1, xyz.shape) * np.array([1.0, 2.0, 0.5]) / np.array(n))


def test_far_from_the_origin(ctx):
    conn, xyz = core.gen_h8block(1.0, 1.0, 1.0, 4, 3, 5)
    # coordinates carry 1e3 in front of differences of 0.2: 1e-12 of them
    check(ctx, conn, xyz + np.array([1e3, -2e3, 3e3]), tol=1e-10)


def test_inverted_and_repeated(ctx):
    conn, xyz = core.gen_h8block(1.0, 1.0, 1.0, 4, 3, 2)
    conn = conn.copy()
    conn[5] = conn[5][[4, 5, 6, 7, 0, 1, 2, 3]]  # det J < 0
    conn[7, 3] = conn[7, 2]  # a collapsed edge
    check(ctx, conn, xyz)
