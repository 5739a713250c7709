"""feasm_bilform with distinct DOF numbers that are not node-major (the ranked
general pattern) against the COO path on the same mesh: the same CSC pattern
bit for bit, values to the rounding of their sums (at most 48 terms of either
sign an entry: 1e-14 of the largest entry), for free-then-fixed, permuted and
gapped numberings, every DOF count, both element types, nodes of no element
(whose DOF numbers may be anything), elements that list a node twice, and a
node with more neighbours than the node pattern takes."""
import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

pytestmark = pytest.mark.gpu


def block(etype, n):
    if etype == L.H8:
        conn, xyz = core.gen_h8block(1.0, 1.0, 1.0, *n)
        return conn, core.gen_perturb(xyz, [0, 0, 0], [1, 1, 1], 0.1 / max(n), 3), (L.RULE_GAUSS, 2)
    conn, xyz = core.gen_t10block(1.0, 1.0, 1.0, *n, 0.1 / max(n), 0.03 / max(n), 3)
    return conn, xyz, (L.RULE_TET, 4)


def numbering(kind, xyz, ndn):
    n = xyz.shape[0] * ndn
    if kind == "fixed last":
        fixed = np.repeat(xyz[:, 0] == 0.0, ndn)
        d = np.where(fixed, np.cumsum(fixed) + (~fixed).sum(), np.cumsum(~fixed))
        return d.reshape(-1, ndn), n
    if kind == "permuted":
        return np.random.default_rng(5).permutation(n).reshape(-1, ndn) + 1, n
    return np.arange(n).reshape(-1, ndn) * 3 + 2, 3 * n + 7  # gaps, and columns of no DOF


def form_of(name, ndn):
    if name == "elastic":
        D = np.diag([4.0, 4, 4, 1, 1, 1])
        D[:3, :3] += 1.5
        return L.LIN_ELASTIC, D
    return (L.DIFFUSION_ISO, [1.3]) if name == "diffusion" else (L.DOT, np.arange(1.0, ndn * ndn + 1))


def check(mesh, form, rule, coeff, precision=L.FP64):
    got = mesh.bilform(form, *rule, coeff, precision=precision).csc_arrays(1)
    ref = mesh.bilform(form, *rule, coeff, precision=precision, path="coo").csc_arrays(1)
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
    assert np.max(np.abs(got[2] - ref[2]), initial=0.0) <= 1e-14 * np.max(np.abs(ref[2]), initial=1.0)
    again = mesh.bilform(form, *rule, coeff, precision=precision).csc_arrays(1)
    assert np.array_equal(got[2], again[2])


@pytest.mark.parametrize("kind", ["fixed last", "permuted", "gaps"])
@pytest.mark.parametrize("etype,n", [(L.H8, (1, 1, 1)), (L.H8, (7, 5, 3)), (L.T10, (3, 2, 4))])
@pytest.mark.parametrize("name,ndn", [("elastic", 3), ("diffusion", 1), ("mass", 2), ("mass", 3)])
def test_numberings(ctx, kind, etype, n, name, ndn):
    conn, xyz, rule = block(etype, n)
    mesh = core.DeviceMesh(ctx, etype, conn, xyz)
    d, nall = numbering(kind, xyz, ndn)
    mesh.set_dofs(ndn, d, nall)
    form, coeff = form_of(name, ndn)
    check(mesh, form, rule, coeff)
    check(mesh, form, rule, coeff, L.MIXED)
    # another numbering on the same mesh, then node-major
    mesh.set_dofs(ndn, nall + 1 - d, nall)
    check(mesh, form, rule, coeff)
    mesh.set_dofs(ndn)
    check(mesh, form, rule, coeff)
    mesh.close()


@pytest.mark.parametrize("order", [1, 3, 4])
def test_other_rules(ctx, order):
    conn, xyz, _ = block(L.H8, (4, 3, 5))
    mesh = core.DeviceMesh(ctx, L.H8, conn, xyz)
    mesh.set_dofs(3, *numbering("fixed last", xyz, 3))
    check(mesh, *((L.LIN_ELASTIC, (L.RULE_GAUSS, order)) + (form_of("elastic", 3)[1],)))
    mesh.close()


def test_nodes_of_no_element_and_repeated_nodes(ctx):
    conn, xyz, rule = block(L.H8, (5, 4, 3))
    conn = conn[: conn.shape[0] // 2].copy()
    conn[3, 4:] = conn[3, :4]  # an element that lists nodes twice
    d, n = numbering("permuted", xyz, 1)
    unused = np.setdiff1d(np.arange(xyz.shape[0]), conn - 1)
    assert len(unused)
    d[unused, 0] = np.where(np.arange(len(unused)) % 2, -5, n + 100)
    mesh = core.DeviceMesh(ctx, L.H8, conn, xyz)
    mesh.set_dofs(1, d, n)
    check(mesh, L.DOT, rule, [2.0])
    mesh.close()


def test_node_beyond_the_pattern_takes_the_coo_path(ctx):
    # 45 H8 elements around one node, seven nodes of its own each: 316 neighbours
    ne = 45
    conn = np.empty((ne, 8), np.int64)
    conn[:, 0] = 1
    conn[:, 1:] = 2 + np.arange(7 * ne).reshape(ne, 7)
    xyz = np.random.default_rng(2).uniform(0.0, 1.0, (1 + 7 * ne, 3))
    mesh = core.DeviceMesh(ctx, L.H8, conn, xyz)
    mesh.set_dofs(1, *numbering("permuted", xyz, 1))
    check(mesh, L.DOT, (L.RULE_GAUSS, 2), [1.0])
    mesh.close()
