"""Meshes whose elements list nodes several times: wedges around an axis
(hexahedra with a collapsed face edge at both ends) and a cube of six pyramids
(the apex listed four times).  A block of such a node has more items than the
node has incidences, and the device tile builder's tables follow the items:
its tiles are the host builder's byte for byte, and the fused kernels' values
the oracle's to 1e-12 of the norm in FP64 (sums of at most 128 items an
entry) and 1e-5 in mixed precision (2^-24 in each of a few factors of a
product, and cancellation between them)."""
import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

import oracle as O

pytestmark = pytest.mark.gpu


def fan(n, layers):
    """n wedges a layer around the z axis; ring nodes, then the axis node, layer by layer."""
    a = 2.0 * np.pi * np.arange(n) / n
    ring = np.stack([np.cos(a), np.sin(a)], 1)
    xyz = np.concatenate([np.c_[np.r_[ring, [[0.0, 0.0]]], np.full(n + 1, 0.4 * l)] for l in range(layers + 1)])
    conn = []
    for l in range(layers):
        b, t = l * (n + 1), (l + 1) * (n + 1)
        for i in range(n):
            j = (i + 1) % n
            conn.append([b + n, b + i, b + j, b + n, t + n, t + i, t + j, t + n])
    return np.array(conn, np.int64) + 1, xyz


def pyramids():
    corner = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]
    xyz = np.array(corner + [(0.52, 0.47, 0.55)], float)
    faces = [(0, 1, 2, 3), (7, 6, 5, 4), (4, 5, 1, 0), (5, 6, 2, 1), (6, 7, 3, 2), (7, 4, 0, 3)]
    return np.array([list(f) + [8] * 4 for f in faces], np.int64) + 1, xyz


MESHES = {"fan 8x1": fan(8, 1), "fan 24x1": fan(24, 1), "fan 16x3": fan(16, 3), "fan 12x9": fan(12, 9),
          "pyramids": pyramids()}
FORMS = [("diffusion", L.DIFFUSION_ISO, 1, [1.7], L.FP64), ("diffusion", L.DIFFUSION_ISO, 1, [1.7], L.MIXED),
         ("elasticity", L.LIN_ELASTIC, 3, O.iso_D(200.0, 0.3), L.MIXED),
         ("mass", L.DOT, 2, [[2.0, 0.5], [0.5, 1.0]], L.FP64), ("mass", L.DOT, 1, [2.0], L.MIXED)]
ELASTIC = ("elasticity", L.LIN_ELASTIC, 3, O.iso_D(200.0, 0.3), L.FP64)


def check(ctx, name, form, ndn, coeff, precision, nodes):
    conn, xyz = MESHES[name]
    coeff = np.ravel(coeff)
    ocp, orv, onz = O.assemble_csc(O.H8, form, conn, xyz, ndn, coeff)
    mesh = core.DeviceMesh(ctx, L.H8, conn, xyz)
    mesh.set_dofs(ndn)
    mesh.set_tile_params(max_nodes=nodes)
    mesh.build_pattern()
    print(name, form, precision, nodes, flush=True)
    assert mesh.tiles_compare(form, precision)[1] == -1
    mesh.set_numeric_path("fused")
    cp, rv, nz = mesh.bilform(form, L.RULE_GAUSS, 2, coeff, precision=precision).csc_arrays(1)
    assert np.array_equal(cp, ocp) and np.array_equal(rv, orv)
    tol = 1e-12 if precision == L.FP64 else 1e-5
    assert np.linalg.norm(nz - onz) <= tol * np.linalg.norm(onz)
    mesh.close()


@pytest.mark.parametrize("name", list(MESHES))
@pytest.mark.parametrize("fname,form,ndn,coeff,precision", FORMS)
def test_items_beyond_incidences(ctx, name, fname, form, ndn, coeff, precision):
    for nodes in (0, 5):
        check(ctx, name, form, ndn, coeff, precision, nodes)


@pytest.mark.parametrize("name", list(MESHES))
def test_items_beyond_incidences_with_bank_numbering(ctx, name):
    # the pyramids' tile has 204 read sets, of which a bound from the
    # incidences alone would leave room for 148: the fused path is not refused
    for nodes in (0, 5):
        check(ctx, name, *ELASTIC[1:], nodes)
