"""The fused launches hand their tiles out from a queue when there are at least
three per workgroup, and in a fixed stride when there are fewer or the launch is
recorded into a graph: the values are the same bits for every tile size (so for
both walks), launch after launch, and in a batch and the replays of its graph."""
import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

import oracle as O

pytestmark = pytest.mark.gpu

D = O.iso_D(200.0, 0.3)
FORMS = [(L.LIN_ELASTIC, 3, D, L.FP64), (L.LIN_ELASTIC, 3, D, L.MIXED), (L.DIFFUSION_ISO, 1, [1.7], L.FP64),
         (L.DOT, 1, [2.5], L.FP64), (L.DOT, 3, 2.5 * np.eye(3), L.MIXED)]


def make(ctx, etype, ndn):
    if etype == L.H8:
        conn, xyz = core.gen_h8block(1.0, 2.0, 0.5, 23, 19, 17)
    else:
        conn, xyz = core.gen_t10block(1.0, 2.0, 0.5, 9, 11, 8)
    mesh = core.DeviceMesh(ctx, etype, conn, xyz)
    mesh.set_dofs(ndn)
    return mesh


@pytest.mark.parametrize("etype", [L.H8, L.T10])
@pytest.mark.parametrize("form,ndn,coeff,precision", FORMS)
def test_same_bits_from_queue_and_stride(ctx, etype, form, ndn, coeff, precision):
    rule = (L.RULE_GAUSS, 2) if etype == L.H8 else (L.RULE_TET, 4)
    mesh = make(ctx, etype, ndn)
    mesh.set_tile_params(max_nodes=0)
    want = mesh.bilform(form, *rule, np.ravel(coeff), precision=precision).csc_arrays(1)
    few = mesh.tile_info()[0]
    twice = mesh.bilform(form, *rule, 2.0 * np.ravel(coeff), precision=precision).csc_arrays(1)[2]
    mesh.set_tile_params(max_nodes=2)
    M = mesh.bilform(form, *rule, np.ravel(coeff), precision=precision)
    assert mesh.tile_info()[0] >= 3 * 512 > few  # 256 CUs, up to two workgroups each
    for _ in range(4):
        got = M.csc_arrays(1)
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
        mesh.bilform_into(M, form, *rule, np.ravel(coeff), precision=precision)

    batch = core.Batch(ctx)
    batch.add(mesh, form, *rule, np.ravel(coeff), precision)
    batch.add(mesh, form, *rule, 2.0 * np.ravel(coeff), precision)
    batch.prepare(use_graph=True, max_nodes=2)
    for _ in range(4):
        batch.run()
        ctx.synchronize()
        assert np.array_equal(batch.matrix(0).csc_arrays(1)[2], want[2])
        assert np.array_equal(batch.matrix(1).csc_arrays(1)[2], twice)
        mesh.bilform_into(M, form, *rule, np.ravel(coeff), precision=precision)
    assert np.array_equal(M.csc_arrays(1)[2], want[2])
    batch.close()
    M.close()
    mesh.close()
