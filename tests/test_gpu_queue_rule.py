"""The number of tiles from which a launch hands them out: with tiles of one node
the meshes here have fewer, exactly and more tiles a workgroup than the rule
asks (256 CUs; 6 for FP64 gradient records, 12 for the others, of which the
packed diffusion kernel has two workgroups a CU; none for the mass of one
component; in a batch 4 for FP32 and 8 for FP64 gradient records and packed
ones, 10 for the mass).  The same bits as from the default tiles, launch after
launch."""
import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

import oracle as O

pytestmark = pytest.mark.gpu

# nodes along each axis: 256 times the tiles a workgroup
SIZES = {4: (8, 8, 16), 6: (12, 8, 16), 8: (16, 8, 16), 10: (20, 8, 16), 12: (12, 16, 16), 16: (16, 16, 16),
         24: (24, 16, 16)}
# the rule alone and in a batch
FORMS = [(L.LIN_ELASTIC, 3, O.iso_D(200.0, 0.3), L.FP64, 6, 8), (L.LIN_ELASTIC, 3, O.iso_D(200.0, 0.3), L.MIXED, 12, 4),
         (L.DIFFUSION_ISO, 1, [1.7], L.FP64, 24, 16), (L.DIFFUSION_MAT, 1, np.diag([1.0, 2.0, 3.0]), L.MIXED, 12, 4),
         (L.DOT, 3, 2.5 * np.eye(3), L.FP64, 12, 10), (L.DOT, 2, 2.5 * np.eye(2), L.MIXED, 12, 10),
         (L.DOT, 1, [2.5], L.MIXED, 12, 12)]


def made(ctx, per, step, form, ndn, coeff, precision):
    a, b, c = SIZES[per]
    conn, xyz = core.gen_h8block(1.0, 2.0, 0.5, a - 1, b - 1, c - 1 + step)
    assert len(xyz) == a * b * (c + step)
    mesh = core.DeviceMesh(ctx, L.H8, conn, core.gen_perturb(xyz, [0, 0, 0], [1, 2, 0.5], 0.01, 4))
    mesh.set_dofs(ndn)
    want = mesh.bilform(form, L.RULE_GAUSS, 2, np.ravel(coeff), precision=precision).csc_arrays(1)[2]
    return mesh, want, len(xyz)


@pytest.mark.parametrize("form,ndn,coeff,precision,per,batched", FORMS)
@pytest.mark.parametrize("step", [-1, 0, 1])
def test_around_the_rule(ctx, form, ndn, coeff, precision, per, batched, step):
    mesh, want, nodes = made(ctx, per, step, form, ndn, coeff, precision)
    before = mesh.tile_info()[0]
    mesh.set_tile_params(max_nodes=1)
    M = mesh.bilform(form, L.RULE_GAUSS, 2, np.ravel(coeff), precision=precision)
    assert mesh.tile_info()[0] - before == nodes
    for _ in range(3):
        assert np.array_equal(M.csc_arrays(1)[2], want)
        mesh.bilform_into(M, form, L.RULE_GAUSS, 2, np.ravel(coeff), precision=precision)
    mesh.close()
    mesh, want, nodes = made(ctx, batched, step, form, ndn, coeff, precision)
    batch = core.Batch(ctx)
    batch.add(mesh, form, L.RULE_GAUSS, 2, np.ravel(coeff), precision)
    batch.prepare(use_graph=True, max_nodes=1)
    assert batch.stats()["tiles"] == nodes
    for _ in range(3):
        batch.run()
        ctx.synchronize()
        assert np.array_equal(batch.matrix(0).csc_arrays(1)[2], want)
    batch.close()
    mesh.close()
