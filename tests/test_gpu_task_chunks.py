"""Symmetric diagonal blocks are summed in wavefronts of their own: tiles whose
nodes (one such block each) just miss, fill or overflow a wavefront, built the
same by the host and the device builder, give the bits of the default tiles."""
import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("etype", [L.H8, L.T10])
@pytest.mark.parametrize("form,ndn,coeff", [(L.LIN_ELASTIC, 3, O.iso_D(200.0, 0.3)),
                                            (L.DIFFUSION_MAT, 1, np.diag([1.0, 2.0, 3.0]))])
def test_same_bits_for_every_tile_size(ctx, etype, form, ndn, coeff):
    rule = (L.RULE_GAUSS, 2) if etype == L.H8 else (L.RULE_TET, 4)
    conn, xyz = core.gen_h8block(1.0, 2.0, 0.5, 9, 7, 8) if etype == L.H8 else core.gen_t10block(1.0, 2.0, 0.5, 5, 4, 6)
    mesh = core.DeviceMesh(ctx, etype, conn, xyz)
    mesh.set_dofs(ndn)
    for precision in (L.FP64, L.MIXED):
        mesh.set_tile_params()
        want = mesh.bilform(form, *rule, np.ravel(coeff), precision=precision).csc_arrays(1)[2]
        for nodes in (1, 63, 64, 65, 128, 200):
            mesh.set_tile_params(max_nodes=nodes)
            assert mesh.tiles_compare(form, precision)[1] == -1
            got = mesh.bilform(form, *rule, np.ravel(coeff), precision=precision).csc_arrays(1)[2]
            assert np.array_equal(got, want), (precision, nodes)
    mesh.close()
