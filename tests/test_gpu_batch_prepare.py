"""A batch's tile queue and headers are made on the stream its launches run on:
a run queued right after they are made, with device memory that held other
numbers before, gives the single meshes' matrices bit for bit, batch after
batch."""
import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

pytestmark = pytest.mark.gpu


def test_first_run_of_new_batches(ctx):
    mesh = []
    for i, n in enumerate([(23, 19, 17), (31, 12, 20), (9, 30, 25)]):
        conn, xyz = core.gen_h8block(1.0, 2.0, 0.5, *n)
        m = core.DeviceMesh(ctx, L.H8, conn, core.gen_perturb(xyz, [0, 0, 0], [1, 2, 0.5], 0.01, i))
        m.set_dofs(1)
        mesh.append(m)
    want = [m.bilform(L.DIFFUSION_ISO, L.RULE_GAUSS, 2, [1.0 + i]).csc_arrays(1)[2] for i, m in enumerate(mesh)]
    ones = np.full(300, -1.0)  # no zero word: blocks that small are the pool's next ones
    for _ in range(6):
        core.sparse(ctx, np.arange(1, 301), np.arange(1, 301), ones, 300, 300).close()
        batch = core.Batch(ctx)
        for i, m in enumerate(mesh):
            batch.add(m, L.DIFFUSION_ISO, L.RULE_GAUSS, 2, [1.0 + i], L.FP64)
        batch.prepare(use_graph=False, max_nodes=2)
        assert batch.stats()["tiles"] >= 12 * 512  # 12 tiles a workgroup, two workgroups a CU: the queue is on
        # another entry drops the launches: the next run makes them again and starts at once
        batch.add(mesh[0], L.DIFFUSION_ISO, L.RULE_GAUSS, 2, [7.0], L.FP64)
        batch.run()
        ctx.synchronize()
        for i, w in enumerate(want):
            assert np.array_equal(batch.matrix(i).csc_arrays(1)[2], w)
        seven = batch.matrix(3).csc_arrays(1)[2]
        assert np.linalg.norm(seven - 7.0 * want[0]) <= 1e-13 * np.linalg.norm(seven)
        batch.close()
    for m in mesh:
        m.close()
