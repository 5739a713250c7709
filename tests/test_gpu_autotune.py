"""The batch autotuner on kernels with one budget and one number of threads (H8
FP64 diffusion): it keeps what the launches run, and a batch prepared from the
stored line gives the same matrices."""
import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

import oracle as O

pytestmark = pytest.mark.gpu


def batch_of(ctx, forms):
    batch, meshes = core.Batch(ctx), []
    for i, (form, ndn, coeff) in enumerate(forms):
        conn, xyz = core.gen_h8block(1.0, 2.0, 0.5, 6 + i, 5, 7)
        m = core.DeviceMesh(ctx, L.H8, conn, core.gen_perturb(xyz, [0, 0, 0], [1, 2, 0.5], 0.01, i))
        m.set_dofs(ndn)
        batch.add(m, form, L.RULE_GAUSS, 2, np.ravel(coeff), L.FP64)
        meshes.append(m)
    return batch, meshes


DIFFUSION = [(L.DIFFUSION_ISO, 1, [1.7]), (L.DIFFUSION_MAT, 1, np.diag([1.0, 2.0, 3.0]))]


def test_packed_batch(ctx, tmp_path):
    db = str(tmp_path / "tuned.txt")
    batch, meshes = batch_of(ctx, DIFFUSION)
    tuned = batch.autotune(db_path=db, key="packed", reps=2)
    assert tuned["threads"] == 256 and tuned["budget_kib"] == 80 and tuned["max_nodes"] in (32, 64)
    for m in meshes:  # two tile sizes, one shape each
        assert m.tile_info()[0] >= 2
    batch.run()
    want = [batch.matrix(i).csc_arrays(1)[2] for i in range(2)]
    other, _ = batch_of(ctx, DIFFUSION)
    again = other.autotune(db_path=db, key="packed", reps=2)
    assert {k: again[k] for k in ("threads", "budget_kib", "max_nodes")} == \
        {k: tuned[k] for k in ("threads", "budget_kib", "max_nodes")}
    other.run()
    for i in range(2):
        assert np.array_equal(other.matrix(i).csc_arrays(1)[2], want[i])
    batch.close()
    other.close()


def test_mixed_kernels_keep_the_candidate(ctx):
    batch, _ = batch_of(ctx, DIFFUSION[:1] + [(L.LIN_ELASTIC, 3, O.iso_D(200.0, 0.3))])
    tuned = batch.autotune(reps=2)
    assert tuned["threads"] in (512, 1024) and tuned["budget_kib"] in (80, 160)
    batch.close()
