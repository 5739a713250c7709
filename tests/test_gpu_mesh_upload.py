"""Meshes from host arrays go to the device in pieces through a bounded pinned
buffer: one element up to more than the buffer holds, either order of the
coordinates, give the matrix of the same mesh made from device arrays, bit for
bit; a node number out of range is refused wherever it sits."""
import ctypes

import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1, 1, 1), (25, 25, 26), (57, 60, 59)])
def test_uploads_agree(ctx, hiprt, n):
    conn, xyz = core.gen_h8block(1.0, 2.0, 0.5, *n)
    xyz = xyz + np.random.default_rng(1).uniform(-1e-3, 1e-3, xyz.shape)
    bufs = []
    for a in ((conn - 1).astype(np.int32), np.ascontiguousarray(xyz)):
        p = ctypes.c_void_p()
        assert hiprt.hipMalloc(ctypes.byref(p), a.nbytes) == 0
        assert hiprt.hipMemcpy(p, a.ctypes.data, a.nbytes, 1) == 0  # hipMemcpyHostToDevice
        bufs.append(p)
    digests = []
    for make in ("rows", "columns", "device"):
        if make == "device":
            mesh = core.DeviceMesh.__new__(core.DeviceMesh)
            mesh.ctx, mesh.etype, mesh.ndn = ctx, L.H8, 0
            (mesh.nelem, mesh.npe), mesh.nnodes = conn.shape, len(xyz)
            h = ctypes.c_void_p()
            core.check(core.lib().feasm_mesh_create_device(ctx.h, L.H8, mesh.nelem, 8, bufs[0],
                                                           mesh.nnodes, bufs[1],
                                                           ctypes.byref(h)), ctx.h)
            mesh.h = h
        else:
            mesh = core.DeviceMesh(ctx, L.H8, conn, np.ascontiguousarray(xyz) if make == "rows" else np.asfortranarray(xyz))
        mesh.set_dofs(1)
        M = mesh.bilform(L.DIFFUSION_ISO, L.RULE_GAUSS, 2, [1.0])
        digests.append(M.checksum())
        M.close()
        mesh.close()
    for p in bufs:
        hiprt.hipFree(p)
    assert digests[0] == digests[1] == digests[2]


@pytest.mark.parametrize("at", [0, 131071, 131072, -1])
@pytest.mark.parametrize("value", [0, -1, -2**63, 2**63 - 1, "nnodes + 1", 2**32 + 1])
def test_out_of_range_is_refused(ctx, at, value):
    conn, xyz = core.gen_h8block(1.0, 1.0, 1.0, 26, 26, 26)
    conn = conn.copy()
    conn.reshape(-1)[at] = len(xyz) + 1 if value == "nnodes + 1" else value
    with pytest.raises(L.FeasmError, match="missing node"):
        core.DeviceMesh(ctx, L.H8, conn, xyz)
