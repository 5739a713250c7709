"""Meshes from host arrays of growing and shrinking sizes, on both sides of the 256
KiB up to which a kernel reads the pinned buffer, by one thread and by several
at once with contexts of their own: the matrix of the same mesh is the same bits
whichever way its arrays went."""
import threading

import numpy as np
import pytest

from feasm import _lib as L
from feasm import core

pytestmark = pytest.mark.gpu

# 248,984 and 264,112 bytes of connectivity and coordinates beside others
SIZES = [(1, 1, 1), (2, 1, 1), (2, 3, 2), (5, 4, 6), (9, 9, 8), (16, 16, 16), (17, 16, 16), (30, 31, 29), (45, 41, 37)]


def digest(ctx, n, columns=False, etype=L.H8):
    gen = core.gen_h8block if etype == L.H8 else core.gen_t10block
    conn, xyz = gen(1.0, 2.0, 0.5, *n)
    xyz = xyz + np.random.default_rng(1).uniform(-1e-3, 1e-3, xyz.shape)
    mesh = core.DeviceMesh(ctx, etype, conn, np.asfortranarray(xyz) if columns else xyz)
    mesh.set_dofs(1)
    mesh.set_numeric_path("staged")
    M = mesh.bilform(L.DIFFUSION_ISO, *((L.RULE_GAUSS, 2) if etype == L.H8 else (L.RULE_TET, 4)), [1.0])
    out = M.checksum()
    M.close()
    mesh.close()
    return out


def device_digest(ctx, hiprt, n, etype=L.H8):
    """The same from arrays already on the device."""
    import ctypes

    gen = core.gen_h8block if etype == L.H8 else core.gen_t10block
    conn, xyz = gen(1.0, 2.0, 0.5, *n)
    xyz = np.ascontiguousarray(xyz + np.random.default_rng(1).uniform(-1e-3, 1e-3, xyz.shape))
    bufs = []
    for a in ((conn - 1).astype(np.int32), xyz):
        p = ctypes.c_void_p()
        assert hiprt.hipMalloc(ctypes.byref(p), a.nbytes) == 0
        assert hiprt.hipMemcpy(p, a.ctypes.data, a.nbytes, 1) == 0
        bufs.append(p)
    mesh = core.DeviceMesh.__new__(core.DeviceMesh)
    mesh.ctx, mesh.etype, mesh.ndn = ctx, etype, 0
    (mesh.nelem, mesh.npe), mesh.nnodes = conn.shape, len(xyz)
    h = ctypes.c_void_p()
    core.check(core.lib().feasm_mesh_create_device(ctx.h, etype, mesh.nelem, mesh.npe, bufs[0], mesh.nnodes, bufs[1],
                                                   ctypes.byref(h)), ctx.h)
    mesh.h = h
    mesh.set_dofs(1)
    mesh.set_numeric_path("staged")
    M = mesh.bilform(L.DIFFUSION_ISO, *((L.RULE_GAUSS, 2) if etype == L.H8 else (L.RULE_TET, 4)), [1.0])
    out = M.checksum()
    M.close()
    mesh.close()
    for p in bufs:
        hiprt.hipFree(p)
    return out


def test_growing_and_shrinking(ctx, hiprt):
    want = {n: device_digest(ctx, hiprt, n) for n in SIZES}
    for n in SIZES + SIZES[::-1]:
        assert digest(ctx, n) == want[n]
        assert digest(ctx, n, columns=True) == want[n]


@pytest.mark.parametrize("n", [(1, 1, 1), (3, 1, 2), (8, 8, 8), (9, 9, 9)])
def test_t10(ctx, hiprt, n):
    assert digest(ctx, n, etype=L.T10) == device_digest(ctx, hiprt, n, L.T10)


def test_threads(ctx):
    want = {n: digest(ctx, n) for n in SIZES}
    bad = []

    def work(k):
        own = core.Context(0)
        for n in SIZES[k % 3::2]:
            if digest(own, n) != want[n]:
                bad.append((k, n))
        own.close()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
