"""Performance cases of the assembly library: what a program that uses it
spends its device time on, through the public entry points.

listed() names the cases, draw() gives more of the same ranges, prepare() makes
what a program has in hand before the call (host or device inputs, the
resident mesh, its pattern and its result matrix), run() is one pass, work()
the bytes and operations it cannot do without, and exact() the same result in
64 bits from plain torch.

Meshes are structured H8 or T10 blocks with seeded node perturbations, as the
library's own benchmark uses; every size is a number of cells per axis (a T10
cell is six tetrahedra).  Kinds of case:

  reassemble  values into a resident CSC pattern (the numeric phase that a
              time-stepping, nonlinear or parameter-study program repeats)
  bilform     a new device matrix from a mesh whose numbering puts the fixed
              DOFs last (essential boundary conditions): the general numbering
  new_mesh    host arrays -> device mesh -> numbering -> first matrix
  served      one request of a new mesh to the assembly server
  sparse      device triples -> CSC (makematrix! of an external element loop)
  load        load vector of a constant body force
  lumped      HRZ-lumped mass
  batch       many uneven meshes in one launch sequence
"""
import ctypes
import functools
import os
import sys

import torch  # before the library: both then share one HIP runtime
import numpy as np

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "finetools.jl_amd"))

import feasm  # noqa: E402
from feasm import _lib as L  # noqa: E402
from feasm import core  # noqa: E402

FORMS = {"elastic": L.LIN_ELASTIC, "elastic-general": L.LIN_ELASTIC, "diffusion": L.DIFFUSION_ISO,
         "diffusion-tensor": L.DIFFUSION_MAT, "mass": L.DOT}


def listed():
    return [
        # stiffness values of a million-element block, the library's headline workload
        {"name": "h8-elastic-1m", "kind": "reassemble", "elem": "h8", "nx": 100, "ny": 100, "nz": 100,
         "form": "elastic", "order": 2, "mixed": False},
        # the same call on a coarse test mesh: launch and host latency
        {"name": "h8-elastic-small", "kind": "reassemble", "elem": "h8", "nx": 6, "ny": 5, "nz": 4,
         "form": "elastic", "order": 2, "mixed": False},
        # heat conduction, one DOF per node, uneven block
        {"name": "h8-diffusion", "kind": "reassemble", "elem": "h8", "nx": 71, "ny": 53, "nz": 47,
         "form": "diffusion", "order": 2, "mixed": False},
        # quadratic tetrahedra stiffness, the usual solid mesh
        {"name": "t10-elastic", "kind": "reassemble", "elem": "t10", "nx": 33, "ny": 29, "nz": 31,
         "form": "elastic", "order": 4, "mixed": False},
        # consistent mass of quadratic tetrahedra in mixed precision
        {"name": "t10-mass-mixed", "kind": "reassemble", "elem": "t10", "nx": 23, "ny": 25, "nz": 21,
         "form": "mass", "order": 4, "mixed": True},
        # first assembly of a mesh that comes from host arrays
        {"name": "new-mesh", "kind": "new_mesh", "elem": "h8", "nx": 45, "ny": 41, "nz": 37,
         "form": "elastic", "order": 2, "mixed": False},
        # a median request of the served stream
        {"name": "served-new-mesh", "kind": "served", "elem": "t10", "nx": 20, "ny": 20, "nz": 20,
         "form": "elastic", "order": 4, "mixed": True},
        # stiffness with one face fixed (free DOFs numbered first)
        {"name": "ebc-numbering", "kind": "bilform", "elem": "h8", "nx": 36, "ny": 33, "nz": 31,
         "form": "elastic", "order": 2, "mixed": False},
        # triples of an external element loop
        {"name": "sparse-triples", "kind": "sparse", "elem": "h8", "nx": 29, "ny": 27, "nz": 25,
         "form": "elastic", "order": 2, "mixed": False},
        # body load
        {"name": "load-vector", "kind": "load", "elem": "h8", "nx": 87, "ny": 79, "nz": 61,
         "form": "mass", "order": 2, "mixed": False},
        # lumped mass for explicit dynamics
        {"name": "lumped-mass", "kind": "lumped", "elem": "h8", "nx": 73, "ny": 61, "nz": 59,
         "form": "mass", "order": 2, "mixed": False},
        # many uneven meshes, diffusion and elasticity alternating
        {"name": "batch-mixed", "kind": "batch", "elem": "h8", "nmesh": 24, "nmax": 40, "nx": 0, "ny": 0, "nz": 0,
         "form": "elastic", "order": 2, "mixed": True},
    ]


def draw(rng):
    kind = rng.choice(["reassemble"] * 5 + ["bilform", "new_mesh", "served", "sparse", "load", "lumped", "batch"])
    elem = rng.choice(["h8", "t10"])
    # the most elements of each kind (the listed cases span the same range)
    most = {"reassemble": 6e5, "bilform": 4e4, "new_mesh": 7e4, "served": 5e4, "sparse": 2e4, "load": 5e5,
            "lumped": 3e5, "batch": 0}[kind]
    form = {"load": "mass", "lumped": "mass", "batch": "elastic"}.get(kind) or rng.choice(
        ["elastic", "elastic", "diffusion", "mass", "elastic-general", "diffusion-tensor"])
    if kind == "sparse":
        form = "elastic"
    usual = 2 if elem == "h8" else 4
    # now and then a rule beyond the usual one
    order = rng.choice([usual] * 5 + [usual + 1]) if kind in ("reassemble", "load", "lumped") else usual
    mixed = kind in ("reassemble", "bilform", "new_mesh", "served", "batch") and rng.random() < 0.4
    case = {"kind": kind, "elem": elem, "form": form, "order": order, "mixed": mixed}
    if kind == "batch":
        case.update(elem="h8", order=2, nmesh=rng.randint(3, 24), nmax=rng.randint(8, 40), nx=0, ny=0, nz=0)
        return case
    if elem == "t10" or form == "elastic-general" or order != usual:
        most /= 3  # more work per element
    cells = 64.0 * (most / (6 if elem == "t10" else 1) / 64.0) ** rng.random()
    ax = [rng.uniform(0.6, 1.6) for _ in range(3)]
    scale = (cells / (ax[0] * ax[1] * ax[2])) ** (1.0 / 3.0)
    case.update({k: max(1, int(a * scale)) for k, a in zip(("nx", "ny", "nz"), ax)})
    return case


# ------------------------------------------------------------------ meshes
TETS = np.array([[1, 8, 5, 6], [3, 4, 2, 7], [7, 2, 6, 8], [4, 7, 8, 2], [2, 1, 6, 8], [4, 8, 1, 2]]) - 1
EDGES = [(0, 1), (1, 2), (2, 0), (3, 0), (3, 1), (3, 2)]


def _corners(nx, ny, nz):
    """The eight corner nodes (0-based) of every cell; nodes x fastest."""
    i, j, k = np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij")
    f = (i + (nx + 1) * (j + (ny + 1) * k)).transpose(2, 1, 0).reshape(-1, 1).astype(np.int64)
    low = np.array([0, 1, nx + 2, nx + 1], np.int64)
    return f + np.concatenate([low, low + (nx + 1) * (ny + 1)])


@functools.lru_cache(maxsize=3)
def _t10_topology(nx, ny, nz):
    """Connectivity (0-based, elements x 10), edge end nodes."""
    nv = (nx + 1) * (ny + 1) * (nz + 1)
    tet = _corners(nx, ny, nz)[:, TETS].reshape(-1, 4)
    ends = np.stack([np.sort(tet[:, list(e)], axis=1) for e in EDGES], axis=1)
    key, inv = np.unique(ends[..., 0] * nv + ends[..., 1], return_inverse=True)
    return np.concatenate([tet, nv + inv.reshape(-1, 6)], axis=1), np.stack([key // nv, key % nv], axis=1)


def _mesh(elem, nx, ny, nz, rng):
    """(connectivity, 1-based; coordinates) of a perturbed block."""
    h = 1.0 / max(nx, ny, nz)
    z, y, x = np.meshgrid(np.arange(nz + 1) * h, np.arange(ny + 1) * h, np.arange(nx + 1) * h, indexing="ij")
    xyz = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    top = np.array([nx, ny, nz]) * h

    def moved(p, amp):
        inside = np.all((p > 1e-9) & (p < top - 1e-9), axis=1, keepdims=True)
        return p + inside * rng.uniform(-amp * h, amp * h, p.shape)

    if elem == "h8":
        return _corners(nx, ny, nz) + 1, moved(xyz, 0.15)
    conn, ends = _t10_topology(nx, ny, nz)
    xyz = moved(xyz, 0.1)
    return conn + 1, np.concatenate([xyz, moved(xyz[ends].mean(axis=1), 0.03)])


def _coefficients(form, rng):
    if form == "diffusion":
        return np.array([rng.uniform(0.5, 2.0)])
    if form == "diffusion-tensor":
        a = rng.uniform(-0.3, 0.3, (3, 3))
        return np.diag(rng.uniform(1.0, 2.0, 3)) + (a + a.T) / 2
    if form == "mass":
        return rng.uniform(1.0, 8.0) * np.eye(3)
    E, nu = rng.uniform(1e3, 1e5), rng.uniform(0.2, 0.4)
    lam, mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
    D = np.diag([2 * mu] * 3 + [mu] * 3)
    D[:3, :3] += lam
    if form == "elastic-general":  # a stiffer direction and some coupling
        a = rng.uniform(-0.05, 0.05, (6, 6)) * mu
        D[0, 0] *= 3
        D += (a + a.T) / 2
    return D


def _dofs(case, xyz):
    """DOF numbers (1-based, nodes x ndn): node by node, or for the general
    numbering the free DOFs first and those of the face x = 0 last."""
    ndn = _ndn(case)
    n = xyz.shape[0] * ndn
    if case["kind"] != "bilform":
        return np.arange(1, n + 1).reshape(-1, ndn)
    fixed = np.repeat(xyz[:, 0] == 0.0, ndn)
    d = np.where(fixed, np.cumsum(fixed) + (~fixed).sum(), np.cumsum(~fixed))
    return d.reshape(-1, ndn)


def _ndn(case):
    return 1 if case["form"].startswith("diffusion") else 3


def _members(case, rng):
    """(elem, n, form, coefficients) of a batch's meshes; the sizes belong to
    the case, the rest to its inputs."""
    sizes = np.random.default_rng((case["nmesh"], case["nmax"])).integers(4, case["nmax"] + 1, (case["nmesh"], 3))
    for i in range(case["nmesh"]):
        n = tuple(int(v) for v in sizes[i])
        form = "diffusion" if i % 2 == 0 else "elastic"
        yield case["elem"], n, form, _coefficients(form, rng)


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    conn, xyz = _mesh(case["elem"], case["nx"], case["ny"], case["nz"], rng)
    return conn, xyz, _coefficients(case["form"], rng), rng


# ------------------------------------------------------------------ device arrays
class _Owned:
    """A device array of the library as torch sees it, with its owner."""

    def __init__(self, ptr, n, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (ptr, False), "version": 2}


def _view(ptr, n, typestr, owner):
    if n == 0:
        return torch.empty(0, dtype={"<i8": torch.int64, "<i4": torch.int32, "<f8": torch.float64}[typestr],
                           device="cuda")
    return torch.as_tensor(_Owned(ptr, n, typestr, owner), device="cuda")


def _csc(mat, owner=None):
    """A device matrix's arrays, as a program hands them to its solver."""
    _, n, nnz = mat.dims
    c, r, v = mat.device_ptrs()
    own = (mat, owner)
    return {"colptr": _view(c, n + 1, "<i8", own), "rowval": _view(r, nnz, "<i4", own),
            "nzval": _view(v, nnz, "<f8", own)}


@functools.lru_cache(maxsize=1)
def _context():
    return feasm.Context(0)


# ------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    kind, ctx = case["kind"], _context()
    prec = L.MIXED if case["mixed"] else L.FP64
    s = {"kind": kind, "prec": prec}
    if kind == "batch":
        rng = np.random.default_rng(seed)
        s["batch"], s["meshes"] = core.Batch(ctx), []
        for elem, n, form, coeff in _members(case, rng):
            conn, xyz = _mesh(elem, *n, rng)
            mesh = core.DeviceMesh(ctx, L.H8, conn, xyz)
            mesh.set_dofs(1 if form == "diffusion" else 3)
            s["batch"].add(mesh, FORMS[form], L.RULE_GAUSS, 2, coeff, prec)
            s["meshes"].append(mesh)
        s["batch"].prepare(use_graph=True)
        mats = [s["batch"].matrix(i) for i in range(case["nmesh"])]
        s["out"] = [_view(m.device_ptrs()[2], m.nnz, "<f8", s["batch"]) for m in mats]
        return s
    conn, xyz, coeff, rng = _inputs(case, seed)
    etype, ndn = (L.H8, L.T10)[case["elem"] == "t10"], _ndn(case)
    rule = L.RULE_GAUSS if etype == L.H8 else L.RULE_TET
    s.update(etype=etype, conn=conn, xyz=xyz, ndn=ndn, args=(FORMS[case["form"]], rule, case["order"], coeff))
    if kind == "new_mesh":
        return s
    if kind == "served":
        s["server"], s["rid"] = core.Server(0, workers=4, hbm_fraction=0.2), None
        return s
    if kind == "sparse":
        d = torch.from_numpy(_dofs(case, xyz)[conn - 1].reshape(conn.shape[0], -1) - 1).to("cuda", torch.int32)
        k = d.shape[1]
        s["J"] = d[:, :, None].expand(-1, k, k).contiguous().view(-1)  # columns slowest, as assemble! buffers them
        s["I"] = d[:, None, :].expand(-1, k, k).contiguous().view(-1)
        s["V"] = _triple_values(s["I"].numel(), seed)
        s["n"] = ndn * xyz.shape[0]
        return s
    mesh = s["mesh"] = core.DeviceMesh(ctx, etype, conn, xyz)
    if kind == "bilform":
        mesh.set_dofs(ndn, _dofs(case, xyz), ndn * xyz.shape[0])
        return s
    mesh.set_dofs(ndn)
    if kind == "reassemble":
        s["mat"] = mesh.bilform(*s["args"], precision=prec)
        s["out"] = _view(s["mat"].device_ptrs()[2], s["mat"].nnz, "<f8", s["mat"])
    elif kind == "load":
        s["force"] = np.ascontiguousarray(rng.uniform(-10.0, 10.0, ndn))
        s["F"] = torch.empty(ndn * xyz.shape[0], dtype=torch.float64, device="cuda")
    return s


def _triple_values(n, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(n, dtype=torch.float64, device="cuda", generator=g)


def run(s):
    kind, ctx = s["kind"], _context()
    if kind == "reassemble":
        s["mesh"].bilform_into(s["mat"], *s["args"], precision=s["prec"])
        return {"nzval": s["out"]}
    if kind == "bilform":
        return _csc(s["mesh"].bilform(*s["args"], precision=s["prec"]))
    if kind == "new_mesh":
        mesh = core.DeviceMesh(ctx, s["etype"], s["conn"], s["xyz"])
        mesh.set_dofs(s["ndn"])
        return _csc(mesh.bilform(*s["args"], precision=s["prec"]), mesh)
    if kind == "served":
        srv = s["server"]
        rid, _ = srv.submit_mesh(s["etype"], s["conn"], s["xyz"], s["ndn"], *s["args"], precision=s["prec"], borrow=True)
        status, _, _ = srv.wait(rid)
        if status != 2:
            raise RuntimeError("request ended with status %d" % status)
        before, s["rid"] = s["rid"], rid
        if before is not None:
            srv.release(before)
        return _csc(srv.result(rid), srv)
    if kind == "sparse":
        h = ctypes.c_void_p()
        L.check(L.lib().feasm_sparse_device(ctx.h, s["V"].numel(), s["I"].data_ptr(), s["J"].data_ptr(),
                                            s["V"].data_ptr(), s["n"], s["n"], ctypes.byref(h)), ctx.h)
        return _csc(core.DeviceMatrix(ctx, h))
    if kind == "load":
        _, rule, order, _ = s["args"]
        L.check(L.lib().feasm_linform_dot_device(s["mesh"].h, rule, order, L.ptr(s["force"]), len(s["force"]),
                                                 s["F"].data_ptr()), ctx.h)
        return {"F": s["F"]}
    if kind == "lumped":
        _, rule, order, coeff = s["args"]
        return _csc(s["mesh"].bilform_dot_lumped(rule, order, coeff))
    s["batch"].run()
    return {"nzval": s["out"]}


# ------------------------------------------------------------------ work
def _sizes(elem, nx, ny, nz):
    """(elements, nodes, node pairs that share an element) of a block."""
    v = (nx + 1) * (ny + 1) * (nz + 1)
    if elem == "h8":
        return nx * ny * nz, v, (3 * nx + 1) * (3 * ny + 1) * (3 * nz + 1)
    t = 6 * nx * ny * nz
    e = (nx * (ny + 1) * (nz + 1) + (nx + 1) * ny * (nz + 1) + (nx + 1) * (ny + 1) * nz + nx * ny * (nz + 1) +
         nx * (ny + 1) * nz + (nx + 1) * ny * nz + nx * ny * nz)
    f = 1 - v + e + t  # Euler's formula for a ball
    return t, v + e, v + 7 * e + 12 * f + 6 * t


def work(case):
    if case["kind"] == "batch":
        total = {"bytes": 0, "flops": 0}
        for elem, n, form, _ in _members(case, np.random.default_rng(1)):
            w = work(dict(case, kind="reassemble", nx=n[0], ny=n[1], nz=n[2], form=form))
            total = {k: total[k] + w[k] for k in total}
        return total
    ne, nn, nb = _sizes(case["elem"], case["nx"], case["ny"], case["nz"])
    npe, ndn = (8, 10)[case["elem"] == "t10"], _ndn(case)
    nqp = case["order"] ** 3 if case["elem"] == "h8" else case["order"]
    n, nnz = ndn * nn, ndn * ndn * nb
    mesh = 4 * npe * ne + 24 * nn
    csc = 8 * (n + 1) + 12 * nnz
    jac = nqp * (18 * npe + 15)  # J = X' dN, its determinant and the weight
    grad = nqp * (38 + 15 * npe)
    pairs = npe * (npe + 1) // 2
    per = {"elastic": jac + grad + 18 * nqp * pairs, "elastic-general": jac + grad + 18 * nqp * pairs,
           "diffusion": jac + grad + 6 * nqp * pairs, "diffusion-tensor": jac + grad + 18 * nqp * pairs,
           "mass": jac + 2 * nqp * pairs}[case["form"]]
    material = {"elastic": 32, "elastic-general": 162, "diffusion": 0, "diffusion-tensor": 18, "mass": 9}[case["form"]]
    matrix = ne * per + nb * material
    kind = case["kind"]
    if kind == "reassemble":
        return {"bytes": mesh + 8 * nnz, "flops": matrix}
    if kind == "bilform":
        return {"bytes": mesh + 4 * n + csc, "flops": matrix}
    if kind in ("new_mesh", "served"):
        return {"bytes": 8 * npe * ne + 24 * nn + csc, "flops": matrix}
    if kind == "sparse":
        nt = ne * (npe * ndn) ** 2
        return {"bytes": 16 * nt + csc, "flops": nt - nnz}
    if kind == "load":
        return {"bytes": mesh + 4 * n + 8 * n, "flops": ne * (jac + 2 * nqp * npe)}
    return {"bytes": mesh + 4 * n + 8 * (n + 1) + 12 * n, "flops": ne * (jac + 2 * nqp * npe)}  # lumped


# ------------------------------------------------------------------ exact values
def _rule(elem, order):
    """Points and weights as the reference types them."""
    if elem == "t10":
        if order == 4:
            a, b = 0.13819660, 0.58541020
            return np.array([[a, a, a], [b, a, a], [a, b, a], [a, a, b]]), np.full(4, 1.0 / 24)
        a = 1.0 / 6
        return (np.array([[0.25] * 3, [0.5, a, a], [a, 0.5, a], [a, a, 0.5], [a, a, a]]),
                np.array([-0.8, 0.45, 0.45, 0.45, 0.45]) / 6)
    p, w = {2: ([-0.577350269189626, 0.577350269189626], [1.0, 1.0]),
            3: ([-0.774596669241483, 0.0, 0.774596669241483],
                [0.5555555555555556, 0.8888888888888889, 0.5555555555555556])}[order]
    p, w = np.array(p), np.array(w)
    pts = np.stack(np.meshgrid(p, p, p, indexing="ij"), axis=-1).reshape(-1, 3)
    return pts, (w[:, None, None] * w[None, :, None] * w[None, None, :]).ravel()


def _basis(elem, pts):
    """N (points x nodes), dN (points x nodes x 3) on the device."""
    if elem == "h8":
        sign = np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1], [-1, -1, 1], [1, -1, 1], [1, 1, 1],
                         [-1, 1, 1]])
        f = 1.0 + sign[None] * pts[:, None, :]
        N = f.prod(axis=2) / 8
        dN = np.stack([sign[None, :, k] * f[..., (k + 1) % 3] * f[..., (k + 2) % 3] for k in range(3)], axis=2) / 8
    else:
        bary = np.concatenate([1 - pts.sum(axis=1, keepdims=True), pts], axis=1)
        db = np.array([[-1.0, -1, -1], [1, 0, 0], [0, 1, 0], [0, 0, 1]])
        N = [b * (2 * b - 1) for b in bary.T] + [4 * bary[:, i] * bary[:, j] for i, j in EDGES]
        dN = [(4 * bary[:, i:i + 1] - 1) * db[i] for i in range(4)]
        dN += [4 * (bary[:, i:i + 1] * db[j] + bary[:, j:j + 1] * db[i]) for i, j in EDGES]
        N, dN = np.stack(N, axis=1), np.stack(dN, axis=1)
    return torch.from_numpy(N).cuda(), torch.from_numpy(np.ascontiguousarray(dN)).cuda()


def _jacobians(elem, order, X):
    """X: elements x nodes x 3.  N, dN, J w (elements x points) and inverse Jacobians."""
    pts, w = _rule(elem, order)
    N, dN = _basis(elem, pts)
    J = torch.matmul(X.transpose(1, 2).contiguous()[:, None], dN[None])  # J[r][c] = sum_a X[a][r] dN[a][c]
    det = torch.linalg.det(J)
    return N, dN, det * torch.from_numpy(w).cuda(), J


def _element_blocks(case, form, coeff, X):
    """Element matrices as elements x column node x row node x ndn x ndn
    (row component, then column component)."""
    N, dN, jw, J = _jacobians(case["elem"], case["order"], X)
    c = torch.from_numpy(np.ascontiguousarray(coeff)).cuda()
    ne, npe = X.shape[0], X.shape[1]
    if form == "mass":
        m = torch.matmul(jw, (N[:, :, None] * N[:, None, :]).reshape(len(N), -1)).view(ne, npe, npe)
        return m[..., None, None] * c
    g = torch.matmul(dN[None], torch.linalg.inv(J))  # elements x points x nodes x 3
    g = g.reshape(ne, len(N), npe * 3)
    M = torch.bmm((g * jw[..., None]).transpose(1, 2).contiguous(), g)  # (a, k), (b, l)
    M = M.view(ne, npe, 3, npe, 3).permute(0, 3, 1, 2, 4).reshape(ne, npe, npe, 9)  # column b, row a, (k, l)
    if form == "diffusion":
        return (c * (M[..., 0] + M[..., 4] + M[..., 8]))[..., None, None]
    if form == "diffusion-tensor":
        return torch.matmul(M, c.reshape(9, 1))[..., None]
    v = torch.tensor([[0, 3, 4], [3, 1, 5], [4, 5, 2]], device="cuda")
    T = c[v[:, :, None, None], v[None, None, :, :]]  # i k j l
    return torch.matmul(M, T.permute(1, 3, 0, 2).reshape(9, 9)).view(ne, npe, npe, 3, 3)


def _exact_values(case, form, conn, xyz, coeff, dofs):
    """CSC values of the assembled matrix for the numbering dofs (1-based)."""
    c, x = torch.from_numpy(conn - 1).cuda(), torch.from_numpy(xyz).cuda()
    ne, npe, nn, ndn = c.shape[0], c.shape[1], x.shape[0], dofs.shape[1]
    key = (c[:, :, None] * nn + c[:, None, :]).reshape(-1)  # column node, row node
    blocks, where = torch.unique(key, return_inverse=True)
    del key
    where = where.view(ne, -1)
    val = torch.zeros(blocks.numel(), ndn * ndn, dtype=torch.float64, device="cuda")
    for e in range(0, ne, 32768):
        b = _element_blocks(case, form, coeff, x[c[e:e + 32768]])
        val.index_add_(0, where[e:e + 32768].reshape(-1), b.reshape(-1, ndn * ndn))
    del where
    d = torch.from_numpy(dofs - 1).cuda()
    row, col = d[blocks % nn], d[blocks // nn]
    order = torch.argsort((col[:, None, :] * (nn * ndn) + row[:, :, None]).reshape(-1))
    return val.reshape(-1)[order]


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        rng, out = np.random.default_rng(seed), []
        for elem, n, form, coeff in _members(case, rng):
            conn, xyz = _mesh(elem, *n, rng)
            dofs = np.arange(1, xyz.shape[0] * (1 if form == "diffusion" else 3) + 1).reshape(xyz.shape[0], -1)
            out.append(_exact_values(case, form, conn, xyz, coeff, dofs))
        return {"nzval": out}
    conn, xyz, coeff, rng = _inputs(case, seed)
    dofs = _dofs(case, xyz)
    n = dofs.size
    if kind == "reassemble":
        return {"nzval": _exact_values(case, case["form"], conn, xyz, coeff, dofs)}
    if kind in ("bilform", "new_mesh", "served"):
        return {"colptr": None, "rowval": None, "nzval": _exact_values(case, case["form"], conn, xyz, coeff, dofs)}
    if kind == "sparse":
        d = torch.from_numpy(dofs[conn - 1].reshape(conn.shape[0], -1) - 1).cuda()
        _, where = torch.unique((d[:, :, None] * n + d[:, None, :]).reshape(-1), return_inverse=True)
        val = torch.zeros(int(where.max()) + 1, dtype=torch.float64, device="cuda")
        return {"colptr": None, "rowval": None,
                "nzval": val.index_add_(0, where, _triple_values(where.numel(), seed))}
    c, x = torch.from_numpy(conn - 1).cuda(), torch.from_numpy(xyz).cuda()
    N, _, jw, _ = _jacobians(case["elem"], case["order"], x[c])
    out = torch.zeros(xyz.shape[0], 3, dtype=torch.float64, device="cuda")
    if kind == "load":
        force = torch.from_numpy(rng.uniform(-10.0, 10.0, 3)).cuda()
        out.index_add_(0, c.reshape(-1), torch.matmul(jw, N).reshape(-1, 1) * force)
        return {"F": out.view(-1)}
    m = torch.matmul(jw, N * N)  # lumped: the diagonal scaled to the element's total
    rho = torch.from_numpy(coeff).cuda()
    total = torch.matmul(jw, N.sum(dim=1) ** 2) * rho.sum()
    diag = m[..., None] * rho.diagonal()
    diag = diag * (total / diag.sum(dim=(1, 2)))[:, None, None]
    out.index_add_(0, c.reshape(-1), diag.reshape(-1, 3))
    return {"colptr": None, "rowval": None, "nzval": out.view(-1)}
