"""The workloads that assembly speed is judged by: sizes, inputs, one pass of each, and what it must return.

A case is one use of the library through its public entry points (the ctypes binding fem_amd): a resident plan, a
residual-only plan, the drop-in dispatchers with the reference's arguments, the NONLINEAR strain, a batch of resident
meshes, the device-side pattern and map. Meshes are the repository's two shapes, the unit square and the annulus with
a periodic seam, on tensor-product cosine knots with interior nodes moved by up to a fifth of the gap beside them.
Their nodes are numbered either "tensor" (row by row, as the repository's own generators do) or "entity" (all corner
nodes, then nodes on edges, then interior nodes: the order in which mesh generators such as gmsh number a high-order
mesh, so an element's columns are scattered over a matrix row).

exact() forms the same outputs in float64 with torch alone, with node coordinates and displacements taken relative to
the element's first node (the gradients of the basis sum to zero, so nothing changes but the cancellation).
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-fem-project_amd"))
import fem_amd as F  # noqa: E402

YOUNG, POISSON, THICKNESS = 70e9, 0.3, 1.0
JITTER = 0.2


# ---- the cases ---------------------------------------------------------------------------------------
def _case(name, what, shape, nx, ny, order, precision="fp64", numbering="tensor", flags="", meshes=1):
    return {"name": name, "what": what, "shape": shape, "nx": nx, "ny": ny, "order": order, "precision": precision,
            "numbering": numbering, "flags": flags, "meshes": meshes}


def listed():
    return [
        # The smallest resident assembly: the 64 x 64 bilinear mesh of the reference's CPU configuration, where
        # launches and the latency of one part count.
        _case("plan-p1-64", "plan", "square", 64, 64, 1),
        # The headline: residual and Jacobian of one million quadratic elements in FP64.
        _case("plan-p2-1000", "plan", "square", 1000, 1000, 2),
        # The high-order headline: the 250 000-element quartic annulus in FP64.
        _case("plan-p4-annulus", "plan", "annulus", 200, 1250, 4),
        # A served mid-size quadratic mesh: mixed precision, generator numbering, ragged sizes.
        _case("plan-p2-mixed", "plan", "annulus", 97, 411, 2, "mixed", "entity"),
        # A served mid-size cubic mesh in mixed precision.
        _case("plan-p3-mixed", "plan", "square", 151, 149, 3, "mixed", "entity"),
        # Residual evaluations of a line search: a residual-only plan, no matrix.
        _case("plan-residual-p2", "plan", "square", 701, 699, 2, flags="residual"),
        # The reference's residual dispatcher on its profiled mesh size (one million unknowns, quadratic).
        _case("dropin-residual-p2", "residual", "square", 351, 350, 2, numbering="entity"),
        # The reference's Jacobian dispatcher on the same mesh: outputs zeroed, then added to.
        _case("dropin-jacobian-p2", "jacobian", "square", 351, 350, 2, numbering="entity"),
        # The same dispatcher at order 4 and one million unknowns.
        _case("dropin-jacobian-p4", "jacobian", "square", 175, 175, 4, numbering="entity"),
        # A Newton step of the NONLINEAR (Green) strain at order 3 and one million unknowns: tangent and residual.
        _case("nonlinear-p3", "nonlinear", "square", 243, 241, 3, numbering="entity"),
        # Many small and mid-size resident meshes of all orders in one recorded batch call, mixed precision.
        _case("batch-mixed", "batch", "square", 90, 110, 0, "mixed", "tensor", "graph", 24),
        # Set-up of a new mesh on the device: block pattern and element map (whole numbers).
        _case("pattern-p2", "pattern", "square", 500, 500, 2, numbering="entity"),
    ]


def draw(rng):
    what = rng.choice(["plan", "plan", "plan", "plan-residual", "residual", "jacobian", "nonlinear", "batch", "pattern"])
    flags = ""
    if what == "plan-residual":
        what, flags = "plan", "residual"
    order = rng.randint(1, 4)
    shape = rng.choice(["square", "square", "annulus"])
    numbering = rng.choice(["tensor", "entity"])
    precision = "fp64" if what in ("nonlinear", "pattern") else rng.choice(["fp64", "mixed"])
    if what == "plan" and not flags:
        flags = rng.choice(["", "", "", "deterministic"])
    most = {1: 1.5e6, 2: 8e5, 3: 3e5, 4: 1.8e5}[order]  # elements
    if what == "pattern":
        most = min(most, 2.5e5)
    elif what in ("jacobian", "nonlinear"):
        most /= 3
    meshes = 1
    if what == "batch":
        order, shape, numbering, flags = 0, "square", "tensor", rng.choice(["graph", ""])
        meshes = rng.randint(2, 24)
        most = 2e4
    elements = math.exp(rng.uniform(math.log(60.0), math.log(most)))
    aspect = math.exp(rng.uniform(-1.0, 1.0))
    nx = max(1, round(math.sqrt(elements * aspect)))
    ny = max(3, round(elements / nx))
    if shape == "annulus":
        ny = max(ny, _least_around(nx))
    c = _case("", what, shape, nx, ny, order, precision, numbering, flags, meshes)
    del c["name"]
    return c


def _least_around(nx):
    """Elements around an annulus of nx radial elements whose straight-sided quads all keep a positive Jacobian."""
    return max(12, math.ceil(7.0 * math.sqrt(nx)))


# ---- meshes and fields -------------------------------------------------------------------------------
def _members(case):
    """The (order, shape, nx, ny) of each mesh of a case: one, or a batch's, of all orders around nx x ny."""
    if case["what"] != "batch":
        return [(case["order"], case["shape"], case["nx"], case["ny"])]
    out = []
    for i in range(case["meshes"]):
        order = 1 + i % 4
        scale = (0.3, 0.55, 1.0)[i % 3] * (1.6, 1.0, 0.8, 0.6)[order - 1]
        shape = "annulus" if i % 5 == 4 else "square"
        nx, ny = max(1, round(case["nx"] * scale) + i % 3), max(3, round(case["ny"] * scale) - i % 2)
        out.append((order, shape, nx, max(ny, _least_around(nx)) if shape == "annulus" else ny))
    return out


def _knots(n, p):
    j = np.arange(p * n + 1)
    e = np.minimum(j // p, n - 1)
    return (e + 0.5 * (1.0 - np.cos(np.pi * (j - e * p) / p))) / n


def _gaps(x, periodic):
    d = np.diff(x)
    left, right = np.concatenate([d[-1:] if periodic else d[:1], d]), np.concatenate([d, d[:1] if periodic else d[-1:]])
    return np.minimum(left, right)


def _mesh(member, numbering, seed):
    """(coords [nodes, 2], conn [elements, N] int32) of one mesh."""
    p, shape, nx, ny = member
    rng = np.random.default_rng([seed, p, nx, ny])
    periodic = shape == "annulus"
    kx, ky = _knots(nx, p), _knots(ny, p)
    gx, gy = _gaps(kx, False), _gaps(ky, periodic)
    if periodic:
        ky, gy = ky[:-1], gy[:-1]
    mx, my = kx.size, ky.size
    move = rng.uniform(-JITTER, JITTER, (my, mx, 2))
    move[:, [0, -1]] = 0
    if not periodic:
        move[[0, -1]] = 0
    x = kx[None, :] + move[..., 0] * gx[None, :]
    y = ky[:, None] + move[..., 1] * gy[:, None]
    if periodic:
        r, th = 1.0 + x, 2.0 * np.pi * y
        x, y = r * np.cos(th), r * np.sin(th)
    coords = np.stack([x, y], axis=-1).reshape(-1, 2)
    a = np.arange(p + 1)
    jx = (np.arange(nx)[:, None] * p + a).astype(np.int32)
    jy = ((np.arange(ny)[:, None] * p + a) % my).astype(np.int32)
    conn = (jy[:, None, :, None] * np.int32(mx) + jx[None, :, None, :]).reshape(nx * ny, (p + 1) ** 2)
    if numbering == "entity":  # corners, nodes on edges, interior nodes
        kind = ((np.arange(my) % p != 0).astype(np.int8)[:, None] + (np.arange(mx) % p != 0)[None, :]).reshape(-1)
        old = np.argsort(kind, kind="stable")
        new = np.empty(old.size, dtype=np.int32)
        new[old] = np.arange(old.size, dtype=np.int32)
        coords, conn = coords[old], new[conn]
    return np.ascontiguousarray(coords), np.ascontiguousarray(conn)


def _states(coords, seed, amplitude=1e-3):
    """A smooth displacement field with a small random part."""
    rng = np.random.default_rng([seed, 7])
    ph = rng.uniform(0.0, 2.0 * np.pi, 4)
    x, y = 2.0 * np.pi * coords[:, 0], 2.0 * np.pi * coords[:, 1]
    u = amplitude * (np.sin(x + ph[0]) + np.sin(y + ph[1]))
    v = amplitude * (np.cos(x + ph[2]) + np.cos(y + ph[3]))
    return (np.stack([u, v], axis=1) + rng.uniform(-1e-5, 1e-5, coords.shape)).reshape(-1)


def _line_blocks(n, p, periodic):
    inner = n * (p - 1) * (p + 1)
    return inner + (n * (2 * p + 1) if periodic else (n - 1) * (2 * p + 1) + 2 * (p + 1))


def _counts(member):
    """(nodes, elements, BSR blocks) of a mesh."""
    p, shape, nx, ny = member
    periodic = shape == "annulus"
    nodes = (p * nx + 1) * (p * ny if periodic else p * ny + 1)
    return nodes, nx * ny, _line_blocks(nx, p, False) * _line_blocks(ny, p, periodic)


# ---- one pass ----------------------------------------------------------------------------------------
def _prepare_one(case, member, seed):
    what, flags = case["what"], case["flags"]
    order = member[0]
    coords, conn = _mesh(member, case["numbering"], seed)
    states = _states(coords, seed, 1e-2 if what == "nonlinear" else 1e-3)
    mesh = F.Mesh(order, coords, conn)
    dev = torch.device("cuda")
    d = lambda x: torch.from_numpy(x).to(dev)  # noqa: E731
    s = {"what": what, "order": order, "ne": mesh.num_elements, "nn": mesh.num_nodes, "states": d(states),
         "coords": d(coords), "prec": F.FEM_PREC_MIXED if case["precision"] == "mixed" else F.FEM_PREC_FP64}
    if what == "pattern":  # elements in patches of 64, as a generator's fronts lay them down, in an order of the seed
        pad = -conn.shape[0] % 64
        ids = np.concatenate([np.arange(conn.shape[0]), np.full(pad, -1)]).reshape(-1, 64)
        ids = np.random.default_rng([seed, 3]).permutation(ids).reshape(-1)
        conn = conn[ids[ids >= 0]]
    if what in ("residual", "jacobian", "nonlinear", "pattern"):
        s["conn_ptr"], s["conn"] = d(mesh.conn_ptr), d(conn)
    if what == "pattern":
        return s
    s["res"] = torch.empty(2 * mesh.num_nodes, dtype=torch.float64, device=dev)
    if what == "residual":
        return s
    if what in ("jacobian", "nonlinear"):
        rowp, cols = F.bsr_pattern_device(s["nn"], s["ne"], mesh.npe, s["conn_ptr"], s["conn"])
        s["map"] = F.element_bcsr_map_device(s["conn_ptr"], s["conn"], s["ne"], mesh.npe, s["nn"], rowp, cols)
        blocks = cols.numel()
    else:
        pattern = F.bsr_pattern(mesh)
        bits = {"residual": F.FEM_PLAN_RESIDUAL_ONLY, "deterministic": F.FEM_PLAN_DETERMINISTIC}
        s["plan"] = F.Plan(mesh, pattern, flags=bits.get(flags, 0))
        blocks = pattern.num_blocks
    s["vals"] = None
    if flags != "residual":
        s["vals"] = torch.empty(4 * blocks, dtype=torch.float64, device=dev)
    return s


def prepare(case, seed):
    if case["what"] != "batch":
        return _prepare_one(case, _members(case)[0], seed)
    jobs = [_prepare_one(case, m, seed) for m in _members(case)]
    batch = F.Batch(max_jobs=32, graph=case["flags"] == "graph")
    for j in jobs:
        batch.add(j["plan"], j["states"], j["coords"], YOUNG, POISSON, THICKNESS, res=j["res"], values=j["vals"])
    return {"what": "batch", "jobs": jobs, "batch": batch, "prec": jobs[0]["prec"]}


def run(s):
    what = s["what"]
    if what == "plan":
        s["plan"].assemble(s["states"], s["coords"], YOUNG, POISSON, THICKNESS, res=s["res"], values=s["vals"],
                           precision=s["prec"])
    elif what == "batch":
        s["batch"].assemble(precision=s["prec"])
        return [[j["res"], j["vals"]] for j in s["jobs"]]
    elif what == "pattern":
        npe = (s["order"] + 1) ** 2
        rowp, cols = F.bsr_pattern_device(s["nn"], s["ne"], npe, s["conn_ptr"], s["conn"])
        return [rowp, cols, F.element_bcsr_map_device(s["conn_ptr"], s["conn"], s["ne"], npe, s["nn"], rowp, cols)]
    elif what == "residual":
        s["res"].zero_()
        F.residual(s["order"], s["conn_ptr"], s["conn"], s["ne"], s["states"], s["coords"], YOUNG, POISSON, THICKNESS,
                   s["res"], precision=s["prec"])
        return [s["res"]]
    else:  # the reference's dispatchers add to what the caller zeroed
        s["res"].zero_()
        s["vals"].zero_()
        F.jacobian(s["order"], s["conn_ptr"], s["conn"], s["ne"], s["states"], s["coords"], YOUNG, POISSON, THICKNESS,
                   s["map"], s["res"], s["vals"], precision=s["prec"], nonlinear=what == "nonlinear",
                   dropin=what == "jacobian")
    return [s["res"]] if s["vals"] is None else [s["res"], s["vals"]]


def work(case):
    """Coordinates, states and connectivity in, residual and blocks out (and, where the caller's element map is an
    input or an output, the map); the multiply-adds of the geometry, the residual and the weighted Gram sums."""
    nbytes = flops = 0.0
    what = case["what"]
    for m in _members(case):
        nodes, elements, blocks = _counts(m)
        n = q = (m[0] + 1) ** 2
        if what == "pattern":
            nbytes += 4 * n * elements + 4 * nodes + 4 * blocks + 4 * n * n * elements
            continue
        nbytes += 48 * nodes + 4 * n * elements
        flops += elements * q * (16.0 * n + 14.0 * n)
        if what != "residual" and case["flags"] != "residual":
            nbytes += 32 * blocks
            flops += elements * 2.0 * q * (2 * n * n + n) * (2 if what == "nonlinear" else 1)
        if what in ("jacobian", "nonlinear"):
            nbytes += 4 * n * n * elements
    return {"bytes": nbytes, "flops": flops}


# ---- the same outputs by torch in float64 -------------------------------------------------------------
def _basis(p):
    """Weights [Q] and reference gradients [Q, N, 2] of the tensor-product basis at the Gauss points."""
    x, w = np.polynomial.legendre.leggauss(p + 1)
    knots = -np.cos(np.pi * np.arange(p + 1) / p)
    v = np.zeros((p + 1, p + 1))
    dv = np.zeros((p + 1, p + 1))
    for j in range(p + 1):
        c = np.poly1d([1.0])
        for i in range(p + 1):
            if i != j:
                c = c * np.poly1d([1.0, -knots[i]]) / (knots[j] - knots[i])
        v[:, j], dv[:, j] = c(x), c.deriv()(x)
    n = p + 1
    g = np.zeros((n, n, n, n, 2))  # qy, qx, ay, ax
    g[..., 0] = v[:, None, :, None] * dv[None, :, None, :]
    g[..., 1] = dv[:, None, :, None] * v[None, :, None, :]
    return np.outer(w, w).reshape(-1), g.reshape(n * n, n * n, 2)


def _exact_one(case, member, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    p, what = member[0], case["what"]
    jac = what != "residual" and case["flags"] != "residual"
    coords_h, conn_h = _mesh(member, case["numbering"], seed)
    states_h = _states(coords_h, seed, 1e-2 if what == "nonlinear" else 1e-3)
    coords, conn = torch.from_numpy(coords_h).to(dev), torch.from_numpy(conn_h).to(dev).long()
    u = torch.from_numpy(states_h).to(dev).view(-1, 2)
    w, g = (torch.from_numpy(t).to(dev) for t in _basis(p))
    nodes, (elements, n) = coords.shape[0], conn.shape
    q = w.numel()
    mu = 0.5 * YOUNG / (1.0 + POISSON)
    lam = 2.0 * mu * POISSON / (1.0 - POISSON)
    res = torch.zeros((nodes, 2), dtype=torch.float64, device=dev)
    vals = slot = None
    if jac:
        keys = (conn[:, :, None] * nodes + conn[:, None, :]).reshape(-1)
        distinct, slot = torch.unique(keys, return_inverse=True)
        vals = torch.zeros((distinct.numel(), 4), dtype=torch.float64, device=dev)
        slot = slot.view(elements, n * n)
        del keys, distinct
    one = torch.eye(2, dtype=torch.float64, device=dev)
    gm = g.permute(1, 0, 2).reshape(n, 2 * q).contiguous()  # [N, (q, d)]
    chunk = 20000
    for at in range(0, elements, chunk):
        c = conn[at:at + chunk]
        e = c.shape[0]
        xe, ue = coords[c], u[c]
        xe, ue = xe - xe[:, :1], ue - ue[:, :1]

        def grad(f):  # [E, N, 2] nodal values to [E, Q, 2, 2] derivatives: component, reference direction
            return (f.transpose(1, 2).reshape(2 * e, n) @ gm).view(e, 2, q, 2).permute(0, 2, 1, 3)

        jm = grad(xe)
        det = jm[..., 0, 0] * jm[..., 1, 1] - jm[..., 0, 1] * jm[..., 1, 0]
        inv = torch.stack([jm[..., 1, 1], -jm[..., 0, 1], -jm[..., 1, 0], jm[..., 0, 0]], dim=-1).view(e, q, 2, 2)
        inv = inv / det[..., None, None]
        ux = (grad(ue)[..., :, :, None] * inv[..., None, :, :]).sum(-2)
        s = w * det * THICKNESS
        # physical gradients [E, Q, N, 2]
        ng = g[None, :, :, 0, None] * inv[:, :, None, 0, :] + g[None, :, :, 1, None] * inv[:, :, None, 1, :]
        strain = 0.5 * (ux + ux.transpose(-1, -2))
        if what == "nonlinear":
            strain = strain + 0.5 * (ux[..., :, :, None] * ux[..., :, None, :]).sum(-3)
        stress = 2.0 * mu * strain + lam * (strain[..., 0, 0] + strain[..., 1, 1])[..., None, None] * one
        force = stress
        if what == "nonlinear":
            f = one + ux
            force = (f[..., :, :, None] * stress[..., None, :, :]).sum(-2)
        r = ((s[..., None, None] * force)[:, :, None] * ng[..., None, :]).sum(-1).sum(1)
        res.index_add_(0, c.reshape(-1), r.reshape(-1, 2))
        if not jac:
            continue

        def gram(a, b):  # sum over points: [E, Q, X] and [E, Q, Y] to [E, X, Y]
            return torch.bmm(a.transpose(1, 2).contiguous(), b.contiguous())

        k = torch.zeros((e, n, n, 2, 2), dtype=torch.float64, device=dev)
        if what == "nonlinear":
            pg = (f[:, :, None] * ng[..., None, :]).sum(-1)
            t = gram((s[..., None, None] * pg).reshape(e, q, 2 * n), pg.reshape(e, q, 2 * n))
            t = t.view(e, n, 2, n, 2).permute(0, 1, 3, 2, 4)
            k += lam * t + mu * t.transpose(-1, -2)
            ff = (f[..., :, None, :] * f[..., None, :, :]).sum(-1)
            flat = ng.permute(0, 1, 3, 2).reshape(e, 2 * q, n)
            for i in range(2):
                for j in range(2):
                    wgt = (s * ff[..., i, j]).repeat_interleave(2, dim=1)[..., None]
                    k[..., i, j] += mu * gram(wgt * flat, flat)
            sn = (stress[:, :, None] * ng[..., None, :]).sum(-1)
            h = gram((s[..., None, None] * sn).permute(0, 1, 3, 2).reshape(e, 2 * q, n), flat)
            k[..., 0, 0] += h
            k[..., 1, 1] += h
        else:
            t = gram((s[..., None, None] * ng).reshape(e, q, 2 * n), ng.reshape(e, q, 2 * n))
            t = t.view(e, n, 2, n, 2).permute(0, 1, 3, 2, 4)
            k += lam * t + mu * t.transpose(-1, -2)
            dot = t[..., 0, 0] + t[..., 1, 1]
            k[..., 0, 0] += mu * dot
            k[..., 1, 1] += mu * dot
        vals.index_add_(0, slot[at:at + chunk].reshape(-1), k.reshape(-1, 4))
    res = res.reshape(-1)
    return [res] if vals is None else [res, vals.reshape(-1)]


def exact(case, seed):
    if case["what"] == "pattern":
        return None
    out = [_exact_one(case, m, seed) for m in _members(case)]
    return out if case["what"] == "batch" else out[0]
