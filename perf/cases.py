"""The work a user of this framework has it do, as cases that can be timed.

A case is a dict of plain values; prepare() makes what a program holds before
the call (mesh, matrix handle, right-hand sides on the device), run() takes it
through the framework's public entry points once.

Kinds:
  step     numeric assembly, penalty supports, Jacobi-PCG from zero with the
           vectors on the device: one load step of an analysis (the benchmark's
           step); nrhs > 1 solves all load cases together, mixed = 1 takes the
           FP32 inner iteration
  oneshot  a single analysis from mesh arrays on the host to displacements on
           the host: upload, structure and coloring on the device, assembly,
           penalty, solve
  force    new element moduli, assembly, supports, internal forces K u of a
           displacement field: the residual or sensitivity evaluation around a
           solver or a design loop
  group    many independent plates of uneven sizes assembled and solved as one
           system with new moduli (a parameter study)
  train    loss and parameter gradient of the warm-start network over one
           batch: forward and backward, the gradient read as an outer optimiser
           or a reduction over ranks reads it
"""
import ctypes as C
import math
import types

import numpy as np
import torch

import gpufem_amd as gf

E0, NU = 210000.0, 0.3
DIM = {"q4": 2, "q8": 2, "brick8": 3, "brick20": 3}
QUADRATIC = {"q4": False, "q8": True, "brick8": False, "brick20": True}
TYPE = {"q4": gf.GF_Q4, "q8": gf.GF_Q8, "brick8": gf.GF_BRICK8, "brick20": gf.GF_BRICK20}
NATURAL = {
    "q4": [(-1, -1), (1, -1), (1, 1), (-1, 1)],
    "q8": [(-1, -1), (0, -1), (1, -1), (1, 0), (1, 1), (0, 1), (-1, 1), (-1, 0)],
    "brick8": [(1, -1, -1), (1, 1, -1), (1, 1, 1), (1, -1, 1),
               (-1, -1, -1), (-1, 1, -1), (-1, 1, 1), (-1, -1, 1)],
    "brick20": [(1, -1, -1), (1, 0, -1), (1, 1, -1), (1, 1, 0), (1, 1, 1), (1, 0, 1), (1, -1, 1),
                (1, -1, 0), (0, -1, -1), (0, 1, -1), (0, 1, 1), (0, -1, 1), (-1, -1, -1),
                (-1, 0, -1), (-1, 1, -1), (-1, 1, 0), (-1, 1, 1), (-1, 0, 1), (-1, -1, 1),
                (-1, -1, 0)],
}
# neighbours per node inside a mesh and Jacobi-PCG iterations to 1e-8 per
# element along the longest side (about: for the work estimate only)
NEIGHBOURS = {"q4": 9.0, "q8": 15.7, "brick8": 27.0, "brick20": 60.0}
ITERATIONS = {"q4": 10.0, "q8": 13.0, "brick8": 16.0, "brick20": 40.0}


def listed():
    return [
        # the reference's smallest plate: latency and launches count
        {"name": "step_q4_64x32", "kind": "step", "elem": "q4", "nx": 64, "ny": 32, "nz": 0,
         "jitter": 0.0, "nrhs": 1, "mixed": 0, "rtol": 1e-8},
        # one analysis of a distorted mid-size plate, host to host
        {"name": "oneshot_q8_201x67", "kind": "oneshot", "elem": "q8", "nx": 201, "ny": 67,
         "nz": 0, "jitter": 0.15, "rtol": 1e-8},
        # a large 2D plate: thousands of iterations over a matrix that stays
        # in the last-level cache
        {"name": "step_q8_512x256", "kind": "step", "elem": "q8", "nx": 512, "ny": 256, "nz": 0,
         "jitter": 0.0, "nrhs": 1, "mixed": 0, "rtol": 1e-8},
        # the cantilever of the warm-start family: an ordinary 3D solve
        {"name": "step_brick8_64x32x32", "kind": "step", "elem": "brick8", "nx": 64, "ny": 32,
         "nz": 32, "jitter": 0.0, "nrhs": 1, "mixed": 0, "rtol": 1e-8},
        # the large 3D cube, streamed from HBM every iteration
        {"name": "step_brick8_96x96x96", "kind": "step", "elem": "brick8", "nx": 96, "ny": 96,
         "nz": 96, "jitter": 0.0, "nrhs": 1, "mixed": 0, "rtol": 1e-8},
        # mixed precision at the tolerance that meets FP64 accuracy, ragged box
        {"name": "mixed_brick8_83x97x71", "kind": "step", "elem": "brick8", "nx": 83, "ny": 97,
         "nz": 71, "jitter": 0.1, "nrhs": 1, "mixed": 1, "rtol": 1e-9},
        # 32 load cases of a 20-node cube advanced together
        {"name": "block32_brick20_24", "kind": "step", "elem": "brick20", "nx": 24, "ny": 24,
         "nz": 24, "jitter": 0.0, "nrhs": 32, "mixed": 0, "rtol": 1e-8},
        # an uneven number of load cases, mixed precision, ragged box
        {"name": "blockmixed12_brick20_20x17x13", "kind": "step", "elem": "brick20", "nx": 20,
         "ny": 17, "nz": 13, "jitter": 0.1, "nrhs": 12, "mixed": 1, "rtol": 1e-9},
        # a study over uneven small plates in one launch sequence
        {"name": "group_64_q4", "kind": "group", "count": 64, "lo": 16, "hi": 160, "sizes": 5,
         "rtol": 1e-8},
        # internal forces: assembly is most of the pass
        {"name": "force_brick8_101x90x88", "kind": "force", "elem": "brick8", "nx": 101, "ny": 90,
         "nz": 88, "jitter": 0.15},
        {"name": "force_brick20_30x33x28", "kind": "force", "elem": "brick20", "nx": 30, "ny": 33,
         "nz": 28, "jitter": 0.1},
        # the warm-start network on the cantilever's node grid, the training batch
        {"name": "train_65x33x33_b8", "kind": "train", "gx": 65, "gy": 33, "gz": 33, "batch": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "oneshot", "force", "force", "group", "train"])
    if kind == "train":
        g = [8 * rng.randint(2, 8) + 1, 8 * rng.randint(2, 4) + 1, 8 * rng.randint(2, 4) + 1]
        return {"kind": kind, "gx": g[0], "gy": g[1], "gz": g[2], "batch": rng.randint(1, 8)}
    if kind == "group":
        return {"kind": kind, "count": _log(rng, 4, 64), "lo": rng.randint(8, 24),
                "hi": rng.randint(40, 160), "sizes": rng.randint(1, 10 ** 6), "rtol": 1e-8}
    elem = rng.choice(["q4", "q8", "brick8", "brick8", "brick20"])
    if kind == "oneshot":
        top = {"q4": 40000, "q8": 14000, "brick8": 30000, "brick20": 4000}[elem]
    else:
        top = {"q4": 200000, "q8": 100000, "brick8": 500000, "brick20": 24000}[elem]
    nrhs, mixed = 1, 0
    if kind == "step":
        nrhs = rng.choice([1, 1, 1, 2, 5, 12, 24, 32])
        mixed = rng.choice([0, 0, 1]) if DIM[elem] == 3 else 0
        if nrhs > 1:
            top = {"q4": 20000, "q8": 8000, "brick8": 60000, "brick20": 8000}[elem]
    nel = _log(rng, 500, top)
    if DIM[elem] == 2:
        ny = max(4, int(math.sqrt(nel / rng.uniform(1.5, 3.0))))
        nx, nz = max(8, nel // ny), 0
    else:
        s = nel ** (1.0 / 3.0)
        ny, nz = max(3, int(s * rng.uniform(0.7, 1.2))), max(3, int(s * rng.uniform(0.7, 1.2)))
        nx = max(3, nel // (ny * nz))
    case = {"kind": kind, "elem": elem, "nx": nx, "ny": ny, "nz": nz,
            "jitter": rng.choice([0.0, 0.1, 0.15])}
    if kind == "step":
        case.update(nrhs=nrhs, mixed=mixed, rtol=1e-9 if mixed else 1e-8)
    elif kind == "oneshot":
        case.update(rtol=1e-8)
    return case


# ---- inputs -----------------------------------------------------------------
def _mesh(elem, nx, ny, nz, jitter, rng):
    """Connectivity (1-based), coordinates and the lattice points of the nodes:
    a box of unit elements, nodes numbered lexicographically (x fastest), the
    corners moved by up to `jitter` and midside nodes halfway between them."""
    d, quad = DIM[elem], QUADRATIC[elem]
    nel = (nx, ny, nz)[:d]
    m = 2 if quad else 1
    pts = [m * k + 1 for k in nel]
    axes = np.meshgrid(*[np.arange(p) for p in pts[::-1]], indexing="ij")[::-1]
    live = np.ones(pts[::-1], dtype=bool)
    if quad:
        live = sum(a % 2 for a in axes) <= 1
    number = np.cumsum(live.reshape(-1)).reshape(live.shape)
    corner = np.stack([a[tuple(slice(None, None, m) for _ in nel)] / m for a in axes], axis=-1)
    corner = corner.astype(np.float64)
    if jitter:
        corner = corner + rng.uniform(-jitter, jitter, corner.shape)
    full = corner
    if quad:
        full = np.zeros(live.shape + (d,))
        full[tuple(slice(None, None, 2) for _ in nel)] = corner
        for ax in range(d):  # halfway along one axis, the others at corners
            dst = [slice(None, None, 2)] * d
            dst[ax] = slice(1, None, 2)
            lo, hi = [slice(None)] * d, [slice(None)] * d
            lo[ax], hi[ax] = slice(0, -1), slice(1, None)
            full[tuple(dst)] = 0.5 * (corner[tuple(lo)] + corner[tuple(hi)])
    at = np.stack([a[live] for a in axes], axis=-1)
    coords = np.ascontiguousarray(full[live])
    cells = np.meshgrid(*[np.arange(k) for k in nel[::-1]], indexing="ij")[::-1]
    cells = [c.reshape(-1) for c in cells]
    conn = np.empty((cells[0].size, len(NATURAL[elem])), dtype=np.int32)
    for a, nat in enumerate(NATURAL[elem]):
        place = [m * c + (m * (x + 1)) // 2 for c, x in zip(cells, nat)]
        conn[:, a] = number[tuple(place[::-1])]
    return conn, coords, at, pts


def _problem(elem, nx, ny, nz, jitter, nrhs, seed):
    """Mesh, lognormal moduli, clamped face and nodal loads on the far face."""
    rng = np.random.default_rng(seed)
    conn, coords, at, pts = _mesh(elem, nx, ny, nz, jitter, rng)
    d = DIM[elem]
    moduli = E0 * np.exp(0.5 * rng.standard_normal(conn.shape[0]))
    # plates hang from x = 0 and carry their load on the far edge; a beam
    # (longest along x) likewise with a loaded top; cubes stand on z = 0
    beam = d == 3 and nx >= 2 * max(ny, nz)
    clamp_axis = 0 if d == 2 or beam else 2
    load_axis = 0 if d == 2 else 2
    clamped = np.nonzero(at[:, clamp_axis] == 0)[0]
    dofs = (d * clamped[:, None] + np.arange(d)).reshape(-1).astype(np.int32)
    loaded = np.nonzero(at[:, load_axis] == pts[load_axis] - 1)[0]
    f = np.zeros((nrhs, at.shape[0], d))
    pull = 0.5 * rng.standard_normal((nrhs, loaded.size, d))
    pull[..., d - 1] -= 1.0
    f[:, loaded] = pull
    f[:, clamped] = 0.0
    return types.SimpleNamespace(
        elem_type=TYPE[elem], ngauss=3 if QUADRATIC[elem] else 2, conn=conn, coords=coords,
        E=E0, nu=NU, elem_E=moduli, fixed_dofs=dofs, f=f.reshape(nrhs, -1),
        ndof=at.shape[0] * d, elem=elem)


def _plates(case, seed):
    sizes = np.random.default_rng(case["sizes"]).integers(case["lo"], case["hi"] + 1,
                                                          case["count"])
    out = []
    for k, nx in enumerate(int(v) for v in sizes):
        p = _problem("q4", nx, max(2, nx // 2), 0, 0.0, 1, 1000 * seed + k)
        p.f = p.f[0]
        out.append(p)
    return out


def _net_inputs(case, seed):
    """He-scaled weights, bf16 features (smooth fields, mask, coordinates) and
    fp32 targets of a batch, channels last."""
    rng = np.random.default_rng(seed)
    z, y, x, b = case["gz"], case["gy"], case["gx"], case["batch"]
    params = []
    for _, cin, cout, _, _ in NET:
        params += [rng.standard_normal(27 * cin * cout) * math.sqrt(2.0 / (27 * cin)),
                   0.01 * rng.standard_normal(cout)]
    params = np.concatenate(params).astype(np.float32)
    gz, gy, gx = np.meshgrid(np.linspace(0, 1, z), np.linspace(0, 1, y), np.linspace(0, 1, x),
                             indexing="ij")
    feats = np.zeros((b, z, y, x, 16))
    target = np.zeros((b, z, y, x, 4), dtype=np.float32)
    for s in range(b):
        a = rng.standard_normal((14, 4))
        for c in range(14):
            feats[s, ..., c] = (a[c, 0] * gx + a[c, 1] * np.sin(3 * gy + a[c, 2])
                                + a[c, 3] * gz * gx)
        feats[s, ..., 0] += 0.3 * rng.standard_normal((z, y, x))
        feats[s, ..., 4] = gx == 0
        feats[s, ..., 5], feats[s, ..., 6], feats[s, ..., 7] = gx, gy, gz
        for c in range(3):
            target[s, ..., c] = a[c, 0] * gx ** 2 + 0.3 * a[c, 1] * gx * gy + 0.1 * a[c, 2] * gz
    return params, torch.from_numpy(feats).to(torch.bfloat16), torch.from_numpy(target)


# ---- passes -----------------------------------------------------------------
_CTX = []


def _context():
    if not _CTX:
        _CTX.append(gf.Context(0))
    return _CTX[0]


def _solve(ctx, ell, b, x, nrhs, opts):
    stats = gf._lib.SolveStats()
    code = ctx.lib.gf_pcg(ctx.handle, ell.handle, C.c_void_p(b.data_ptr()),
                          C.c_void_p(x.data_ptr()), nrhs, C.byref(opts), C.byref(stats))
    gf.check(code, ctx.handle)


def prepare(case, seed):
    s = types.SimpleNamespace(kind=case["kind"], ctx=_context())
    kind, ctx = s.kind, s.ctx
    if kind == "train":
        params, feats, target = _net_inputs(case, seed)
        s.net = gf.Net(ctx, case["gx"], case["gy"], case["gz"], case["batch"])
        s.net.set_params(params)
        s.batch, s.feats, s.target = case["batch"], feats.cuda(), target.cuda()
        return s
    if kind == "group":
        s.problems = _plates(case, seed)
        s.group = ctx.group(s.problems)
        s.moduli = [p.elem_E for p in s.problems]
        s.b = np.concatenate([p.f for p in s.problems])
        s.rtol = case["rtol"]
        s.group.assemble()
        return s
    nrhs = case.get("nrhs", 1)
    p = _problem(case["elem"], case["nx"], case["ny"], case["nz"], case["jitter"], nrhs, seed)
    s.p = p
    if kind == "oneshot":
        s.rtol, s.b = case["rtol"], np.ascontiguousarray(p.f[0])
        return s
    s.mesh = ctx.upload_mesh(p.elem_type, p.ngauss, p.conn, p.coords, p.E, p.nu, elem_E=p.elem_E)
    s.ell = ctx.symbolic(s.mesh, device=True)
    ctx.assemble(s.mesh, s.ell)
    ctx.apply_penalty(s.ell, p.fixed_dofs)
    ctx.tune(s.ell)
    if kind == "force":
        s.u = np.random.default_rng(seed + 7).standard_normal(p.ndof)
        return s
    s.nrhs = nrhs
    s.opts = gf.solve_opts(device_ptrs=1, rtol=case["rtol"],
                           precision=gf.GF_PREC_MIXED if case["mixed"] else gf.GF_PREC_FP64)
    s.b = torch.from_numpy(p.f).cuda()
    s.x = torch.zeros_like(s.b)
    torch.cuda.synchronize()
    return s


def run(s):
    ctx = s.ctx
    if s.kind == "train":
        loss = s.net.backward(C.c_void_p(s.feats.data_ptr()), C.c_void_p(s.target.data_ptr()),
                              s.batch)
        return {"loss": np.float32(loss), "grads": s.net.grads()}
    if s.kind == "group":
        s.group.set_E(s.moduli)
        s.group.assemble()
        s.group.apply_penalty()
        return s.group.pcg(s.b, rtol=s.rtol)[0]
    p = s.p
    if s.kind == "oneshot":
        mesh = ctx.upload_mesh(p.elem_type, p.ngauss, p.conn, p.coords, p.E, p.nu,
                               elem_E=p.elem_E)
        ell = ctx.symbolic(mesh, device=True)
        ctx.assemble(mesh, ell)
        ctx.apply_penalty(ell, p.fixed_dofs)
        x, _ = ctx.pcg(ell, s.b, rtol=s.rtol)
        ell.free()
        mesh.free()
        return x
    if s.kind == "force":
        s.mesh.set_E(p.elem_E)
        ctx.assemble(s.mesh, s.ell)
        ctx.apply_penalty(s.ell, p.fixed_dofs)
        return ctx.spmv(s.ell, s.u)[0]
    ctx.assemble(s.mesh, s.ell)
    ctx.apply_penalty(s.ell, p.fixed_dofs)
    _solve(ctx, s.ell, s.b, s.x, s.nrhs, s.opts)
    return s.x


# ---- what a pass cannot do without ---------------------------------------------
def _counts(elem, nx, ny, nz):
    d, quad = DIM[elem], QUADRATIC[elem]
    nel = (nx, ny, nz)[:d]
    elements = math.prod(nel)
    nodes = math.prod(k + 1 for k in nel)
    if quad:
        nodes += sum(k * math.prod(j + 1 for i, j in enumerate(nel) if i != a)
                     for a, k in enumerate(nel))
    return elements, nodes, NEIGHBOURS[elem] * nodes * d * d


def _assembly_work(elem, elements, nodes, nnz):
    """Connectivity, coordinates and moduli read once, the upper half of the
    symmetric values written once; the products T_pq of the node pairs."""
    d, nen = DIM[elem], len(NATURAL[elem])
    ngp = (3 if QUADRATIC[elem] else 2) ** d
    return (4.0 * elements * nen + 8.0 * elements + 8.0 * d * nodes + 4.0 * nnz,
            float(elements) * ngp * nen * (nen + 1) * d * d)


def _solve_work(elem, longest, n, nnz, nrhs, mixed, rtol):
    """Per iteration the upper half of the matrix read once, each direction
    read and each product written once; the iteration count is an estimate."""
    its = ITERATIONS[elem] * longest * (1.0 + 0.12 * max(0.0, -math.log10(rtol) - 8.0))
    size = 4.0 if mixed else 8.0
    return (its * (0.5 * size * nnz + 2.0 * size * n * nrhs),
            its * nrhs * (2.0 * nnz + 10.0 * n))


def work(case):
    kind = case["kind"]
    if kind == "train":
        vox = [case["batch"] * math.prod((g - 1) // 2 ** l + 1
                                         for g in (case["gx"], case["gy"], case["gz"]))
               for l in range(4)]
        # forward, data gradient and weight gradient of every convolution
        flops = sum(6.0 * 27 * cin * cout * vox[level] for _, cin, cout, _, level in NET)
        return {"bytes": vox[0] * (32.0 + 16.0) + 8.0 * sum(27 * c * k + k
                                                              for _, c, k, _, _ in NET),
                "flops": flops}
    if kind == "group":
        by = fl = 0.0
        sizes = np.random.default_rng(case["sizes"]).integers(case["lo"], case["hi"] + 1,
                                                              case["count"])
        for nx in (int(v) for v in sizes):
            ne, nn, nnz = _counts("q4", nx, max(2, nx // 2), 0)
            a, s = (_assembly_work("q4", ne, nn, nnz),
                    _solve_work("q4", nx, 2 * nn, nnz, 1, 0, case["rtol"]))
            by, fl = by + a[0] + s[0], fl + a[1] + s[1]
        return {"bytes": by, "flops": fl}
    elem = case["elem"]
    ne, nn, nnz = _counts(elem, case["nx"], case["ny"], case["nz"])
    n = nn * DIM[elem]
    by, fl = _assembly_work(elem, ne, nn, nnz)
    if kind == "force":
        return {"bytes": by + 4.0 * nnz + 16.0 * n, "flops": fl + 2.0 * nnz}
    s = _solve_work(elem, max(case["nx"], case["ny"], case["nz"]), n, nnz, case.get("nrhs", 1),
                    case.get("mixed", 0), case["rtol"])
    return {"bytes": by + s[0], "flops": fl + s[1]}


# ---- the same in 64 bits, without the framework ----------------------------------
def _shape_derivs(elem, x):
    """dN_a/dxi_i [nen, d] at the natural point x (multilinear or serendipity)."""
    d, out = DIM[elem], []
    for nat in NATURAL[elem]:
        lin = [1.0 + x[i] * nat[i] for i in range(d)]
        mid = [i for i in range(d) if nat[i] == 0]
        row = []
        for k in range(d):
            others = [lin[i] for i in range(d) if i != k and nat[i] != 0]
            if not QUADRATIC[elem]:
                v = nat[k] * math.prod(others) / 2 ** d
            elif not mid:
                v = (nat[k] * math.prod(others) * (sum(x[i] * nat[i] for i in range(d))
                                                   + x[k] * nat[k] - (d - 2)) / 2 ** d)
            elif k == mid[0]:
                v = -2.0 * x[k] * math.prod(others) / 2 ** (d - 1)
            else:
                v = (1.0 - x[mid[0]] ** 2) * nat[k] * math.prod(others) / 2 ** (d - 1)
            row.append(v)
        out.append(row)
    return out


def _element_matrices(p, dev, lo, hi):
    """Ke of elements lo..hi: [elements, nen, d, nen, d], and their DOFs."""
    elem, d = p.elem, DIM[p.elem]
    conn = torch.from_numpy(p.conn[lo:hi].astype(np.int64) - 1).to(dev)
    xe = torch.from_numpy(p.coords).to(dev)[conn]
    mod = torch.from_numpy(p.elem_E[lo:hi]).to(dev)
    mu = mod / (2 * (1 + NU))
    lam = mod * NU / (1 - NU ** 2) if d == 2 else mod * NU / ((1 + NU) * (1 - 2 * NU))
    if p.ngauss == 2:
        rule = [(-1 / math.sqrt(3), 1.0), (1 / math.sqrt(3), 1.0)]
    else:
        rule = [(-math.sqrt(0.6), 5 / 9), (0.0, 8 / 9), (math.sqrt(0.6), 5 / 9)]
    nen = conn.shape[1]
    ke = torch.zeros(conn.shape[0], nen, d, nen, d, dtype=torch.float64, device=dev)
    for g in np.ndindex(*([len(rule)] * d)):
        dn = torch.tensor(_shape_derivs(elem, [rule[i][0] for i in g]), dtype=torch.float64,
                          device=dev)
        jac = torch.stack([(xe * dn[:, k, None]).sum(1) for k in range(d)], dim=1)
        w = torch.linalg.det(jac) * math.prod(rule[i][1] for i in g)
        inv = torch.linalg.inv(jac)
        gr = sum(dn[None, :, None, k] * inv[:, None, :, k] for k in range(d))  # [e, a, i]
        outer = gr[:, :, :, None, None] * gr[:, None, None, :, :]  # G_ai G_bj
        ke += (lam * w)[:, None, None, None, None] * outer
        ke += (mu * w)[:, None, None, None, None] * outer.transpose(2, 4)
        tr = (mu * w)[:, None, None] * torch.diagonal(outer, dim1=2, dim2=4).sum(-1)
        for i in range(d):
            ke[:, :, i, :, i] += tr
    dofs = (conn[:, :, None] * d + torch.arange(d, device=dev)).reshape(conn.shape[0], -1)
    return ke.reshape(conn.shape[0], nen * d, nen * d), dofs


def _chunks(p):
    step = max(1, 40_000_000 // (p.conn.shape[1] * DIM[p.elem]) ** 2)
    return [(lo, min(p.conn.shape[0], lo + step)) for lo in range(0, p.conn.shape[0], step)]


def _penalised(p, diag, dev):
    """The factors of the diagonal: 1, and 1e4 max K_ii on the supports."""
    f = torch.ones_like(diag)
    f[torch.from_numpy(p.fixed_dofs.astype(np.int64)).to(dev)] = 1e4 * float(diag.max())
    return f


def _forces(p, u, dev):
    u = torch.from_numpy(u).to(dev)
    y, diag = torch.zeros_like(u), torch.zeros_like(u)
    for lo, hi in _chunks(p):
        ke, dofs = _element_matrices(p, dev, lo, hi)
        y.index_add_(0, dofs.reshape(-1), (ke * u[dofs][:, None, :]).sum(-1).reshape(-1))
        diag.index_add_(0, dofs.reshape(-1), torch.diagonal(ke, dim1=1, dim2=2).reshape(-1))
    return y + (_penalised(p, diag, dev) - 1.0) * diag * u


def _matrix(p, dev):
    """The penalised matrix as CSR (node blocks summed by sorting) and its diagonal."""
    n = p.ndof
    keys, vals = [], []
    for lo, hi in _chunks(p):
        ke, dofs = _element_matrices(p, dev, lo, hi)
        key, at = torch.unique((dofs[:, :, None] * n + dofs[:, None, :]).reshape(-1),
                               return_inverse=True)
        keys.append(key)
        vals.append(torch.zeros(key.numel(), dtype=torch.float64, device=dev).index_add_(
            0, at, ke.reshape(-1)))
    key, at = torch.unique(torch.cat(keys), return_inverse=True)
    val = torch.zeros(key.numel(), dtype=torch.float64, device=dev).index_add_(
        0, at, torch.cat(vals))
    rows, cols = key // n, key % n
    on = rows == cols
    diag = val[on]
    diag = diag * _penalised(p, diag, dev)
    val[on] = diag
    crow = torch.zeros(n + 1, dtype=torch.int64, device=dev)
    crow[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    return torch.sparse_csr_tensor(crow.to(torch.int32), cols.to(torch.int32), val,
                                   size=(n, n)), diag


def _pcg(mat, diag, b):
    """Jacobi-PCG on the columns of b, restarted from the true residual until
    it falls no more."""
    x = torch.zeros_like(b)
    r = b.clone()
    best, bn = None, b.norm(dim=0)
    for _ in range(5):
        z = r / diag[:, None]
        q = z.clone()
        rz = (r * z).sum(0)
        goal, it = 1e-7 * r.norm(dim=0).clamp_min(1e-8 * bn), 0
        if best is None:
            goal = 1e-12 * bn
        corr = torch.zeros_like(b)
        while it < 60000:
            aq = mat @ q
            alpha = rz / (q * aq).sum(0).clamp_min(1e-300)
            corr += alpha * q
            r = r - alpha * aq
            z = r / diag[:, None]
            new = (r * z).sum(0)
            q = z + (new / rz.clamp_min(1e-300)) * q
            rz = new
            it += 1
            if it % 64 == 0 and bool((r.norm(dim=0) <= goal).all()):
                break
        x = x + corr
        r = b - mat @ x
        rel = float((r.norm(dim=0) / bn).max())
        if best is not None and rel > 0.3 * best:
            break
        best = rel
        if rel < 1e-13:
            break
    return x


# the network's convolutions: name, input channels, output channels, stride,
# level of the output grid
NET = [("e0a", 16, 16, 1, 0), ("e0b", 16, 16, 1, 0), ("e1a", 16, 32, 2, 1), ("e1b", 32, 32, 1, 1),
       ("e2a", 32, 64, 2, 2), ("e2b", 64, 64, 1, 2), ("e3a", 64, 128, 2, 3),
       ("d2a", 192, 64, 1, 2), ("d2b", 64, 64, 1, 2), ("d1a", 96, 32, 1, 1),
       ("d1b", 32, 32, 1, 1), ("d0a", 48, 16, 1, 0), ("d0b", 16, 16, 1, 0), ("out", 16, 16, 1, 0)]


def _conv(x, w, bias, stride, act):
    b, z, y, xx, _ = x.shape
    oz, oy, ox = [(v + stride - 1) // stride for v in (z, y, xx)]
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = bias
    for t in range(27):
        dz, dy, dx = t // 9, (t // 3) % 3, t % 3
        win = xp[:, dz:dz + stride * (oz - 1) + 1:stride, dy:dy + stride * (oy - 1) + 1:stride,
                 dx:dx + stride * (ox - 1) + 1:stride]
        out = out + win @ w[t]
    return torch.where(out > 0, out, 0.1 * out) if act else out


def _up(a):
    for ax in (1, 2, 3):
        lo, hi = a.narrow(ax, 0, a.shape[ax] - 1), a.narrow(ax, 1, a.shape[ax] - 1)
        odd = torch.cat([0.5 * (lo + hi), a.narrow(ax, 0, 1)], dim=ax)
        a = torch.stack([a, odd], dim=ax + 1).flatten(ax, ax + 1).narrow(ax, 0, 2 * a.shape[ax] - 1)
    return a


def _net_gradient(params, feats, target, dev):
    p = torch.from_numpy(params).to(dev, torch.float64).requires_grad_()
    x = feats.to(dev, torch.float64)
    w, at = {}, 0
    for name, cin, cout, stride, _ in NET:
        k = 27 * cin * cout
        w[name] = (p[at:at + k].reshape(27, cin, cout), p[at + k:at + k + cout], stride,
                   name != "out")
        at += k + cout

    def conv(a, name):
        return _conv(a, *w[name])

    s0 = conv(conv(x, "e0a"), "e0b")
    s1 = conv(conv(s0, "e1a"), "e1b")
    s2 = conv(conv(s1, "e2a"), "e2b")
    a = conv(s2, "e3a")
    a = conv(conv(torch.cat([_up(a), s2], -1), "d2a"), "d2b")
    a = conv(conv(torch.cat([_up(a), s1], -1), "d1a"), "d1b")
    a = conv(conv(conv(torch.cat([_up(a), s0], -1), "d0a"), "d0b"), "out")
    loss = ((a[..., :3] - target.to(dev, torch.float64)[..., :3]) ** 2).mean()
    loss.backward()
    return {"loss": float(loss.detach()), "grads": p.grad.cpu().numpy()}


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    kind = case["kind"]
    if kind == "train":
        out = _net_gradient(*_net_inputs(case, seed), dev)
        return {"loss": np.float64(out["loss"]), "grads": out["grads"]}
    if kind == "group":
        xs = []
        for p in _plates(case, seed):
            mat, diag = _matrix(p, dev)
            xs.append(_pcg(mat, diag, torch.from_numpy(p.f).to(dev)[:, None])[:, 0])
        return torch.cat(xs).cpu().numpy()
    nrhs = case.get("nrhs", 1)
    p = _problem(case["elem"], case["nx"], case["ny"], case["nz"], case["jitter"], nrhs, seed)
    if kind == "force":
        return _forces(p, np.random.default_rng(seed + 7).standard_normal(p.ndof),
                       dev).cpu().numpy()
    mat, diag = _matrix(p, dev)
    x = _pcg(mat, diag, torch.from_numpy(p.f).to(dev).T.contiguous())
    if kind == "oneshot":
        return x[:, 0].cpu().numpy()
    return x.T.contiguous()
