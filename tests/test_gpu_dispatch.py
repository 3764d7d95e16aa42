"""The rules that pick a kernel by size and type, each against the oracle at
the edges of its range."""
import numpy as np
import pytest

import gpufem_amd as gf
import oracle as O
from gpufem_amd import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,nx,ny,nz,want", [
    (gf.GF_Q4, 1, 1, 0, 0), (gf.GF_Q8, 7, 3, 0, 0),
    (gf.GF_BRICK8, 1, 1, 1, 3), (gf.GF_BRICK8, 5, 4, 3, 3),
    (gf.GF_BRICK20, 1, 1, 1, 2), (gf.GF_BRICK20, 3, 4, 2, 2),
])
def test_untimed_assembly_kernel(gpu_ctx, t, nx, ny, nz, want):
    """Small meshes: the first assembly takes the rule's kernel (bitwise the
    forced one) and agrees with the oracle to 1e-12 of the largest value."""
    g = gf.Grid(t, nx, ny, nz)
    conn, coords = g.fill()
    coords = coords + 0.05 * np.random.default_rng(3).uniform(-1, 1, coords.shape)
    ng = 3 if t in (gf.GF_Q8, gf.GF_BRICK20) else 2
    mesh = gpu_ctx.upload_mesh(t, ng, conn, coords, 210000.0, 0.3)
    K, F = gpu_ctx.symbolic(mesh), gpu_ctx.symbolic(mesh)
    gpu_ctx.assemble(mesh, K)
    gpu_ctx.assemble_tune(mesh, F, want)
    gpu_ctx.assemble(mesh, F)
    val = gpu_ctx.download(K)[0]
    assert np.array_equal(val, gpu_ctx.download(F)[0])
    Ko, _ = O.assemble(g.dim, ng, conn, coords, 210000.0, 0.3, skip_zero=False)
    ov = Ko.export(Ko.max_rownnz())[0]
    assert np.abs(val - ov).max() <= 1e-12 * np.abs(ov).max()


def assembled(ctx, t, nx, ny, nz):
    p = P.structured(t, nx, ny, nz)
    mesh = ctx.upload_mesh(p.elem_type, p.ngauss, p.conn, p.coords, p.E, p.nu)
    K = ctx.symbolic(mesh)
    ctx.assemble(mesh, K)
    ctx.apply_penalty(K, p.fixed_dofs)
    return p, K


# what a solve whose caller chose no variant runs, by size: the iterations of a
# small system in one workgroup, two launches an iteration, or three where the
# matrix does not stay in the last-level cache (test_host_paths.py checks which)
ONE_WORKGROUP = [
    (gf.GF_Q4, 1, 1, 0), (gf.GF_Q4, 7, 7, 0), (gf.GF_Q4, 15, 7, 0),      # 1, 1 and 2 slices
    (gf.GF_Q4, 20, 2, 0), (gf.GF_Q4, 47, 38, 0), (gf.GF_Q4, 63, 41, 0),
    (gf.GF_Q4, 63, 42, 0),                                               # 0.744 of 0.750 MB
    (gf.GF_Q8, 21, 13, 0), (gf.GF_Q8, 33, 9, 0), (gf.GF_BRICK8, 1, 1, 1), (gf.GF_BRICK8, 7, 7, 7),
    (gf.GF_BRICK20, 2, 1, 1), (gf.GF_BRICK20, 4, 4, 3)]                  # 1.17 of 1.25 MB
TWO_LAUNCHES = [
    (gf.GF_Q4, 63, 43, 0),                                               # the first past it
    (gf.GF_Q4, 80, 50, 0), (gf.GF_Q8, 40, 30, 0), (gf.GF_Q8, 60, 25, 0),
    (gf.GF_BRICK8, 15, 7, 7), (gf.GF_BRICK8, 12, 12, 12), (gf.GF_BRICK20, 5, 4, 3),
    (gf.GF_Q4, 520, 519, 0)]                                             # two sweeps
THREE_LAUNCHES = [(gf.GF_Q4, 850, 850, 0), (gf.GF_BRICK8, 52, 51, 51)]


@pytest.mark.parametrize("t,nx,ny,nz", TWO_LAUNCHES)
def test_two_launch_iteration(gpu_ctx, t, nx, ny, nz):
    """A solve whose caller chose no variant takes the split kernels; its
    answer is the thread-per-row solve's at the same tolerance, preconditioned
    and not, and its schedules agree bitwise."""
    p, K = assembled(gpu_ctx, t, nx, ny, nz)
    _, R = assembled(gpu_ctx, t, nx, ny, nz)
    gpu_ctx.tune(R, 0)
    big = p.ndof > 100000
    for kw in ([dict()] if big else [dict(), dict(precond=gf.GF_PRECOND_NONE, verify=0)]):
        plain = "precond" in kw
        # without a preconditioner the penalty rows keep plain CG from
        # converging: a fixed number of iterations is compared instead
        opts = dict(kw, rtol=1e-4 if big else (0.0 if plain else 1e-10), raise_on_fail=not plain)
        if plain:
            opts.update(maxit=3)
        x, s = gpu_ctx.pcg(K, p.f, **opts)
        xr, sr = gpu_ctx.pcg(R, p.f, **opts)
        assert abs(s.iterations - sr.iterations) <= 2 + sr.iterations // 100
        # the same iterates to rounding; near the tolerance, to it times the
        # condition of these meshes (below 1e6 for the converged ones)
        assert np.linalg.norm(x - xr) <= (1e-4 if big else 1e-9) * np.linalg.norm(xr)
        if not big:
            for sched in (gf.GF_SCHED_KERNELS, gf.GF_SCHED_PERSISTENT):
                xs, ss = gpu_ctx.pcg(K, p.f, schedule=sched, **opts)
                assert ss.iterations == s.iterations and np.array_equal(xs, x)


@pytest.mark.parametrize("t,nx,ny,nz", [(gf.GF_Q4, 9, 5, 0),                # one workgroup
                                        (gf.GF_Q4, 80, 50, 0), (gf.GF_BRICK8, 12, 12, 12)])
def test_breakdown_at_the_start(gpu_ctx, t, nx, ny, nz):
    """A negative definite matrix breaks down at the first iteration and zero
    right-hand sides stop at none, on every schedule."""
    g = gf.Grid(t, nx, ny, nz)
    conn, coords = g.fill()
    mesh = gpu_ctx.upload_mesh(t, 2, conn, coords, -1.0, 0.3)
    K = gpu_ctx.symbolic(mesh)
    gpu_ctx.assemble(mesh, K)
    f = np.random.default_rng(0).normal(size=g.ndof)
    for sched in (gf.GF_SCHED_KERNELS, gf.GF_SCHED_GRAPH, gf.GF_SCHED_PERSISTENT):
        x, s = gpu_ctx.pcg(K, f, schedule=sched, precond=gf.GF_PRECOND_NONE, raise_on_fail=False)
        assert s.code == gf.GF_ERR_BREAKDOWN and s.iterations == 0
        assert s.relres == 1.0
        x, s = gpu_ctx.pcg(K, 0.0 * f, schedule=sched)
        assert s.converged and s.iterations == 0 and not x.any()


@pytest.mark.parametrize("t,nx,ny,nz", THREE_LAUNCHES)
def test_three_launches_past_the_cache(gpu_ctx, t, nx, ny, nz):
    """The slice-group variant of a matrix that does not stay in the last-level
    cache: its schedules agree bitwise, and after 20 iterations with the
    thread-per-row variant to rounding (their products are the same bits, the
    dot products' orders differ)."""
    p = P.structured(t, nx, ny, nz)
    mesh = gpu_ctx.upload_mesh(p.elem_type, p.ngauss, p.conn, p.coords, p.E, p.nu)
    K = gpu_ctx.symbolic(mesh, device=True)
    gpu_ctx.assemble(mesh, K)
    gpu_ctx.apply_penalty(K, p.fixed_dofs)
    kw = dict(rtol=0.0, maxit=20, verify=0, raise_on_fail=False)
    gpu_ctx.tune(K, 9 if t == gf.GF_Q4 else 10)
    x, s = gpu_ctx.pcg(K, p.f, schedule=gf.GF_SCHED_KERNELS, **kw)
    assert s.iterations == 20
    for sched in (gf.GF_SCHED_GRAPH, gf.GF_SCHED_PERSISTENT):
        y, s2 = gpu_ctx.pcg(K, p.f, schedule=sched, **kw)
        assert s2.iterations == 20 and np.array_equal(x, y) and s2.relres == s.relres
    gpu_ctx.tune(K, 0)
    y, s2 = gpu_ctx.pcg(K, p.f, **kw)
    assert np.linalg.norm(x - y) <= 1e-9 * np.linalg.norm(y)


def weak_corner(t, nx, ny, nz, scale):
    """A problem whose first three elements have `scale` (negative) times the
    modulus: the matrix is indefinite, CG breaks down after a few iterations."""
    p = P.structured(t, nx, ny, nz)
    p.elem_E = np.full(p.conn.shape[0], p.E)
    p.elem_E[:3] *= scale
    p.f = np.random.default_rng(0).normal(size=p.ndof)
    return p


def weak_matrix(ctx, p):
    mesh = ctx.upload_mesh(p.elem_type, p.ngauss, p.conn, p.coords, p.E, p.nu, elem_E=p.elem_E)
    K = ctx.symbolic(mesh)
    ctx.assemble(mesh, K)
    return K


@pytest.mark.parametrize("t,nx,ny,nz,its", [
    (gf.GF_Q4, 80, 50, 0, 11), (gf.GF_Q8, 60, 25, 0, 8), (gf.GF_BRICK8, 12, 12, 12, 15)])
def test_late_breakdown_reports_its_own_residual(gpu_ctx, t, nx, ny, nz, its):
    """A breakdown between two looks of the host at the state, iteration `its`
    in 64 bits on the CPU: every schedule of the two-launch iteration reports
    that iteration and its residual, which is the thread-per-row solve's to the
    rounding of a dozen iterations."""
    p = weak_corner(t, nx, ny, nz, -0.1)
    K, R = weak_matrix(gpu_ctx, p), weak_matrix(gpu_ctx, p)
    gpu_ctx.tune(R, 0)
    kw = dict(precond=gf.GF_PRECOND_NONE, raise_on_fail=False)
    _, want = gpu_ctx.pcg(R, p.f, **kw)
    assert want.code == gf.GF_ERR_BREAKDOWN and want.iterations == its
    for sched in (gf.GF_SCHED_KERNELS, gf.GF_SCHED_GRAPH, gf.GF_SCHED_PERSISTENT):
        _, s = gpu_ctx.pcg(K, p.f, schedule=sched, **kw)
        assert s.code == gf.GF_ERR_BREAKDOWN and s.iterations == its
        assert abs(s.relres - want.relres) <= 1e-9 * want.relres


def test_group_two_launch_iteration(gpu_ctx):
    """A grouped solve whose matrix stays in the last-level cache, meshes of one
    element to several slices: each mesh as solved alone (its own stopping
    test) as nearly as the single system's own variants agree (the slender plate
    cannot reach this tolerance in FP64: they take 1733 to 2002 iterations), the
    schedules bitwise alike, a capped solve stopping at the cap."""
    for t, sizes in ((gf.GF_Q4, [(1, 1), (40, 20), (7, 7), (64, 1)]),
                     (gf.GF_BRICK8, [(3, 2, 2), (1, 1, 1), (9, 8, 7)])):
        probs = [P.structured(t, *s) for s in sizes]
        G = gpu_ctx.group(probs)
        G.assemble()
        G.apply_penalty()
        x, st, its = G.pcg(rtol=1e-10)
        xk, sk, ik = G.pcg(rtol=1e-10, schedule=gf.GF_SCHED_KERNELS)
        assert np.array_equal(x, xk) and np.array_equal(its, ik)
        for p, xs, it in zip(probs, G.split(x), its):
            q, K = assembled(gpu_ctx, t, *(list(sizes[probs.index(p)]) + [0])[:3])
            alone = []
            for v in (0, 3, 4, 9 if t == gf.GF_Q4 else 10):
                gpu_ctx.tune(K, v)
                alone.append(gpu_ctx.pcg(K, q.f, rtol=1e-10))
            xo, counts = alone[0][0], [s.iterations for _, s in alone]
            apart = max(np.linalg.norm(xv - xo) for xv, _ in alone)
            assert abs(int(it) - counts[0]) <= 2 + counts[0] // 100 + max(counts) - min(counts)
            assert np.linalg.norm(xs - xo) <= 1e-9 * np.linalg.norm(xo) + 2 * apart
        xc, sc, ic = G.pcg(rtol=1e-10, maxit=5, verify=0, raise_on_fail=False)
        assert sc.code == gf.GF_ERR_NOCONV and ic.max() == 5


def test_group_late_breakdown_reports_its_own_residual(gpu_ctx):
    """Each mesh's breakdown (a few iterations in) is
    reported with its own iteration, the group with the larger residual of
    the two, to the rounding of a few iterations."""
    probs = [weak_corner(gf.GF_Q8, 60, 25, 0, -0.5), weak_corner(gf.GF_Q8, 60, 25, 0, -0.5)]
    probs[1].f = 2.0 * probs[1].f + 1.0
    alone = []
    for p in probs:
        R = weak_matrix(gpu_ctx, p)
        gpu_ctx.tune(R, 0)
        alone.append(gpu_ctx.pcg(R, p.f, raise_on_fail=False)[1])
        assert alone[-1].code == gf.GF_ERR_BREAKDOWN and 0 < alone[-1].iterations < 16
    G = gpu_ctx.group(probs)
    G.assemble()
    for sched in (gf.GF_SCHED_KERNELS, gf.GF_SCHED_GRAPH):
        _, s, its = G.pcg(schedule=sched, raise_on_fail=False)
        assert s.code == gf.GF_ERR_BREAKDOWN
        assert [int(i) for i in its] == [a.iterations for a in alone]
        want = max(a.relres for a in alone)
        assert abs(s.relres - want) <= 1e-9 * want


@pytest.mark.parametrize("precision", [gf.GF_PREC_FP64, gf.GF_PREC_MIXED])
@pytest.mark.parametrize("t,nx,ny,nz,nrhs", [
    (gf.GF_BRICK8, 1, 1, 1, 2), (gf.GF_BRICK8, 3, 3, 3, 9),                # 8 and 64 nodes
    (gf.GF_BRICK20, 3, 2, 2, 17), (gf.GF_BRICK20, 5, 4, 3, 40),
    (gf.GF_BRICK8, 22, 22, 22, 33), (gf.GF_BRICK8, 23, 22, 22, 33)])       # 764 and 796 passes
def test_batched_rows_in_shares(gpu_ctx, t, nx, ny, nz, nrhs, precision):
    """3D load cases advance with each row's blocks in four shares below the
    border and in one above it: every column's residual, formed by the
    thread-per-row product, meets the tolerance the solve reports, and a
    second solve gives the same bits."""
    p, K = assembled(gpu_ctx, t, nx, ny, nz)
    _, R = assembled(gpu_ctx, t, nx, ny, nz)
    gpu_ctx.tune(R, 0)
    F = P.random_top_loads(p, nrhs, 5)
    X, st = gpu_ctx.pcg(K, F, precision=precision)
    assert st.converged and st.true_relres <= 1.05e-8 and st.fallbacks == 0
    for k in range(nrhs):
        assert np.linalg.norm(F[k] - gpu_ctx.spmv(R, X[k])[0]) <= 1.1e-8 * np.linalg.norm(F[k])
    Y, s2 = gpu_ctx.pcg(K, F, precision=precision)
    assert np.array_equal(X, Y) and s2.iterations == st.iterations


@pytest.mark.parametrize("t,nx,ny,nz", ONE_WORKGROUP)
@pytest.mark.parametrize("sched", [gf.GF_SCHED_KERNELS, gf.GF_SCHED_PERSISTENT])
def test_small_system_in_one_workgroup(gpu_ctx, t, nx, ny, nz, sched):
    """Systems at the edges of the single workgroup's range: the residual
    formed by the thread-per-row product meets the tolerance, with and without
    the preconditioner and an initial guess; more iterations than one launch
    takes, an iteration limit inside a launch and a finished state are the
    limits' own."""
    p, K = assembled(gpu_ctx, t, nx, ny, nz)
    _, R = assembled(gpu_ctx, t, nx, ny, nz)
    gpu_ctx.tune(R, 0)
    f = p.f
    x, st = gpu_ctx.pcg(K, f, schedule=sched)
    assert st.converged and st.true_relres <= 1.05e-8
    assert np.linalg.norm(f - gpu_ctx.spmv(R, x)[0]) <= 1.1e-8 * np.linalg.norm(f)
    y, s2 = gpu_ctx.pcg(K, f)
    assert np.array_equal(x, y) and s2.iterations == st.iterations
    _, s3 = gpu_ctx.pcg(K, f, x0=x, rtol=1.1e-8, schedule=sched)
    assert s3.iterations == 0
    _, s4 = gpu_ctx.pcg(K, f, rtol=1e-300, maxit=700, schedule=sched, verify=0, raise_on_fail=False)
    assert s4.iterations == 700 or s4.code == gf.GF_ERR_BREAKDOWN
    _, s5 = gpu_ctx.pcg(K, f, maxit=3, schedule=sched, raise_on_fail=False)
    assert s5.iterations == min(3, st.iterations)
    z, s6 = gpu_ctx.pcg(K, np.zeros_like(f), schedule=sched)
    assert s6.iterations == 0 and not z.any()


@pytest.mark.parametrize("nx", [1535, 1567])   # 48 slices, the most of one workgroup, and 49
@pytest.mark.parametrize("sched", [gf.GF_SCHED_KERNELS, gf.GF_SCHED_PERSISTENT])
def test_strip_at_the_slice_limit(gpu_ctx, nx, sched):
    """A strip one element wide, with every slice of the single workgroup in
    use and with one more: too ill-conditioned (1e13) to converge, so the
    iterates of five iterations are compared with the thread-per-row solve."""
    p, K = assembled(gpu_ctx, gf.GF_Q4, nx, 1, 0)
    _, R = assembled(gpu_ctx, gf.GF_Q4, nx, 1, 0)
    gpu_ctx.tune(R, 0)
    f = np.random.default_rng(1).normal(size=p.ndof)
    kw = dict(rtol=0.0, maxit=5, verify=0, raise_on_fail=False)
    x, s = gpu_ctx.pcg(K, f, schedule=sched, **kw)
    y, s2 = gpu_ctx.pcg(R, f, **kw)
    assert s.iterations == 5 and s2.iterations == 5
    assert np.linalg.norm(x - y) <= 1e-9 * np.linalg.norm(y)


def turned(conn, coords):
    """Every third element's numbering turned by 90 degrees about z."""
    X = coords[conn[0] - 1]
    nat = np.rint(2 * (X - X.min(0)) / np.ptp(X, axis=0) - 1).astype(int)
    at = {tuple(v): k for k, v in enumerate(nat)}
    turn = [at[(-v[1], v[0], v[2])] for v in nat]
    out = conn.copy()
    out[::3] = conn[::3][:, turn]
    return out


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("t,nx,ny,nz,variant", [
    (gf.GF_BRICK8, 1, 1, 1, 3), (gf.GF_BRICK8, 3, 5, 2, 3), (gf.GF_BRICK8, 7, 4, 4, 4),
    (gf.GF_BRICK20, 1, 1, 1, 2), (gf.GF_BRICK20, 3, 2, 4, 2), (gf.GF_BRICK20, 3, 2, 4, 4)])
def test_gather_adds_alike_and_turned_elements(gpu_ctx, t, nx, ny, nz, variant, mixed):
    """The node gathers on elements numbered alike (no two elements around a
    node share a neighbour's number) and on a mesh where some do: against the
    oracle to 1e-12 of the largest value, and the same bits twice."""
    g = gf.Grid(t, nx, ny, nz)
    conn, coords = g.fill()
    conn = np.asarray(conn).reshape(-1, 8 if t == gf.GF_BRICK8 else 20)
    if mixed:
        conn = turned(conn, coords)
    coords = coords + 0.05 * np.random.default_rng(3).uniform(-1, 1, coords.shape)
    ng = 3 if t == gf.GF_BRICK20 else 2
    mesh = gpu_ctx.upload_mesh(t, ng, conn, coords, 210000.0, 0.3)
    K = gpu_ctx.symbolic(mesh)
    gpu_ctx.assemble_tune(mesh, K, variant)
    gpu_ctx.assemble(mesh, K)
    val = gpu_ctx.download(K)[0]
    gpu_ctx.assemble(mesh, K)
    assert np.array_equal(val, gpu_ctx.download(K)[0])
    Ko, _ = O.assemble(g.dim, ng, conn, coords, 210000.0, 0.3, skip_zero=False)
    ov = Ko.export(Ko.max_rownnz())[0]
    assert np.abs(val - ov).max() <= 1e-12 * np.abs(ov).max()


def collapsed(conn, coords):
    """A corner edge of the box drawn together: the elements around it name
    one node twice."""
    X = coords
    a = np.nonzero(np.all(X == X.min(0), axis=1))[0][0]
    d = np.linalg.norm(X - X[a], axis=1)
    b = np.nonzero((d > 0) & np.all(X[:, 1:] == X[a, 1:], axis=1))[0]
    b = b[np.argmin(d[b])]
    out = np.where(conn == b + 1, a + 1, conn)
    return np.where(out > b + 1, out - 1, out), np.delete(coords, b, axis=0)


@pytest.mark.parametrize("t,nx,ny,nz,variant,form", [
    (gf.GF_BRICK8, 1, 1, 1, 3, ""), (gf.GF_BRICK8, 6, 5, 4, 3, "shuffled"),
    (gf.GF_BRICK8, 4, 3, 3, 3, "collapsed"), (gf.GF_BRICK20, 3, 4, 2, 2, "shuffled"),
    (gf.GF_Q8, 9, 7, 0, 3, "shuffled")])
def test_gather_lists_made_on_the_device(gpu_ctx, t, nx, ny, nz, variant, form):
    """The lists the node gather sums in order, after either symbolic phase
    (the device one leaves unordered lists): the same bits, and the oracle's
    values to 1e-12 of the largest."""
    g = gf.Grid(t, nx, ny, nz)
    conn, coords = g.fill()
    conn = np.asarray(conn).reshape(g.nelem, -1)
    if form == "collapsed":
        conn, coords = collapsed(conn, coords)
        assert any(len(set(c)) < conn.shape[1] for c in conn.tolist())
    rng = np.random.default_rng(4)
    conn = rng.permutation(conn) if form else conn
    coords = coords + 0.03 * rng.uniform(-1, 1, coords.shape)
    ng = 3 if t in (gf.GF_Q8, gf.GF_BRICK20) else 2
    mesh = gpu_ctx.upload_mesh(t, ng, conn, coords, 210000.0, 0.3)
    vals = []
    for device in (False, True, True):
        K = gpu_ctx.symbolic(mesh, device=device)
        gpu_ctx.assemble_tune(mesh, K, variant)
        gpu_ctx.assemble(mesh, K)
        vals.append(gpu_ctx.download(K)[0])
    assert np.array_equal(vals[0], vals[1]) and np.array_equal(vals[0], vals[2])
    Ko, _ = O.assemble(g.dim, ng, conn, coords, 210000.0, 0.3, skip_zero=False)
    ov = Ko.export(Ko.max_rownnz())[0]
    assert np.abs(vals[0] - ov).max() <= 1e-12 * np.abs(ov).max()
