"""The host code of libgpufem over a stand-in for the HIP runtime
(tests/cpp/fake_hip.cpp), no GPU: what it does when an allocation fails and
which kernels it picks.  Each case runs in a process of its own, where the
stand-in is loaded before the library."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, sys
fake = C.CDLL(%r, mode=C.RTLD_GLOBAL)
fake.fake_fail_at.argtypes = [C.c_int64]
fake.fake_memory.argtypes = [C.c_int64, C.c_int64]
fake.fake_cost.argtypes = [C.c_char_p, C.c_double]
fake.fake_log.restype = C.c_char_p
for f in ("live", "live_bytes", "mallocs", "h2d", "last_bytes"):
    getattr(fake, "fake_" + f).restype = C.c_int64
sys.path.insert(0, %r)
import numpy as np
import gpufem_amd as gf
from gpufem_amd import problems as P
ctx = gf.Context(0)

def kernels():
    return [k for k in fake.fake_log().decode().split("\\n") if k]

def launched(name):
    return any(name in k for k in kernels())

def mesh_of(p):
    return ctx.upload_mesh(p.elem_type, p.ngauss, p.conn, p.coords, p.E, p.nu)
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-fPIC", "-shared",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "cpp", "fake_hip.cpp"), "-o", so], check=True)

    def go(body):
        out = subprocess.run([sys.executable, "-c", PRELUDE % (so, ROOT) + body],
                             capture_output=True, text=True, timeout=300)
        assert out.returncode == 0, out.stdout + out.stderr
    return go


def test_a_reported_failure_is_not_reported_again(run):
    """An allocation that failed is the error of its own call only."""
    run("""
p = P.structured(gf.GF_Q4, 9, 5)
mesh = mesh_of(p)
fake.fake_fail_at(0)
try:
    mesh_of(p)
    assert False, "the upload was to fail"
except gf.GpufemError:
    pass
ctx.symbolic(mesh)
""")


def test_group_solve_after_a_failed_allocation(run):
    """Whatever allocation of the first grouped solve fails, the next solve
    builds everything it needs, and the group gives back all it took."""
    run("""
probs = [P.structured(gf.GF_Q4, 9, 5), P.structured(gf.GF_Q4, 20, 9)]
fake.fake_stop(b"k_gs_product")     # the iteration itself does not run here

def solve(fail):
    before = fake.fake_live()
    G = ctx.group(probs)
    G.assemble()
    G.apply_penalty()
    start = fake.fake_mallocs()
    if fail is not None:
        fake.fake_fail_at(fail)
        st = G.pcg(schedule=gf.GF_SCHED_KERNELS, raise_on_fail=False)[1]
        fake.fake_fail_at(-1)
        assert st.code in (-2, -3) and not launched("k_gs_product"), st.code
    st = G.pcg(schedule=gf.GF_SCHED_KERNELS, raise_on_fail=False)[1]
    assert launched("k_gs_product")
    fake.fake_clear_log()
    held, taken = fake.fake_live(), fake.fake_mallocs() - start
    G.free()
    assert fake.fake_live() == before
    return held - before, taken

held, taken = solve(None)
assert taken > 20
for k in range(taken):
    assert solve(k)[0] == held, k
""")


def test_first_assembly_of_a_small_mesh_needs_no_memory(run):
    """The kernel of a small mesh is picked without timing; where its arrays
    cannot be allocated the assembly runs all the same, then and later."""
    run("""
for p in (P.structured(gf.GF_BRICK8, 3, 2, 2), P.structured(gf.GF_BRICK20, 3, 2, 2)):
    mesh = mesh_of(p)
    k = 0
    while True:
        K = ctx.symbolic(mesh)
        start = fake.fake_mallocs()
        fake.fake_fail_at(k)
        ctx.assemble(mesh, K)
        fake.fake_fail_at(-1)
        taken = fake.fake_mallocs() - start
        ctx.assemble(mesh, K)
        if k >= taken:
            break
        k += 1
    assert k > 0
""")


def test_small_mesh_assembly_leaves_room_for_the_solve(run):
    """With room for the scatter's assembly and a batched solve, and little
    more, the untimed assembly leaves enough for that solve."""
    run("""
p = P.structured(gf.GF_BRICK20, 10, 10, 10)
F = np.zeros((64, p.ndof))
fake.fake_stop(b"k_mm_spmm_pq")     # the first kernel of an iteration
mesh = mesh_of(p)

def solve(force):
    K = ctx.symbolic(mesh)
    start = fake.fake_live_bytes()
    if force is not None:
        ctx.assemble_tune(mesh, K, force)
    ctx.assemble(mesh, K)
    fake.fake_clear_log()
    x, st = ctx.pcg(K, F, precision=gf.GF_PREC_MIXED, schedule=gf.GF_SCHED_KERNELS,
                    raise_on_fail=False)
    reached = launched("k_mm_spmm_pq")
    K.free()
    return reached, start

held = fake.fake_live_bytes()
low, high = 1, 1 << 33              # the least memory in which it runs
while high - low > 1 << 16:
    mid = (low + high) // 2
    fake.fake_memory(held + mid, 0)
    try:
        ok = solve(0)[0]
    except gf.GpufemError:
        ok = False
    low, high = (low, mid) if ok else (mid, high)
fake.fake_memory(held + int(1.02 * high), 0)
assert solve(None)[0], "%.1f MB are too little" % (1.02e-6 * high)
""")


def test_first_assembly_copies_no_lists(run):
    """The node gather's lists are made on the device: the first assembly of a
    mesh that is already there sends nothing to it."""
    run("""
for p in (P.structured(gf.GF_BRICK8, 9, 9, 9), P.structured(gf.GF_BRICK20, 4, 4, 4)):
    mesh = mesh_of(p)
    K = ctx.symbolic(mesh)
    sent = fake.fake_h2d()
    ctx.assemble(mesh, K)
    assert launched("k_assemble_gather") and fake.fake_h2d() == sent
""")


def test_two_launch_iteration_up_to_the_cache(run):
    """The iteration a solve runs on both sides of the line between matrices
    that stay in the last-level cache and those that do not."""
    run("""
fake.fake_stop(b"_update")          # the second launch of an iteration
for t, nx, ny, two in ((gf.GF_Q4, 700, 700, True), (gf.GF_Q4, 840, 840, False),
                       (gf.GF_Q8, 540, 275, True), (gf.GF_Q8, 576, 290, False),
                       (gf.GF_BRICK8, 50, 50, True), (gf.GF_BRICK8, 51, 51, False)):
    p = P.structured(t, nx, ny, 50 if t == gf.GF_BRICK8 else 0)
    mesh = mesh_of(p)
    K = ctx.symbolic(mesh)
    ctx.assemble(mesh, K)
    fake.fake_clear_log()
    ctx.pcg(K, p.f, schedule=gf.GF_SCHED_KERNELS, raise_on_fail=False)
    assert launched("k_split_product") == two, (nx, ny)
    assert launched("k_spmv_pq") != two
""")


def test_group_takes_two_launches_where_they_are_faster(run):
    """Both borders of the grouped two-launch iteration: the bytes of an
    iteration, and the tiles of the largest mesh."""
    run("""
fake.fake_stop(b"_update")
for sizes, two in (([(600, 600)], True), ([(760, 760)], False), ([(600, 500)] * 2, True),
                   ([(500, 450)] * 3, False), ([(760, 760), (5, 5)], False),
                   ([(120, 60)] * 16, True)):
    G = ctx.group([P.structured(gf.GF_Q4, *s) for s in sizes])
    G.assemble()
    fake.fake_clear_log()
    G.pcg(schedule=gf.GF_SCHED_KERNELS, raise_on_fail=False)
    assert launched("k_gs_product") == two, sizes
    assert launched("k_g_spmv_pq_bs") != two
""")


def test_tuner_reports_products_and_compares_iterations(run):
    """ms_per_variant is the product alone, and the two-launch iteration is
    taken when its whole iteration is the faster one; its entry says by how
    much.  The least entry is the variant taken."""
    run("""
def tuned(p, **us):
    for name, t in us.items():
        fake.fake_cost(name.encode(), t)
    mesh = mesh_of(p)
    K = ctx.symbolic(mesh)
    ctx.assemble(mesh, K)
    chosen, ms = ctx.tune(K)
    assert ms[chosen] == ms[ms > 0].min()
    return chosen, ms

p = P.structured(gf.GF_Q8, 60, 25)
three = dict(k_spmv_pq=6.0, k_direction=3.0, k_update=1.0)
for update, want in ((20.0, 21.0), (2.0, 3.0)):      # 6 + (5 + update) - (6 + 3 + 1)
    chosen, ms = tuned(p, k_split_product=5.0, k_split_update=update, **three)
    assert (chosen == 9) == (want < 6.0), (chosen, ms)
    # 16 products and one launch that readies the state
    assert abs(ms[0] - 6.0e-3) < 1e-4 and abs(ms[9] - 1e-3 * want) < 2e-4, ms
# one workgroup: eight iterations a launch
chosen, ms = tuned(P.structured(gf.GF_Q4, 20, 10), k_single=8 * 7.0)
assert chosen == 9 and abs(ms[9] - 3.0e-3) < 2e-4, ms
""")


def test_convolution_fragments_take_one_direction(run):
    """A weight buffer holds the fragments of one direction: pairs of
    16-channel slabs of the 27 taps, 512 values each per output tile."""
    run("""
dims = np.array([9, 9, 9], dtype=np.int32)
buf = gf.DevBuf(ctx, 9 ** 3 * 256 * 4)
for cin, cout in ((16, 16), (16, 64), (192, 64), (128, 16)):
    ctx._check(ctx.lib.gf_nn_conv3d(ctx.handle, buf.ptr, 1, gf._ptr(dims), cin, buf.ptr, None, cout,
                                    1, 0, 0, 0.0, gf._ptr(dims), buf.ptr, None, 0))
    one = [-(-27 * (a // 16) // 2) * (b // 16) * 512 for a, b in ((cin, cout), (cout, cin))]
    assert fake.fake_last_bytes() == 2 * max(one), (cin, cout)
""")


def test_gpu_tests_run_the_iterations_they_name(run):
    """The sizes the GPU tests use for each kind of iteration lead to it, under
    the kernel and the persistent schedule."""
    run("""
import os
sys.path.insert(0, os.path.join(%r, "tests"))
import test_gpu_dispatch as T

def names(K, p, sched, stop):
    fake.fake_stop(stop)
    fake.fake_clear_log()
    ctx.pcg(K, p.f, schedule=sched, raise_on_fail=False)
    fake.fake_stop(b"")
    return {n for n in ("k_single", "k_split_product", "k_spmv_pq", "k_split_persistent",
                        "k_pcg_persistent") if launched(n)}

for cases, kernel, stop, persistent in (
        (T.ONE_WORKGROUP + [(gf.GF_Q4, 1535, 1, 0)], "k_single", b"k_single", "k_single"),
        (T.TWO_LAUNCHES + [(gf.GF_Q4, 1567, 1, 0), (gf.GF_BRICK8, 24, 24, 24)],
         "k_split_product", b"_update", "k_split_persistent"),
        (T.THREE_LAUNCHES, "k_spmv_pq", b"_update", "k_pcg_persistent")):
    for t, nx, ny, nz in cases:
        p = P.structured(t, nx, ny, nz)
        mesh = mesh_of(p)
        K = ctx.symbolic(mesh)
        ctx.assemble(mesh, K)
        if kernel == "k_spmv_pq":
            ctx.tune(K, 9 if nz == 0 else 10)
        assert names(K, p, gf.GF_SCHED_KERNELS, stop) == {kernel}, (nx, ny, nz)
        assert names(K, p, gf.GF_SCHED_PERSISTENT, persistent.encode()) == {persistent}, (nx, ny, nz)
""" % ROOT)
