"""The rules that pick a kernel by size and type, each against the oracle at
the edges of its range."""
import numpy as np
import pytest

import gpufem_amd as gf
import oracle as O

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
