"""The automatic choice of cells per thread of plain FP64 kernels: bit for bit the fields of one
cell per thread on either side of each of its lines (rows of 160 and 256 cells, launches of 4e6
and 12e6 cells), with extents that the groups do not divide."""
import time

import numpy as np
import pytest

import parallelstencil as ps
from parallelstencil import workloads as W

pytestmark = pytest.mark.gpu

M64 = __name__ + ".f64"
ps.init_parallel_stencil(ps.AMDGPU, ps.Float64, 3, module=M64)


@pytest.mark.parametrize("shape", [(159, 161, 163), (160, 160, 156), (160, 160, 157), (161, 163, 155), (255, 127, 131),
                                   (229, 230, 231), (256, 9, 10), (259, 7, 13)])
def test_automatic_cells_match_one_cell(shape):
    rng = np.random.default_rng(sum(shape))
    auto, one = W.define_diffusion3d(False, M64), W.define_diffusion3d(False, M64, cells_x=1, cells_z=1)
    T, Ci = ps.zeros(*shape), ps.zeros(*shape)
    T.copy_from(np.asfortranarray(rng.standard_normal(shape)))
    Ci.copy_from(np.asfortranarray(1.0 + rng.random(shape)))
    a, b = ps.zeros(*shape), ps.zeros(*shape)
    for k, T2 in ((auto, a), (one, b)):
        T2.copy_from(T.to_host())
        k(T2, T, Ci, 1.3, 1e-3, 0.1, 0.2, 0.3)
    assert np.array_equal(a.to_host().view(np.uint64), b.to_host().view(np.uint64)), shape
    nx, ny, nz = (n - 1 for n in shape)  # staggered arrays: the launch box is the largest of them
    F = [(rng.standard_normal(s)) for s in ((nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1), (nx, ny, nz))]
    out = []
    for kw in ({}, dict(cells_x=1, cells_z=1)):
        V, P = W.define_acoustic3d(M64, **kw)
        D = [ps.zeros(*f.shape) for f in F]
        for d, f in zip(D, F):
            d.copy_from(np.asfortranarray(f))
        V(*D, 1e-2, 1.1, 0.1, 0.2, 0.3)
        P(D[3], D[0], D[1], D[2], 1e-2, 1.2, 0.1, 0.2, 0.3)
        out.append([np.ascontiguousarray(d.to_host()).view(np.uint64) for d in D])
    for x, y in zip(*out):
        assert np.array_equal(x, y), shape


WRITES = """
@parallel_indices (ix, iy, iz) function writes!(A, B, C, s::Data.Number)
    if ix >= 2 && ix <= size(A, 1) - 1 && iz >= 2 && iz <= size(A, 3) - 1
        A[ix, iy, iz] = 0.0
        B[ix, iy, iz] = s * 0.5 + ix
    end
    C[ix, iy, iz] = s
    return
end
"""
READS = WRITES.replace("C[ix, iy, iz] = s\n", "C[ix, iy, iz] += s\n")


@pytest.mark.parametrize("src", [WRITES, READS])
@pytest.mark.parametrize("shape", [(2, 3, 8), (7, 5, 9), (64, 33, 10), (130, 17, 7), (259, 20, 31)])
def test_kernels_without_reads_match_one_cell(src, shape):
    # four z cells per thread where nothing is read; sizes that neither 4 z cells nor the block divide
    out = []
    for kw in ({}, dict(cells_x=1, cells_z=1)):
        k = ps.core._define("parallel_indices", src, kw, M64)
        D = [ps.fill(0.25 * i, *shape) for i in range(3)]
        for _ in range(2):
            k(*D, 1.75)
        out.append([np.ascontiguousarray(d.to_host()).view(np.uint64) for d in D])
    for x, y in zip(*out):
        assert np.array_equal(x, y), shape


@pytest.mark.parametrize("shape", [(160, 161, 157), (200, 170, 121), (257, 40, 33)])
def test_quotients_by_values_match_one_cell(shape):
    # several quotients by array values per cell: one cell per thread in rows below 256, z cells from there on
    nx, ny, nz = shape
    out = []
    for kw in ({}, dict(cells_x=1, cells_z=1)):
        k = ps.core._define("parallel", W.STOKES3D_TIMESTEPS, kw, M64)
        D = [ps.zeros(*s) for s in ((nx - 1, ny - 2, nz - 2), (nx - 2, ny - 1, nz - 2), (nx - 2, ny - 2, nz - 1), shape)]
        Mus = ps.zeros(*shape).copy_from(np.asfortranarray(1.0 + np.random.default_rng(nx).random(shape)))
        k(*D, Mus, 1.0, 0.25, 1e-3, max(shape))
        out.append([np.ascontiguousarray(d.to_host()).view(np.uint64) for d in D])
    for x, y in zip(*out):
        assert np.array_equal(x, y), shape


def test_a_kernel_compiled_ahead_is_not_emitted_again():
    """The first launch after precompile_launch only loads the code object: emitting the grouped source again
    is more than half of what a first launch without it takes (810 us, 310 after precompile_launch)."""
    A = [ps.zeros(253, 190, 127) for _ in range(3)]
    args = (*A, 1.0, 0.1, 0.1, 0.1, 0.1)

    def first(ahead):
        k = W.define_diffusion3d(False, M64)
        if ahead:
            k.precompile_launch(*args)
        t = time.perf_counter()
        k(*args)
        return time.perf_counter() - t

    first(True)  # compiles into the cache of code objects
    assert min(first(True) for _ in range(7)) < 0.7 * min(first(False) for _ in range(7))
