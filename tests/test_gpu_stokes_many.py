"""Several PT iterations per launch (ps_stokes2d_iterate) against the same number of single iterations
through the two-launch kernels, every field bit for bit: each tile size of the rule (from one
workgroup to more workgroups than CUs), the smallest grids, tile remainders, iteration counts that do
not divide evenly over the launches, a batch with a frozen sample, and values whose quotients leave
the range of the corrected reciprocal. Plane-by-plane reductions against those of the plane views."""
import ctypes

import numpy as np
import pytest

import parallelstencil as ps
from parallelstencil import stokes_fused as F
from parallelstencil._lib import lib

pytestmark = pytest.mark.gpu
MOD = __name__
ps.init_parallel_stencil(ps.AMDGPU, ps.Float64, 2, module=MOD)
FIELDS = ("Pt", "divV", "Vx", "Vy", "txx", "tyy", "txy", "Rx", "Ry", "dVxdt", "dVydt")


def _bits(A):
    return np.ascontiguousarray(A.to_host()).view(np.uint64)


def _start(sv, seed, scale=1.0):
    rng = np.random.default_rng(seed)
    sh = sv.Pt.shape
    sv.set_material(np.asfortranarray(1.0 + 3.0 * rng.random(sh)), np.asfortranarray(rng.random(sh)))
    sv.reset(*(scale * (rng.random(A.shape) - 0.5) for A in (sv.Vx, sv.Vy, sv.Pt)))


# tiles of 8 up to 127 x 127 (16 x 16 = 256 of them), of 16 from 128 x 127 to 255 x 255, of 24 to 383 x 383, of 32 beyond
@pytest.mark.parametrize("nx,ny,n", [(8, 8, 2), (9, 31, 3), (33, 8, 16), (127, 127, 17), (128, 127, 33), (199, 257, 9), (255, 260, 8), (300, 310, 6), (383, 383, 9),
                                     (383, 100, 7), (384, 383, 5), (511, 390, 11), (70, 1100, 4)])
def test_many_iterations_match_single_ones(nx, ny, n):
    a, b = (F.Stokes2DFused(MOD, nx, ny, graph=False, eta_ts="maxV") for _ in range(2))
    for sv in (a, b):
        _start(sv, nx * ny)
    a.iterate(n)
    for _ in range(n):
        b.iterate(1)
    ps.synchronize()
    for k in FIELDS:
        assert np.array_equal(_bits(getattr(a, k)), _bits(getattr(b, k))), k


@pytest.mark.parametrize("scale", [1e-200, 1e-300, 1e250])
def test_quotients_outside_the_exact_range(scale):
    # dividends below 2^-600 and above 2^600: the statements are evaluated with IEEE division
    a, b = (F.Stokes2DFused(MOD, 40, 37, graph=False) for _ in range(2))
    for sv in (a, b):
        _start(sv, 4, scale)
        sv.Rog.fill_(0.0)
    a.iterate(9)
    for _ in range(9):
        b.iterate(1)
    ps.synchronize()
    for k in FIELDS:
        assert np.array_equal(_bits(getattr(a, k)), _bits(getattr(b, k))), k


@pytest.mark.parametrize("n,S", [(31, 3), (47, 64), (63, 70)])
def test_batches_with_a_frozen_sample(n, S):
    a, b = (F.Stokes2DBatch(MOD, n, n + 2, S, graph=False) for _ in range(2))
    for sv in (a, b):
        _start(sv, S)
        sv.set_active(1, False)
    before = {k: _bits(getattr(a, k))[:, :, 1].copy() for k in FIELDS}
    a.iterate(13)
    for _ in range(13):
        b.iterate(1)
    ps.synchronize()
    for k in FIELDS:
        ga, gb = _bits(getattr(a, k)), _bits(getattr(b, k))
        assert np.array_equal(ga, gb), k
        assert np.array_equal(ga[:, :, 1], before[k]), k


def test_refused_problems():
    sv = F.Stokes2DFused(MOD, 20, 20, graph=False)
    sv._many(4)  # fills the argument block
    q = sv._many.q
    assert lib.ps_stokes2d_iterate(ctypes.byref(q), 1, None) == -1 and lib.ps_stokes2d_iterate(ctypes.byref(q), -2, None) == -1
    q.alt[0] = q.state[0]
    assert lib.ps_stokes2d_iterate(ctypes.byref(q), 2, None) == -1
    sv._many(2)
    q.coef[1] = sv.Vx.f
    assert lib.ps_stokes2d_iterate(ctypes.byref(q), 2, None) == -1
    assert lib.ps_stokes2d_iterate(None, 2, None) == -1


@pytest.mark.parametrize("shapes", [((30, 20, 5), (7, 9, 5)), ((500, 1100, 2),), ((1, 1, 3), (16, 16, 3), (17, 16, 3), (300, 2, 3))])
def test_plane_reductions_match_the_views(shapes):
    rng = np.random.default_rng(1)
    A = [ps.zeros(*s, eltype=ps.Float64).copy_from(rng.standard_normal(s)) for s in shapes]
    planes = shapes[0][2]
    need = 4 * max(min(-(-s[0] * s[1] // 256), 2048) for s in shapes) * planes * len(A)
    work, out = ps.zeros(need, eltype=ps.Float64), ps.zeros(planes * len(A), eltype=ps.Float64)
    arr = (ps.core.ps_field * len(A))(*[a.f for a in A])
    args = lambda op, nw: (arr, len(A), op, ctypes.c_void_p(work.ptr), nw, ctypes.c_void_p(out.ptr), None)  # noqa: E731
    for code, op in enumerate(("sum", "sum_abs", "max_abs", "mean_abs")):
        assert lib.ps_plane_reduce_noalloc(*args(code, need)) == 0, lib.ps_last_error()
        ps.synchronize()
        want = [a.view((1, 1, s + 1), (a.shape[0], a.shape[1], s + 1)).reduce(op) for s in range(planes) for a in A]
        assert np.array_equal(out.to_host(), want), op
    assert lib.ps_plane_reduce_noalloc(*args(0, need - 1)) == -1


@pytest.mark.parametrize("nx,ny", [(40000, 12), (9, 33000)])
def test_grids_beyond_the_tiles_take_the_two_launches(nx, ny):
    # more than 32768 cells in a dimension: ps_stokes2d_iterate refuses them, the solver does not
    a, b = (F.Stokes2DFused(MOD, nx, ny, nout=4) for _ in range(2))
    for sv in (a, b):
        _start(sv, 3)
    a.iterate_block()
    for _ in range(4):
        b.iterate(1)
    ps.synchronize()
    assert np.isfinite(a.error())
    for k in FIELDS:
        assert np.array_equal(_bits(getattr(a, k)), _bits(getattr(b, k))), k


@pytest.mark.parametrize("batch", [False, True])
def test_without_memory_for_a_second_state(batch, monkeypatch):
    """The second copy of the state is what the blocks of iterations need beyond the solver's arrays: where it
    cannot be had the solver iterates by the two launches."""
    zeros = F.core.zeros
    left = [0]

    def scarce(*shape, **kw):
        left[0] -= 1
        if left[0] < 0:
            raise ps.OutOfMemoryError("device memory")
        return zeros(*shape, **kw)

    make = lambda: F.Stokes2DBatch(MOD, 20, 18, 3, graph=False) if batch else F.Stokes2DFused(MOD, 20, 18, graph=False)  # noqa: E731
    count = [0]
    monkeypatch.setattr(F.core, "zeros", lambda *s, **kw: (count.__setitem__(0, count[0] + 1), zeros(*s, **kw))[1])
    b = make()
    _start(b, 5)
    left[0] = count[0] - 1  # the last array of the second state fails
    monkeypatch.setattr(F.core, "zeros", scarce)
    a = make()
    monkeypatch.undo()
    assert b._many is not None and a._many is None
    _start(a, 5)
    if batch:
        for sv in (a, b):
            for s in range(3):
                sv.set_active(s, True)
    a.iterate(7)
    b.iterate(7)
    ps.synchronize()
    for k in FIELDS:
        assert np.array_equal(_bits(getattr(a, k)), _bits(getattr(b, k))), k


@pytest.mark.parametrize("nx,ny,n", [(700, 520, 2), (700, 520, 3), (300, 200, 2), (300, 200, 3)])
def test_short_blocks(nx, ny, n):
    # either side of the rule by which 2 and 3 iterations of large grids go by the two launches
    a, b = (F.Stokes2DFused(MOD, nx, ny, graph=False) for _ in range(2))
    for sv in (a, b):
        _start(sv, n)
    a.iterate(n)
    for _ in range(n):
        b.iterate(1)
    ps.synchronize()
    for k in FIELDS:
        assert np.array_equal(_bits(getattr(a, k)), _bits(getattr(b, k))), k
