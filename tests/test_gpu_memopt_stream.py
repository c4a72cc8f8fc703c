"""memopt streams against plain kernels, bit for bit, over the grids where the automatic number of planes per
thread changes (2, 4 and 8, with remainders), with 16 and 32 planes given (which the automatic choice takes
from 33 and 67 million cells on), in two and three dimensions and every floating-point type: a stencil,
in-place updates read ahead, quotients of one scalar by an array taken once per value, and the gather form of
a derivative; the latter against the atomic scatter form too."""
import numpy as np
import pytest

import parallelstencil as ps
from parallelstencil import workloads as W

pytestmark = pytest.mark.gpu
MOD = __name__
ps.init_parallel_stencil(ps.AMDGPU, ps.Float64, 3, module=MOD)
DIMS = [(20, 17, 9), (32, 32, 32), (64, 64, 33), (96, 96, 45), (128, 128, 70), (127, 95, 63), (300, 20, 37), (200, 130, 61), (256, 200, 99)]


def _rand(dims, seed, lo=0.0):
    return ps.zeros(*dims, eltype=ps.Float64).copy_from(lo + np.random.default_rng(seed).random(dims))


@pytest.mark.parametrize("dims", DIMS)
def test_stencil_matches_plain(dims):
    T, Cp = _rand(dims, 1), _rand(dims, 2, 1.0)
    outs = []
    for memopt in (False, True):
        T2 = _rand(dims, 3)
        W.define_diffusion3d(memopt, MOD)(T2, T, Cp, 1.1, 0.01, 0.1, 0.2, 0.3)
        outs.append(T2.to_host())
    assert np.array_equal(*outs)


@pytest.mark.parametrize("dims", DIMS)
def test_in_place_updates_match_plain(dims):
    nx, ny, nz = dims
    outs = []
    for memopt in (False, True):
        P, Vx, Vy, Vz = (_rand(d, i) for i, d in enumerate((dims, (nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1))))
        kV, kP = W.define_acoustic3d(MOD, memopt)
        for _ in range(3):
            kV(Vx, Vy, Vz, P, 0.01, 1.3, 0.1, 0.2, 0.3)
            kP(P, Vx, Vy, Vz, 0.01, 0.9, 0.1, 0.2, 0.3)
        outs.append([A.to_host() for A in (P, Vx, Vy, Vz)])
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


QUOT = """
@parallel_indices (ix,iy,iz) function quotients!(B, A, C, s)
    if (1 < ix < size(A,1) && 1 < iy < size(A,2) && 1 < iz < size(A,3))
        B[ix,iy,iz] = B[ix,iy,iz] + A[ix-1,iy,iz]*(s/C[ix-1,iy,iz]) + A[ix+1,iy,iz]*(s/C[ix+1,iy,iz]) + A[ix,iy-1,iz]*(s/C[ix,iy-1,iz]) - A[ix,iy,iz-1]*(s/C[ix,iy,iz-1]) + s/C[ix,iy,iz+1]
    end
    return
end
"""


@pytest.mark.parametrize("fastmath", [False, True])
@pytest.mark.parametrize("dims", [(20, 17, 9), (128, 40, 70), (256, 64, 33)])
def test_quotients_by_an_array_match_plain(dims, fastmath):
    A, C = _rand(dims, 1), _rand(dims, 2, -0.5)  # divisors of both signs, some near zero
    h = C.to_host()
    h[3, 4, 5], h[4, 4, 5] = 0.0, np.inf
    C.copy_from(h)
    outs = []
    for memopt in (False, True):
        B = _rand(dims, 3)
        ps.core._define("parallel_indices", QUOT, {"memopt": memopt, "fastmath": fastmath}, MOD)(B, A, C, 0.7)
        outs.append(B.to_host())
    if fastmath:
        # contraction may differ between the two kernels: each of the six terms (large where C is near
        # zero, and they cancel) within a few roundings, so 16 eps of the sum of their magnitudes
        a, q = A.to_host(), 0.7 / np.abs(np.where(h == 0, np.nan, h))
        mag = 2.0 + sum(np.roll(q * a, s, ax) for s, ax in ((1, 0), (-1, 0), (1, 1), (1, 2))) + np.roll(q, -1, 2)
        ok = np.isfinite(outs[0]) & np.isfinite(mag)
        assert np.array_equal(np.isfinite(outs[0]), np.isfinite(outs[1]))
        assert (np.abs(outs[0] - outs[1])[ok] <= 16 * 2.0 ** -52 * mag[ok]).all()
    else:
        assert np.array_equal(*outs, equal_nan=True)


@pytest.mark.parametrize("memopt", [False, True])
@pytest.mark.parametrize("dims", DIMS[:7])
def test_gather_matches_scatter(dims, memopt):
    k = W.define_diffusion3d(memopt, MOD)
    d = k._derivative("Reverse", {"T2": "DuplicatedNoNeed", "T": "DuplicatedNoNeed"})
    T, T2, Cp = _rand(dims, 1), _rand(dims, 2), _rand(dims, 3, 1.0)
    outs = []
    for gather in (False, True):
        S, R = _rand(dims, 4, -0.5), _rand(dims, 5)
        d.use_gather = gather
        d(T2, T, Cp, 1.1, 0.01, 0.1, 0.2, 0.3, S, R)
        outs.append((S.to_host(), R.to_host()))
    assert np.array_equal(outs[0][0], outs[1][0])
    # seven products a cell, each a few roundings, in either order: 1e-14 of the largest term (about 5)
    assert np.abs(outs[0][1] - outs[1][1]).max() <= 1e-13


NP = {ps.Float64: np.float64, ps.Float32: np.float32, ps.BFloat16: np.float32}
STENCIL2D = """
@parallel function stencil2d!(T2, T, Ci, lam, dt, dx, dy)
    @inn(T2) = @inn(T) + dt*(lam*@inn(Ci)*(@d2_xi(T)/dx/dx + @d2_yi(T)/dy/dy))
    return
end
"""
QUOT2D = """
@parallel_indices (ix,iy) function quotients2d!(B, A, C, s)
    if (1 < ix < size(A,1) && 1 < iy < size(A,2))
        B[ix,iy] = B[ix,iy] + A[ix-1,iy]*(s/C[ix-1,iy]) + A[ix+1,iy]*(s/C[ix+1,iy]) - A[ix,iy-1]*(s/C[ix,iy-1]) + s/C[ix,iy+1]
    end
    return
end
"""
ACOUSTIC2D = """
@parallel function step2d!(P, Vx, Vy, dt, k, dx, dy)
    @all(P) = @all(P) - dt*k*(@d_xa(Vx)/dx + @d_ya(Vy)/dy)
    return
end
"""


def _field(dims, et, seed, lo=0.0):
    h = (lo + np.random.default_rng(seed).random(dims)).astype(np.float32 if et != ps.Float64 else np.float64)
    return ps.zeros(*dims, eltype=et).copy_from(ps.f32_to_bf16(h) if et == ps.BFloat16 else h)


def _module(et, nd):
    mod = f"{MOD}.{et}.{nd}"
    if not ps.is_initialized(mod):
        ps.init_parallel_stencil(ps.AMDGPU, ps.Float64 if et == ps.Float64 else ps.Float32, nd, module=mod)
    return mod


@pytest.mark.parametrize("loopsize", [None, 16, 32])
@pytest.mark.parametrize("et", [ps.Float64, ps.Float32, ps.BFloat16])
@pytest.mark.parametrize("dims", [(20, 17), (256, 130), (257, 131), (96, 515), (1030, 1021), (64, 20, 70), (33, 19, 40), (130, 61, 45)])
def test_types_and_dimensions_match_plain(dims, et, loopsize):
    nd, t = len(dims), NP[et]
    mod = _module(et, nd)
    kw = {} if loopsize is None else {"loopsize": loopsize}
    stag = [tuple(n + (i == d) for i, n in enumerate(dims)) for d in range(nd)]
    outs = []
    for memopt in (False, True):
        opts = dict(kw, memopt=True) if memopt else {}
        d = lambda kind, text: ps.core._define(kind, text, opts, mod)  # noqa: B023, E731
        kst = d("parallel", STENCIL2D) if nd == 2 else d("parallel", W.DIFFUSION3D)
        kq = d("parallel_indices", QUOT2D if nd == 2 else QUOT)
        kp = d("parallel", ACOUSTIC2D) if nd == 2 else d("parallel", W.ACOUSTIC3D_P)
        steps = [t(v) for v in (0.1, 0.2, 0.3)[:nd]]
        T2, B, P, S, R = (_field(dims, et, i) for i in range(5))
        T, C = _field(dims, et, 5), _field(dims, et, 6, 0.5)
        kst(T2, T, C, t(1.1), t(0.001), *steps)
        if dims in ((20, 17), (256, 130), (96, 515), (64, 20, 70)):  # sizes that a block divides: a memopt kernel with indices refuses others
            kq(B, T, C, t(0.7))
        for _ in range(2):
            kp(P, *(_field(s, et, 7 + i) for i, s in enumerate(stag)), t(0.01), t(0.9), *steps)
        g = kst._derivative("Reverse", {"T2": "DuplicatedNoNeed", "T": "DuplicatedNoNeed"})._gather[0]
        assert g.info["memopt"] is memopt
        ps.core.Kernel.__call__(g, T2, T, C, t(1.1), t(0.001), *steps, S, R)
        outs.append([A.to_host() for A in (T2, B, P, R)])
    for name, a, b in zip(("stencil", "quotients", "in place", "gather"), *outs):
        assert np.array_equal(a, b), name


@pytest.mark.parametrize("loopsize", [16, 32])
@pytest.mark.parametrize("dims", [(20, 17, 9), (64, 64, 33), (127, 95, 63), (200, 130, 61)])
def test_gather_with_long_streams_matches_scatter(dims, loopsize):
    k = W.define_diffusion3d(True, MOD, loopsize=loopsize)
    d = k._derivative("Reverse", {"T2": "DuplicatedNoNeed", "T": "DuplicatedNoNeed"})
    T, T2, Cp = _rand(dims, 1), _rand(dims, 2), _rand(dims, 3, 1.0)
    outs = []
    for gather in (False, True):
        S, R = _rand(dims, 4, -0.5), _rand(dims, 5)
        d.use_gather = gather
        d(T2, T, Cp, 1.1, 0.01, 0.1, 0.2, 0.3, S, R)
        outs.append((S.to_host(), R.to_host()))
    assert np.array_equal(outs[0][0], outs[1][0])
    assert np.abs(outs[0][1] - outs[1][1]).max() <= 1e-13  # as in test_gather_matches_scatter

INDIRECT = """
@parallel_indices (ix,iy,iz) function indirect!(B, C, I, s)
    if (1 < ix < size(B,1) && 1 < iy < size(B,2) && 1 < iz < size(B,3))
        B[ix,iy,iz] = s/C[ix,iy,iz-1] + s/C[ix,iy,iz+1] + s/C[I[ix,iy,iz],iy,iz]
    end
    return
end
"""


def test_quotient_of_an_element_found_by_an_index_array():
    # the index is served by a register of the stream, the divisor is not: it is still divided by
    dims = (64, 20, 70)
    C = _rand(dims, 1, 0.5)
    I = ps.zeros(*dims, eltype=ps.Int64).copy_from(np.asfortranarray(np.random.default_rng(2).integers(1, dims[0] + 1, dims)))  # noqa: E741
    outs = []
    for memopt in (False, True):
        B = _rand(dims, 3)
        ps.core._define("parallel_indices", INDIRECT, {"memopt": memopt, "inbounds": True}, MOD)(B, C, I, 0.7)
        outs.append(B.to_host())
    assert np.array_equal(*outs)
