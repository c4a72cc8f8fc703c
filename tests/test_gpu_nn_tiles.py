"""The tiled network kernels at the sizes where their tiles, masks and dispatch rules change: the 3x3
convolution and its weight gradient against the stored column matrix, the piecewise data movement
against one element at a time (a pointer shifted by one element takes that path), the bias gradient
against float64 sums."""
import ctypes

import numpy as np
import pytest

import parallelstencil as ps
from parallelstencil import unet as U
from parallelstencil._lib import lib

pytestmark = pytest.mark.gpu


def _bf(a):
    return ps.bf16_to_f32(ps.f32_to_bf16(np.asarray(a, np.float32)))


# image sizes around the 8- and 16-column tiles, channels around the groups of 8 and 32 and beyond what
# one patch in LDS holds, output channels around 32 and 64. These take the tile of 128 x 32 (or the general
# product), as their tiles are fewer than the CUs, but for 1 x 300 x 260, 32 -> 32.
CONV = [(1, 1, 1, 8, 8), (2, 15, 17, 32, 33), (1, 16, 16, 24, 31), (3, 9, 8, 40, 65), (1, 33, 31, 7, 4), (2, 20, 24, 128, 130), (1, 70, 70, 96, 32),
        (4, 64, 64, 192, 64), (1, 10, 40, 384, 96), (1, 12, 12, 512, 16), (1, 300, 260, 32, 32), (2, 5, 100, 9, 12), (1, 17, 130, 2, 3), (2, 21, 37, 3, 40)]
# the other tiles, which need that many pixels: 256 x 64, 128 x 64 and 256 x 32, each with whole and ragged
# sizes and with channels that are multiples of 32, multiples of 8 and (256 x 32) neither
LARGE = [(1, 256, 256, 192, 64), (3, 130, 170, 160, 70), (2, 200, 180, 136, 70), (8, 64, 64, 192, 64), (1, 128, 128, 384, 128), (2, 150, 130, 168, 40),
         (1, 150, 150, 264, 130), (2, 181, 190, 64, 33), (2, 180, 200, 24, 20), (1, 260, 300, 3, 20)]
# few output channels: the explicit product of so thin a side must not take another order of summation (BF16
# results show one in about ten thousand sums)
THIN_OUT = [(1, 300, 301, 8, 1), (2, 130, 130, 24, 3), (1, 201, 190, 32, 3), (1, 160, 170, 56, 4), (1, 16, 16, 40, 2)]


def _tile(B, H, W, C, N):
    """(pixels, channels) of the convolution's tile, None for the general product, and the kind of its
    channels: the rule of conv3_launch restated."""
    up = lambda a, b: -(-a // b)  # noqa: E731

    def fits(pix, nb):
        w16, w8 = up(W, 16) * up(H, pix // 16), up(W, 8) * up(H, pix // 8)
        lg = 3 if w8 < w16 else 4
        stride = (C // 8 | 1) * 8 if C % 8 == 0 else C
        return min(w16, w8) * B, 2 * (2 * 64 * (nb + 8) + ((pix >> lg) + 2) * ((1 << lg) + 2) * stride)

    tiles = [(256, 64), (128, 64), (256, 32), (128, 32)]
    for t in tiles[2 if fits(256, 32)[1] <= 80 << 10 else 0:]:
        n, lds = fits(*t)
        if lds <= 160 << 10 and (t == (128, 32) or n * up(N, t[1]) >= 256):
            return t, "odd" if C % 8 else "32" if C % 32 == 0 else "8"
    return None, None


def test_the_lists_reach_every_tile():
    taken = {_tile(*c) for c in CONV + LARGE}
    assert taken >= {((256, 64), "32"), ((256, 64), "8"), ((128, 64), "32"), ((128, 64), "8"), ((256, 32), "32"), ((256, 32), "8"), ((256, 32), "odd"),
                     ((128, 32), "32"), ((128, 32), "8"), ((128, 32), "odd"), (None, None)}
    assert all(_tile(*c)[0] not in ((128, 32), None) for c in LARGE)


@pytest.mark.parametrize("B,H,W,C,N", CONV + LARGE + THIN_OUT)
def test_convolution_matches_the_column_matrix(B, H, W, C, N):
    rng = np.random.default_rng(B * H * W + C + N)
    P, K = B * H * W, 9 * C
    x, w = U.Buf((B, H, W, C)).upload(rng.standard_normal((B, H, W, C))), U.Buf((K, N)).upload(rng.standard_normal((K, N)))
    bias, col = U.Buf((N,), "f32").upload(rng.standard_normal(N)), U.Buf((P, K))
    ps.core.check(lib.ps_nn_im2col(x.p, B, H, W, C, col.p, None))
    for epi in (U.EPI_BF16, U.EPI_BIAS, U.EPI_BIAS_RELU):
        ye, yi = U.Buf((P, N)), U.Buf((P, N))
        U.gemm(P, N, K, col, K, 1, w, N, 1, ye, N, bias, epi)
        U.gemm_im2col(0, P, N, K, x, H, W, C, w, N, 1, yi, N, bias, epi)
        assert np.array_equal(ye.download(), yi.download()), epi


@pytest.mark.parametrize("strides", ["transposed", "wide"])
def test_convolution_with_other_weight_and_result_strides(strides):
    rng = np.random.default_rng(3)
    B, H, W, C, N = 1, 20, 20, 32, 40
    P, K = B * H * W, 9 * C
    x, wh = U.Buf((B, H, W, C)).upload(rng.standard_normal((B, H, W, C))), _bf(rng.standard_normal((K, N)))
    col = U.Buf((P, K))
    ps.core.check(lib.ps_nn_im2col(x.p, B, H, W, C, col.p, None))
    if strides == "transposed":
        w, sk, sn, ld = U.Buf((N, K)).upload(wh.T), 1, K, N
    else:
        w, sk, sn, ld = U.Buf((K, N + 3)).upload(np.pad(wh, ((0, 0), (0, 3)))), N + 3, 1, N + 5
    ye, yi = U.Buf((P, ld)), U.Buf((P, ld))
    U.gemm(P, N, K, col, K, 1, w, sk, sn, ye, ld)
    U.gemm_im2col(0, P, N, K, x, H, W, C, w, sk, sn, yi, ld)
    assert np.array_equal(ye.download(), yi.download())


@pytest.mark.parametrize("special", [np.inf, np.nan])
def test_convolution_of_infinities_and_nan(special):
    # a value outside the window of a pixel, or behind the last k, must not reach it
    rng = np.random.default_rng(5)
    B, H, W, C, N = 1, 18, 21, 24, 40
    P, K = B * H * W, 9 * C
    xh = rng.standard_normal((B, H, W, C))
    xh[0, 7, 9, 3] = special
    x, w, col = U.Buf(xh.shape).upload(xh), U.Buf((K, N)).upload(rng.standard_normal((K, N))), U.Buf((P, K))
    ps.core.check(lib.ps_nn_im2col(x.p, B, H, W, C, col.p, None))
    ye, yi = U.Buf((P, N)), U.Buf((P, N))
    U.gemm(P, N, K, col, K, 1, w, N, 1, ye, N)
    U.gemm_im2col(0, P, N, K, x, H, W, C, w, N, 1, yi, N)
    a, b = ye.download(), yi.download()
    assert np.array_equal(a, b, equal_nan=True) and np.isfinite(b).sum() == (P - 9) * N
    dy = U.Buf((P, N)).upload(rng.standard_normal((P, N)))
    ge, gi = U.Buf((K, N), "f32").zero(), U.Buf((K, N), "f32").zero()
    U.gemm(K, N, P, col, 1, K, dy, N, 1, ge, N, epi=U.EPI_F32_ADD, splitk=2)
    U.gemm_im2col(1, K, N, P, x, H, W, C, dy, N, 1, gi, N, epi=U.EPI_F32_ADD, splitk=2)
    assert np.array_equal(np.isfinite(ge.download()), np.isfinite(gi.download()))


@pytest.mark.parametrize("B,H,W,C,N", CONV)
def test_weight_gradient_against_float64(B, H, W, C, N):
    """FP32 sums of P products of BF16 values in any order are within P eps of the sum of magnitudes in the
    worst case, about 0.64 P here; the bound of 8 eps (P + 4 sqrt P), linear in P, is that of eight roundings
    of the sum of magnitudes (pixels of a tile, tiles of a workgroup, wavefronts, workgroups), as the sums
    are taken in pieces."""
    rng = np.random.default_rng(B + H + W + C + N)
    P, K = B * H * W, 9 * C
    xh, dh = _bf(rng.standard_normal((B, H, W, C))), _bf(rng.standard_normal((P, N)))
    x, dy = U.Buf(xh.shape).upload(xh), U.Buf(dh.shape).upload(dh)
    g = U.Buf((K, N), "f32").upload(np.ones((K, N)))
    U.gemm_im2col(1, K, N, P, x, H, W, C, dy, N, 1, g, N, epi=U.EPI_F32_ADD, splitk=2)
    xp = np.pad(xh.astype(np.float64), ((0, 0), (1, 1), (1, 1), (0, 0)))
    d64 = dh.astype(np.float64)
    got = g.download().astype(np.float64) - 1.0
    for t in range(9):
        ref = xp[:, t // 3:t // 3 + H, t % 3:t % 3 + W].reshape(P, C).T @ d64
        assert np.abs(got[t * C:(t + 1) * C] - ref).max() <= 8 * 2.0 ** -24 * (P + 4 * np.sqrt(P)), t


def _shifted(a, off):
    """A device copy of `a` that starts `off` elements into its buffer."""
    b = U.Buf((a.size + 8,))
    b.upload(np.concatenate([np.zeros(off), a.reshape(-1), np.zeros(8 - off)]))
    return b, ctypes.c_void_p(b.p.value + 2 * off)


def _read(b, off, n):
    return b.download()[off:off + n]


@pytest.mark.parametrize("C", [8, 24, 64, 5])
def test_data_movement_in_pieces_matches_single_elements(C):
    rng = np.random.default_rng(C)
    B, H, W = 2, 6, 10
    lo, hi = rng.standard_normal((B, H, W, C)), rng.standard_normal((B, 2 * H, 2 * W, C))
    for name, src, n, args in (("ps_nn_up2", lo, hi.size, (B, H, W, C)), ("ps_nn_up2_bwd", hi, lo.size, (B, H, W, C)),
                               ("ps_nn_pool2", hi, lo.size, (B, 2 * H, 2 * W, C)), ("ps_nn_pool2_bwd", lo, hi.size, (B, 2 * H, 2 * W, C))):
        outs = []
        for off in (0, 1):
            (s, sp), (d, dp) = _shifted(src, off), _shifted(np.zeros(n), off)
            ps.core.check(getattr(lib, name)(sp, *args, dp, None))
            outs.append(_read(d, off, n))
        assert np.array_equal(*outs) and np.any(outs[0]), name
    P, Cb = B * H * W, 16 if C % 8 == 0 else 3
    a, b = rng.standard_normal((P, C)), rng.standard_normal((P, Cb))
    for off in (0, 1):
        (_a, ap), (_b, bp), (y, yp) = _shifted(a, off), _shifted(b, off), _shifted(np.zeros((P, C + Cb)), off)
        ps.core.check(lib.ps_nn_concat(ap, C, bp, Cb, P, yp, None))
        assert np.array_equal(_read(y, off, P * (C + Cb)).reshape(P, -1), np.concatenate([_bf(a), _bf(b)], 1))
        (da, dap), (db, dbp) = _shifted(0 * a, off), _shifted(0 * b, off)
        ps.core.check(lib.ps_nn_split(yp, C, Cb, P, dap, dbp, None))
        assert np.array_equal(_read(da, off, a.size), _bf(a).reshape(-1)) and np.array_equal(_read(db, off, b.size), _bf(b).reshape(-1))
    n = P * C
    for off in (0, 1):
        (d, dp), (y, yp) = _shifted(a, off), _shifted(lo, off)
        ps.core.check(lib.ps_nn_relu_bwd(dp, yp, n, None))
        assert np.array_equal(_read(d, off, n), np.where(_bf(lo).reshape(-1) > 0, _bf(a).reshape(-1), 0))
        ps.core.check(lib.ps_nn_add_bf16(dp, yp, n, None))
        want = _bf(np.where(_bf(lo).reshape(-1) > 0, _bf(a).reshape(-1), 0) + _bf(lo).reshape(-1))
        assert np.array_equal(_read(d, off, n), want)


@pytest.mark.parametrize("M,N", [(1, 8), (63, 3), (65, 24), (4097, 1), (70000, 32), (300, 2056), (20000, 256), (129, 300)])
def test_bias_gradient_against_float64(M, N):
    rng = np.random.default_rng(M + N)
    d = _bf(rng.standard_normal((M, N)))
    db, g = U.Buf((M, N)).upload(d), U.Buf((N,), "f32").upload(np.ones(N))
    ps.core.check(lib.ps_nn_bias_grad(db.p, M, N, g.p, None))
    # FP32 partial sums: at most M roundings of values below the sum of magnitudes
    assert np.abs(g.download() - 1.0 - d.astype(np.float64).sum(0)).max() <= 2.0 ** -24 * (np.abs(d).sum(0).max() * np.sqrt(M) + 8)


@pytest.mark.parametrize("M,N,K", [(1, 1, 8), (257, 3, 32), (1000, 4, 24), (70001, 2, 512), (5, 3, 40), (300, 4, 72), (300, 3, 504)])
def test_thin_results_against_float64(M, N, K):
    # K FP32 products and sums of BF16 values, rounded once to BF16 (2^-8 of the value) at the end
    rng = np.random.default_rng(M + N + K)
    a, w, bias = _bf(rng.standard_normal((M, K))), _bf(rng.standard_normal((K, N))), rng.standard_normal(N).astype(np.float32)
    A, Wb, bb = U.Buf((M, K)).upload(a), U.Buf((K, N)).upload(w), U.Buf((N,), "f32").upload(bias)
    ref = a.astype(np.float64) @ w.astype(np.float64)
    mag = np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64) + 4
    for epi, want in ((U.EPI_BF16, ref), (U.EPI_BIAS, ref + bias), (U.EPI_BIAS_RELU, np.maximum(ref + bias, 0))):
        C = U.Buf((M, N))
        U.gemm(M, N, K, A, K, 1, Wb, N, 1, C, N, bb, epi)
        assert (np.abs(C.download() - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -22 * mag).all(), epi


@pytest.mark.parametrize("M,N,K", [(1, 8, 1), (300, 32, 3), (70001, 24, 4), (65, 512, 2)])
def test_thin_sums_against_float64(M, N, K):
    rng = np.random.default_rng(M + N + K)
    a, w = _bf(rng.standard_normal((M, K))), _bf(rng.standard_normal((N, K)))
    A, Wb, C = U.Buf((M, K)).upload(a), U.Buf((N, K)).upload(w), U.Buf((M, N))
    U.gemm(M, N, K, A, K, 1, Wb, 1, K, C, N)
    ref = a.astype(np.float64) @ w.T.astype(np.float64)
    assert (np.abs(C.download() - ref) <= 2.0 ** -8 * np.abs(ref) + 2.0 ** -20).all()


@pytest.mark.parametrize("M,N,K", [(8, 1, 300), (32, 3, 131072), (24, 4, 1000), (2048, 2, 700), (2056, 2, 700), (64, 3, 50), (256, 3, 600), (256, 4, 70000),
                                   (264, 1, 4000), (8, 4, 5)])
def test_thin_gradients_against_float64(M, N, K):
    rng = np.random.default_rng(M + N + K)
    a, d = _bf(rng.standard_normal((K, M))), _bf(rng.standard_normal((K, N)))
    A, D, G = U.Buf((K, M)).upload(a), U.Buf((K, N)).upload(d), U.Buf((M, N), "f32").upload(np.ones((M, N)))
    U.gemm(M, N, K, A, 1, M, D, N, 1, G, N, epi=U.EPI_F32_ADD, splitk=3)
    ref = a.astype(np.float64).T @ d.astype(np.float64)
    # FP32 sums of K products in any order, as for the weight gradient above
    assert np.abs(G.download() - 1.0 - ref).max() <= 8 * 2.0 ** -24 * (K + 4 * np.sqrt(K))
