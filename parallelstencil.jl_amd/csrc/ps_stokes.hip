// Several pseudo-transient Stokes2D iterations (miniapps/Stokes2D.jl:111-116) per launch.
//
// One iteration reaches one cell: the velocities of a cell after it depend on the velocities,
// pressures and coefficients of the cell and its eight neighbours. A workgroup that holds a tile and
// k cells around it can therefore make k iterations on its own: it reads the state and the
// coefficients once, keeps what neighbours read (Vx, Vy, Pt, txx, tyy, txy) in LDS and the rest in
// registers, and writes the tile once. The two-launch iteration streams 26 array accesses per cell
// and iteration through the caches and pays two launches; k iterations here cost 15 accesses (the
// halo's on top) and one launch. Workgroups read their neighbours' old state while those write the new
// one, so launches alternate between the state and a second copy of it; an even number of launches
// ends in the state itself. The last iteration of the last launch also writes the residuals, the
// divergence and the stresses, which nothing reads between two iterations.
//
// Every statement keeps the miniapp's operations in the miniapp's order (this file is compiled without
// contraction), so the fields are bit for bit those of the two-launch iteration. Quotients by dx and
// dy go through the host's reciprocal with the Markstein correction (P. Markstein, IBM J. Res. Dev.
// 34(1), 1990), exact while the dividend's exponent lies in [-600, 600); a statement group with a
// dividend outside it, or whose values hold a NaN, is evaluated again with IEEE division.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <string>

#include "ps_amd.h"
#include "ps_internal.h"

namespace {

struct Arr {  // one field: sample s is the plane at p + s*plane, cell (i, j) at i + j*pitch
  double* p;
  int pitch;
  long long plane;
  __device__ double* at(int s) const { return p + s * plane; }
};

struct StokesArgs {
  Arr Vx, Vy, Pt, aX, aY;        // state read
  Arr nVx, nVy, nPt, naX, naY;   // state written
  Arr tPt, Mus, tVx, tVy, Rog;   // pseudo-time steps, viscosity, buoyancy
  Arr dV, txx, tyy, txy, Rx, Ry; // written by the last iteration
  const double* act;             // one flag per sample (0: the sample's fields stay as they are), or NULL
  long long act_plane;
  double dx, dy, rdx, rdy, dampX, dampY;
  int nx, ny, k, ntx, nty;
  int ieee;  // the divisors do not suit the corrected reciprocal
};

// a/b through r = RN(1/b); lo, hi: extreme exponents of the dividends so far
__device__ __forceinline__ double quot(double a, double b, double r, int& lo, int& hi) {
  const int e = __builtin_amdgcn_frexp_exp(a);
  lo = min(lo, e);
  hi = max(hi, e);
  const double q = a * r, t = __builtin_fma(q, b, -a);
  return __builtin_fma(-t, r, q);
}

// One cell per lane and CPT cells per thread of a P x PH region (tile and halo; smaller at the walls and
// where the tiles are smaller). The pitch P is a constant so that the neighbours' places in LDS are
// constant offsets, and what a cell takes part in are lane masks made once: the iterations are bound by
// their vector instructions, of which addresses and flags were a third.
template <int CPT, int P, int PH, bool LAST>
__global__ void __launch_bounds__((P * PH / CPT + 63) / 64 * 64) stokes2d_k(StokesArgs A) {
  constexpr int NTH = (P * PH / CPT + 63) / 64 * 64, NC = P * PH;
  static_assert(NTH <= 1024 && P * PH % CPT == 0, "one workgroup holds the region");
  // cells at the region's edge read a row or column outside it, into what they compute in vain: one pitch
  // and one cell of slack on either side of the six arrays keeps that inside
  constexpr int SLACK = P + 1;
  __shared__ double lds[6 * NC + 2 * SLACK];
  double* const vx = lds + SLACK;
  double* const vy = vx + NC;
  double* const pt = vy + NC;
  double* const sxx = pt + NC;
  double* const syy = sxx + NC;
  double* const sxy = syy + NC;
  const int s = blockIdx.y;
  if (A.act && A.act[s * A.act_plane] == 0.0) return;
  const int nx = A.nx, ny = A.ny, k = A.k;
  // Cells -1..n-1 per dimension: cell (i, j) owns Vx(i+1, j) and Vy(i, j+1), so the cells at -1 own the
  // first wall nodes. The tiles split the n + 1 cells evenly.
  const int bx = blockIdx.x % A.ntx, by = blockIdx.x / A.ntx;
  const int x0 = (int)((long long)bx * (nx + 1) / A.ntx) - 1, x1 = (int)((long long)(bx + 1) * (nx + 1) / A.ntx) - 1;  // tile [x0, x1)
  const int y0 = (int)((long long)by * (ny + 1) / A.nty) - 1, y1 = (int)((long long)(by + 1) * (ny + 1) / A.nty) - 1;
  const int rx0 = max(-1, x0 - k), rx1 = min(nx, x1 + k), ry0 = max(-1, y0 - k), ry1 = min(ny, y1 + k);  // with the halo
  const int RW = rx1 - rx0, RH = ry1 - ry0;  // at most P, PH

  for (int e = threadIdx.x; e < 6 * NC + 2 * SLACK; e += NTH) lds[e] = 0.0;
  __syncthreads();
  // divergence and normal stresses; shear stress; Vx; Vy; the free-slip copies of Vx down and up, of Vy
  // left and right; in the tile
  bool dP[CPT], dT[CPT], dX[CPT], dY[CPT], cD[CPT], cU[CPT], cL[CPT], cR[CPT], tile[CPT];
  double mus2[CPT], mun2[CPT], tpt[CPT], tvx[CPT], tvy[CPT], rog[CPT], ax[CPT], ay[CPT], p[CPT];
#pragma unroll
  for (int m = 0; m < CPT; ++m) {
    const int c = threadIdx.x + m * NTH, lj = c / P, li = c - lj * P, i = rx0 + li, j = ry0 + lj;
    const bool have = c < NC && li < RW && lj < RH, in = have && i >= 0 && j >= 0;
    const bool left = li > 0, right = li < RW - 1, down = lj > 0, up = lj < RH - 1;
    dP[m] = in && left && down;
    dT[m] = in && i <= nx - 2 && j <= ny - 2 && right && up;
    dX[m] = in && i <= nx - 2 && j >= 1 && j <= ny - 2 && right && down;
    dY[m] = in && i >= 1 && i <= nx - 2 && j <= ny - 2 && left && up;
    cD[m] = have && j == 1 && down;
    cU[m] = have && j == ny - 2 && up;
    cL[m] = have && i == 1 && left;
    cR[m] = have && i == nx - 2 && right;
    tile[m] = have && i >= x0 && i < x1 && j >= y0 && j < y1;
    mus2[m] = mun2[m] = tpt[m] = tvx[m] = tvy[m] = rog[m] = ax[m] = ay[m] = p[m] = 0.0;
    if (have && j >= 0) vx[c] = A.Vx.at(s)[i + 1 + j * A.Vx.pitch];
    if (have && i >= 0) vy[c] = A.Vy.at(s)[i + (j + 1) * A.Vy.pitch];
    if (in) {
      const double* const M = A.Mus.at(s) + i + j * A.Mus.pitch;
      mus2[m] = 2.0 * M[0];
      if (dT[m]) mun2[m] = 2.0 * ((M[0] + M[1] + M[A.Mus.pitch] + M[A.Mus.pitch + 1]) * 0.25);
      p[m] = A.Pt.at(s)[i + j * A.Pt.pitch];
      tpt[m] = A.tPt.at(s)[i + j * A.tPt.pitch];
      pt[c] = p[m];
    }
    if (dX[m]) {
      ax[m] = A.aX.at(s)[i + (j - 1) * A.aX.pitch];
      tvx[m] = A.tVx.at(s)[i + (j - 1) * A.tVx.pitch];
    }
    if (dY[m]) {
      ay[m] = A.aY.at(s)[i - 1 + j * A.aY.pitch];
      tvy[m] = A.tVy.at(s)[i - 1 + j * A.tVy.pitch];
      const double* const G = A.Rog.at(s) + i + j * A.Rog.pitch;
      rog[m] = (G[0] + G[A.Rog.pitch]) * 0.5;
    }
  }
  __syncthreads();
  const double dx = A.dx, dy = A.dy, rx = A.rdx, ry = A.rdy, third = 1.0 / 3.0;
  const int never = A.ieee ? 1 << 30 : 0;  // divisors the corrected reciprocal does not suit: always divide
  int at[CPT];
#pragma unroll
  for (int m = 0; m < CPT; ++m) at[m] = min((int)threadIdx.x + m * NTH, NC - 1);
  for (int it = 0; it < k; ++it) {
    const bool write = LAST && it == k - 1;
    // Every cell computes every statement, all cells' reads first: what is not valid (outside the region,
    // at walls) is read by no valid cell and not written to memory.
    {
      int lo = 0, hi = never;
      double d1[CPT], d2[CPT], d3[CPT], d4[CPT], pn[CPT], dV[CPT], nxx[CPT], nyy[CPT], nxy[CPT], sum = 0.0;
#pragma unroll
      for (int m = 0; m < CPT; ++m) {
        const int c = at[m];
        const double u = vx[c], v = vy[c];
        d1[m] = u - vx[c - 1];
        d2[m] = v - vy[c - P];
        d3[m] = vx[c + P] - u;
        d4[m] = vy[c + 1] - v;
      }
#pragma unroll
      for (int m = 0; m < CPT; ++m) {
        const double ex = quot(d1[m], dx, rx, lo, hi), ey = quot(d2[m], dy, ry, lo, hi);
        dV[m] = ex + ey;
        pn[m] = p[m] - tpt[m] * dV[m];
        nxx[m] = mus2[m] * (ex - third * dV[m]);
        nyy[m] = mus2[m] * (ey - third * dV[m]);
        nxy[m] = mun2[m] * (0.5 * (quot(d3[m], dy, ry, lo, hi) + quot(d4[m], dx, rx, lo, hi)));
        sum += ((pn[m] + nxx[m]) + nyy[m]) + nxy[m];
      }
      if (lo < -599 || hi > 600 || sum != sum) {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
          const double ex = d1[m] / dx, ey = d2[m] / dy;
          dV[m] = ex + ey;
          pn[m] = p[m] - tpt[m] * dV[m];
          nxx[m] = mus2[m] * (ex - third * dV[m]);
          nyy[m] = mus2[m] * (ey - third * dV[m]);
          nxy[m] = mun2[m] * (0.5 * (d3[m] / dy + d4[m] / dx));
        }
      }
#pragma unroll
      for (int m = 0; m < CPT; ++m) {
        const int c = at[m];
        p[m] = pn[m];
        if (NTH * CPT == NC || (int)threadIdx.x + m * NTH < NC) {
          pt[c] = pn[m];
          sxx[c] = nxx[m];
          syy[c] = nyy[m];
          sxy[c] = nxy[m];
        }
        if (write && tile[m]) {
          const int lj = c / P, i = rx0 + c - lj * P, j = ry0 + lj;
          if (dP[m]) {
            A.dV.at(s)[i + j * A.dV.pitch] = dV[m];
            A.txx.at(s)[i + j * A.txx.pitch] = nxx[m];
            A.tyy.at(s)[i + j * A.tyy.pitch] = nyy[m];
          }
          if (dT[m]) A.txy.at(s)[i + j * A.txy.pitch] = nxy[m];
        }
      }
    }
    __syncthreads();
    {
      int lo = 0, hi = never;
      double e1[CPT], e2[CPT], e3[CPT], g1[CPT], g2[CPT], g3[CPT], fx[CPT], fy[CPT], wx[CPT], wy[CPT], sum = 0.0;
#pragma unroll
      for (int m = 0; m < CPT; ++m) {
        const int c = at[m];
        const double q = pt[c], t = sxy[c];
        e1[m] = sxx[c + 1] - sxx[c];
        e2[m] = t - sxy[c - P];
        e3[m] = pt[c + 1] - q;
        g1[m] = syy[c + P] - syy[c];
        g2[m] = t - sxy[c - 1];
        g3[m] = pt[c + P] - q;
        wx[m] = vx[c];
        wy[m] = vy[c];
      }
#pragma unroll
      for (int m = 0; m < CPT; ++m) {
        fx[m] = (quot(e1[m], dx, rx, lo, hi) + quot(e2[m], dy, ry, lo, hi)) - quot(e3[m], dx, rx, lo, hi);
        fy[m] = ((quot(g1[m], dy, ry, lo, hi) + quot(g2[m], dx, rx, lo, hi)) - quot(g3[m], dy, ry, lo, hi)) + rog[m];
        sum += fx[m] + fy[m];
      }
      if (lo < -599 || hi > 600 || sum != sum) {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int m = 0; m < CPT; ++m) {
          fx[m] = (e1[m] / dx + e2[m] / dy) - e3[m] / dx;
          fy[m] = ((g1[m] / dy + g2[m] / dx) - g3[m] / dy) + rog[m];
        }
      }
#pragma unroll
      for (int m = 0; m < CPT; ++m) {
        const int c = at[m];
        ax[m] = A.dampX * ax[m] + fx[m];
        ay[m] = A.dampY * ay[m] + fy[m];
        const double nx_ = wx[m] + tvx[m] * ax[m], ny_ = wy[m] + tvy[m] * ay[m];
        wx[m] = dX[m] ? nx_ : wx[m];
        wy[m] = dY[m] ? ny_ : wy[m];
        if (dX[m]) vx[c] = wx[m];
        if (dY[m]) vy[c] = wy[m];
        // the free-slip rows and columns, written by nobody else and not read before the barrier
        if (cD[m]) vx[c - P] = wx[m];
        if (cU[m]) vx[c + P] = wx[m];
        if (cL[m]) vy[c - 1] = wy[m];
        if (cR[m]) vy[c + 1] = wy[m];
        if (write && tile[m]) {
          const int lj = c / P, i = rx0 + c - lj * P, j = ry0 + lj;
          if (dX[m]) A.Rx.at(s)[i + (j - 1) * A.Rx.pitch] = fx[m];
          if (dY[m]) A.Ry.at(s)[i - 1 + j * A.Ry.pitch] = fy[m];
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int m = 0; m < CPT; ++m) {
    const int c = threadIdx.x + m * NTH, lj = c / P, i = rx0 + c - lj * P, j = ry0 + lj;
    if (!tile[m]) continue;
    if (j >= 0) A.nVx.at(s)[i + 1 + j * A.nVx.pitch] = vx[c];
    if (i >= 0) A.nVy.at(s)[i + (j + 1) * A.nVy.pitch] = vy[c];
    if (i >= 0 && j >= 0) A.nPt.at(s)[i + j * A.nPt.pitch] = p[m];
    if (dX[m]) A.naX.at(s)[i + (j - 1) * A.naX.pitch] = ax[m];
    if (dY[m]) A.naY.at(s)[i - 1 + j * A.naY.pitch] = ay[m];
  }
}

// the divisor's corrected reciprocal is exact: magnitude in [2^-400, 2^400], significand not all ones
bool reciprocal_exact(double b) {
  const double a = std::fabs(b);
  if (!(a >= std::ldexp(1.0, -400) && a <= std::ldexp(1.0, 400))) return false;
  int e;
  const double f = std::frexp(a, &e);
  return std::nextafter(f, 2.0) != 1.0;
}

}  // namespace

extern "C" int ps_stokes2d_iterate(const ps_stokes2d* q, int n, void* stream) {
  if (int r = ps_internal_require_init()) return r;
  hipStream_t st = ps_internal_stream(stream);
  if (!q) return ps_internal_fail(PS_EARGUMENT, "ps_stokes2d_iterate: NULL arguments");
  if (n < 0 || n == 1) return ps_internal_fail(PS_EARGUMENT, "ps_stokes2d_iterate: n must be 0 or at least 2 (an even number of launches ends in the state)");
  if (n == 0) return 0;
  const int64_t nx = q->state[2].dims[0], ny = q->state[2].dims[1], S = q->state[2].dims[2];
  if (nx < 8 || ny < 8 || nx > 32768 || ny > 32768 || S < 1 || S > 65535)
    return ps_internal_fail(PS_EARGUMENT, "ps_stokes2d_iterate: grids of 8 to 32768 cells per dimension, 1 to 65535 samples");
  const int64_t dims[5][2] = {{nx + 1, ny}, {nx, ny + 1}, {nx, ny}, {nx - 1, ny - 2}, {nx - 2, ny - 1}};  // Vx, Vy, cells, x faces, y faces
  StokesArgs A{};
  auto take = [&](const ps_field& f, int kind, Arr& out) -> bool {
    const int64_t w = kind < 5 ? dims[kind][0] : nx - 1, h = kind < 5 ? dims[kind][1] : ny - 1;  // 5: nodes
    if (f.dtype != PS_F64 || !f.ptr || f.ncomp > 1 || f.dims[0] != w || f.dims[1] != h || f.dims[2] != S) return false;
    if (f.pitch < w || f.pitch * h > 0x7fffffffLL) return false;
    out = Arr{(double*)f.ptr, (int)f.pitch, (long long)f.plane};
    return true;
  };
  Arr s0[5], s1[5];
  bool ok = true;
  for (int i = 0; i < 5; ++i) ok = ok && take(q->state[i], i, s0[i]) && take(q->alt[i], i, s1[i]) && q->state[i].ptr != q->alt[i].ptr;
  ok = ok && take(q->coef[0], 2, A.tPt) && take(q->coef[1], 2, A.Mus) && take(q->coef[2], 3, A.tVx) && take(q->coef[3], 4, A.tVy) && take(q->coef[4], 2, A.Rog);
  ok = ok && take(q->out[0], 2, A.dV) && take(q->out[1], 2, A.txx) && take(q->out[2], 2, A.tyy) && take(q->out[3], 5, A.txy) && take(q->out[4], 3, A.Rx) &&
       take(q->out[5], 4, A.Ry);
  if (!ok) return ps_internal_fail(PS_EARGUMENT, "ps_stokes2d_iterate: FP64 fields of the sizes of one Stokes2D problem, with device memory, are needed");
  if (q->act.ptr) {
    if (q->act.dtype != PS_F64 || q->act.dims[2] < S) return ps_internal_fail(PS_EARGUMENT, "ps_stokes2d_iterate: one FP64 activity flag per sample is needed");
    A.act = (const double*)q->act.ptr;
    A.act_plane = q->act.plane;
  }
  A.dx = q->dx;
  A.dy = q->dy;
  A.rdx = 1.0 / q->dx;
  A.rdy = 1.0 / q->dy;
  A.ieee = !(reciprocal_exact(q->dx) && reciprocal_exact(q->dy));
  A.dampX = q->dampX;
  A.dampY = q->dampY;
  A.nx = (int)nx;
  A.ny = (int)ny;
  // The smallest tiles that still come to at most one workgroup per CU: a launch then lasts as long as one
  // workgroup, whose time per iteration falls with its cells. Small tiles take up to 8 iterations per
  // launch (the halo is computed several times over, on CUs that would otherwise idle). From 32 x 32 on
  // the vector units are busy and the halo is paid for: 5 iterations, 2 cells per thread.
  // us per iteration with tiles of 8 / 16 / 24 / 32: 63^2 1.57 / 1.79 / 2.34 / 3.69, 127^2 1.71 / 1.86 / 2.44 /
  // 3.81, 255^2 5.42 / 2.19 / 2.82 / 3.99, 200 x 333 5.49 / 3.64 / 2.81 / 4.00, 511^2 18.0 / 7.21 / 5.85 / 4.90,
  // 64 samples of 127^2 65 / 26.2 / 21.4 / 17.7 (two launches per iteration: 6.8 at 127^2, 12.3 at 511^2,
  // 45 for the 64).
  static const int sizes[4] = {8, 16, 24, 32}, most[4] = {8, 8, 4, 5};
  int pick = 0;
  while (pick < 3 && ((nx + sizes[pick]) / sizes[pick]) * ((ny + sizes[pick]) / sizes[pick]) * S > 256) ++pick;
  const int T = sizes[pick], KMAX = most[pick];
  A.ntx = (int)((nx + 1 + T - 1) / T);
  A.nty = (int)((ny + 1 + T - 1) / T);
  const dim3 grid((unsigned)(A.ntx * A.nty), (unsigned)S);
  const int launches = 2 * ((n + 2 * KMAX - 1) / (2 * KMAX));
  for (int l = 0, done = 0; l < launches; ++l) {
    A.k = (int)((int64_t)n * (l + 1) / launches) - done;
    done += A.k;
    const Arr* from = l & 1 ? s1 : s0;
    const Arr* to = l & 1 ? s0 : s1;
    A.Vx = from[0], A.Vy = from[1], A.Pt = from[2], A.aX = from[3], A.aY = from[4];
    A.nVx = to[0], A.nVy = to[1], A.nPt = to[2], A.naX = to[3], A.naY = to[4];
    const bool last = l == launches - 1;
#define PS_STOKES(CPT, P)                                                                                                              \
  {                                                                                                                                    \
    constexpr int nth = (P * P / CPT + 63) / 64 * 64;                                                                                  \
    if (last) hipLaunchKernelGGL((stokes2d_k<CPT, P, P, true>), grid, dim3(nth), 0, st, A);                                            \
    else hipLaunchKernelGGL((stokes2d_k<CPT, P, P, false>), grid, dim3(nth), 0, st, A);                                                \
  }
    if (pick == 0) PS_STOKES(1, 24)  // 8 + 2*8
    else if (pick < 3) PS_STOKES(1, 32)  // 16 + 2*8, 24 + 2*4
    else PS_STOKES(2, 42)  // 32 + 2*5
#undef PS_STOKES
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ps_internal_fail(PS_EHIP, std::string("ps_stokes2d_iterate: ") + hipGetErrorString(e));
  return 0;
}
