// Neural-network kernels of the Stokes warm-start U-Net (include/ps_nn.h).
//
// BF16 storage, FP32 accumulation. Activations are NHWC (channels fastest), so a 3x3
// convolution is the product of im2col(x) (rows = pixels, columns = (ky, kx, c)) with the
// weights stored [9*Cin][Cout]; its im2col operand comes out of an input patch in LDS (nn_conv3_k,
// nn_conv3_wgrad_k) or, for the forms those do not serve, is gathered from x as the general GEMM
// loads its tiles (nn_gemm_k; ps_nn_gemm reads a stored matrix with it). That runs on the gfx950 matrix cores:
// v_mfma_f32_16x16x32_bf16, lane l holding A[l%16][(l/16)*8 .. +7], B[(l/16)*8 .. +7][l%16] and
// D[(l/16)*4 + r][l%16], r = 0..3. A workgroup of four waves computes a 64x64 tile, each wave a
// 32x32 quarter as 2x2 MFMA blocks, over K steps of 32 staged through LDS.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <string>
#include <type_traits>

#include "ps_amd.h"
#include "ps_internal.h"
#include "ps_nn.h"

namespace {

typedef unsigned short bf16_t;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(short)))) short s16x8;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

__device__ __forceinline__ float bf2f(bf16_t b) { return __uint_as_float((unsigned)b << 16); }
__device__ __forceinline__ bf16_t f2bf(float f) {  // round to nearest even, NaN -> 0x7fc0
  unsigned u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)0x7fc0u;
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}

constexpr int TM = 64, TN = 64, TK = 32, LDK = TK + 8;

// C[m, n] = sum_k A(m, k) B(k, n), B(k, n) = B[k*sbk + n*sbn]; A(m, k) = A[m*sam + k*sak] (AM 0),
// or A is the 3x3 im2col of the NHWC input A (cH x cW x cC per image) without the column matrix:
// AM 1 A(m, k) = col[m][k] (m a pixel, k = tap*cC + c), AM 2 A(m, k) = col[k][m].
// blockIdx.z splits K into chunks of kchunk (a multiple of TK).
template <int EPI, int AM>
__global__ void __launch_bounds__(256) nn_gemm_k(int M, int N, int K, const bf16_t* __restrict__ A, long long sam, long long sak,
                                                 const bf16_t* __restrict__ B, long long sbk, long long sbn, void* __restrict__ C,
                                                 long long ldc, const float* __restrict__ bias, int kchunk, int cH, int cW, int cC) {
  __shared__ __attribute__((aligned(16))) bf16_t As[TM * LDK];
  __shared__ __attribute__((aligned(16))) bf16_t Bs[TN * LDK];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1;
  const long long m0 = (long long)blockIdx.x * TM, n0 = (long long)blockIdx.y * TN;
  const int kb = blockIdx.z * kchunk, ke = min(K, kb + kchunk);
  f32x4 acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Each thread moves one 8-element piece of each 64x32 tile per K step: 8 consecutive k of one
  // row when k has unit stride, else 8 consecutive rows of one k (unit stride along m / n).
  // Whole, aligned pieces travel as one 16-byte load; edge or strided pieces element by element.
  // The next step's pieces are loaded while the current tile is multiplied.
  const bool a_kfast = AM == 0 ? sak == 1 : AM == 1, b_kfast = sbk == 1;
  const int ar = a_kfast ? tid / 4 : (tid % 8) * 8, ac = a_kfast ? (tid % 4) * 8 : tid / 8;
  const int br = b_kfast ? tid / 4 : (tid % 8) * 8, bc = b_kfast ? (tid % 4) * 8 : tid / 8;
  // A piece starts at an element index that is a multiple of 8 when the stride across pieces is
  // (k0, ac, ar, m0 are all multiples of 8), so the 16-byte load is aligned
  const bool a_vec = AM == 0 ? (a_kfast ? sam : sak) % 8 == 0 && ((uintptr_t)A & 15) == 0 && (a_kfast || sam == 1)
                             : cC % 8 == 0 && ((uintptr_t)A & 15) == 0;
  // implicit im2col: the input element that column j of pixel p reads (0 outside the image)
  // Every call has p < M or p < K and j < K or j < M (all int), so the 32-bit unsigned quotients
  // are exact; only the address needs 64 bits.
  auto col_at = [&](long long p, int j, int& tap, int& c, long long& src) -> bool {
    const unsigned pu = (unsigned)p, ju = (unsigned)j;
    const unsigned tu = ju / (unsigned)cC;
    tap = (int)tu;
    c = (int)(ju - tu * (unsigned)cC);
    const unsigned t2 = pu / (unsigned)cW;
    const int xx = (int)(pu - t2 * (unsigned)cW);
    const unsigned b = t2 / (unsigned)cH;
    const int yy = (int)(t2 - b * (unsigned)cH);
    const int sy = yy + tap / 3 - 1, sx = xx + tap % 3 - 1;
    src = (((long long)b * cH + sy) * cW + sx) * cC + c;
    return sy >= 0 && sy < cH && sx >= 0 && sx < cW;
  };
  const bool b_vec = (b_kfast ? sbn : sbk) % 8 == 0 && ((uintptr_t)B & 15) == 0 && (b_kfast || sbn == 1);
  s16x8 pa, pb;
  auto fetch = [&](int k0) {
    {  // A piece
      const long long m = m0 + ar;
      const int k = k0 + ac;
      const bool full = a_kfast ? (m < M && k + 7 < ke) : (m + 7 < M && k < ke);
      if (AM == 0) {
        if (a_vec && full)
          pa = *(const s16x8*)(A + m * sam + (long long)k * sak);
        else
          for (int t = 0; t < 8; ++t) {
            const long long mm = a_kfast ? m : m + t;
            const int kk = a_kfast ? k + t : k;
            pa[t] = (mm < M && kk < ke) ? (short)A[mm * sam + (long long)kk * sak] : (short)0;
          }
      } else {
        // the piece is columns j..j+7 of pixel p (AM 1: p = m, j = k; AM 2: p = k, j = m); with cC a
        // multiple of 8 they are 8 channels of one tap, one 16-byte load (j is a multiple of 8)
        const long long p = AM == 1 ? m : (long long)k;
        const int j = AM == 1 ? k : (int)m;
        int tap, c;
        long long src;
        if (a_vec && full) {
          if (col_at(p, j, tap, c, src)) pa = *(const s16x8*)(A + src);
          else pa = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
        } else {
          for (int t = 0; t < 8; ++t) {
            const bool in = AM == 1 ? (m < M && k + t < ke) : (m + t < M && k < ke);
            pa[t] = in && col_at(p, j + t, tap, c, src) ? (short)A[src] : (short)0;
          }
        }
      }
    }
    {  // B piece
      const long long n = n0 + br;
      const int k = k0 + bc;
      const bool full = b_kfast ? (n < N && k + 7 < ke) : (n + 7 < N && k < ke);
      if (b_vec && full)
        pb = *(const s16x8*)(B + (long long)k * sbk + n * sbn);
      else
        for (int t = 0; t < 8; ++t) {
          const long long nn = b_kfast ? n : n + t;
          const int kk = b_kfast ? k + t : k;
          pb[t] = (nn < N && kk < ke) ? (short)B[(long long)kk * sbk + nn * sbn] : (short)0;
        }
    }
  };
  fetch(kb);
  for (int k0 = kb; k0 < ke; k0 += TK) {
    // tiles K-fastest in LDS
    if (a_kfast) {
      *(s16x8*)&As[ar * LDK + ac] = pa;
    } else {
      for (int t = 0; t < 8; ++t) As[(ar + t) * LDK + ac] = (bf16_t)pa[t];
    }
    if (b_kfast) {
      *(s16x8*)&Bs[br * LDK + bc] = pb;
    } else {
      for (int t = 0; t < 8; ++t) Bs[(br + t) * LDK + bc] = (bf16_t)pb[t];
    }
    __syncthreads();
    if (k0 + TK < ke) fetch(k0 + TK);
    const int i = lane & 15, kq = (lane >> 4) * 8;
    s16x8 a[2], b[2];
    for (int q = 0; q < 2; ++q) {  // rows are LDK * 2 = 80 bytes apart, kq * 2 a multiple of 16
      a[q] = *(const s16x8*)&As[(wm * 32 + q * 16 + i) * LDK + kq];
      b[q] = *(const s16x8*)&Bs[(wn * 32 + q * 16 + i) * LDK + kq];
    }
    for (int bi = 0; bi < 2; ++bi)
      for (int bj = 0; bj < 2; ++bj)
        acc[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[bi]), __builtin_bit_cast(bf16x8, b[bj]),
                                                              acc[bi][bj], 0, 0, 0);
    __syncthreads();
  }
  for (int bi = 0; bi < 2; ++bi)
    for (int bj = 0; bj < 2; ++bj)
      for (int r = 0; r < 4; ++r) {
        const long long m = m0 + wm * 32 + bi * 16 + (lane >> 4) * 4 + r;
        const long long n = n0 + wn * 32 + bj * 16 + (lane & 15);
        if (m >= M || n >= N) continue;
        float v = acc[bi][bj][r];
        if (EPI == PS_NN_EPI_BF16) {
          ((bf16_t*)C)[m * ldc + n] = f2bf(v);
        } else if (EPI == PS_NN_EPI_BF16_BIAS_RELU) {
          v += bias[n];
          ((bf16_t*)C)[m * ldc + n] = f2bf(v > 0.f ? v : 0.f);
        } else if (EPI == PS_NN_EPI_BF16_BIAS) {
          ((bf16_t*)C)[m * ldc + n] = f2bf(v + bias[n]);
        } else if (EPI == PS_NN_EPI_F32_ADD) {
          atomicAdd(&((float*)C)[m * ldc + n], v);
        } else {
          ((float*)C)[m * ldc + n] = v;
        }
      }
}

// ---- 3x3 convolution: the implicit im2col product with the input patch in LDS -------------------
//
// A workgroup owns a tile of TX columns x rows of one image's output pixels (16*MT*WM pixels) and
// NB = 16*NT*WN output channels. The input patch of that tile (one pixel of halo, every channel) is
// read from memory once into LDS, where all nine taps read it: the gather of nn_gemm_k reads it nine
// times through L2. Only the weights are then staged, KS rows of them per barrier, double buffered.
// The products take the pixels as the columns and the output channels as the rows of the MFMA, so
// that a lane ends up with 4 consecutive channels of one pixel: one 8-byte store. The weights' operand
// (8 consecutive k of one channel per lane) comes out of their [k][n] rows by the transposing LDS
// read. k runs over tap*C + c in groups of 32 in ascending order, as in nn_gemm_k, so the sums are
// bit for bit those of the stored column matrix.
// Pixel stride in LDS: an odd number of 16-byte units, so that 16 lanes reading 16 bytes of 16
// neighbouring pixels touch distinct banks.
// With C below 8 (VEC false) the k of one 16-byte piece cross taps: the lane collects its 8 values
// one by one from the patch.
constexpr int KS = 64;

__device__ __forceinline__ unsigned fdiv(unsigned e, unsigned d, unsigned magic) { return d == 1u ? e : __umulhi(e, magic); }

__device__ __forceinline__ s16x4 lds_tr(const bf16_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
}
__device__ __forceinline__ s16x8 cat8(s16x4 a, s16x4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }
__device__ __forceinline__ f32x4 mfma(s16x8 a, s16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// f2bf of 4 values, by the rounding instruction (which keeps a NaN's payload: NaNs become 0x7fc00000 first)
__device__ __forceinline__ s16x4 f2bf4(f32x4 v) {
  typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = v[r] == v[r] ? v[r] : __uint_as_float(0x7fc00000u);
  return __builtin_bit_cast(s16x4, __builtin_convertvector(v, bf16x4));
}

// MODE: 0 C below 8, 1 C a multiple of 8, 2 C a multiple of 32 (a group of 32 k stays in one tap, whose
// place in the patch is then the same for all lanes)
template <int EPI, int MT, int NT, int WM, int WN, int MODE>
__global__ void __launch_bounds__(64 * WM * WN) nn_conv3_k(const bf16_t* __restrict__ x, int H, int W, int C, const bf16_t* __restrict__ B,
                                                           long long sbk, long long sbn, int N, bf16_t* __restrict__ Y, int ldc,
                                                           const float* __restrict__ bias, int lgTX, int tilesx, int tilesy, unsigned cmagic,
                                                           unsigned pmagic) {
  constexpr bool VEC = MODE != 0;
  constexpr int NTH = 64 * WM * WN, NB = 16 * NT * WN, LDB = NB + 8;
  // weight stages in flight ahead of the one in LDS (even: stage s goes through LDS buffer s & 1): 4 for the
  // tiles of the long sums, where one workgroup is on a CU and little hides a miss (256 -> 256 at 64^2 18.9
  // -> 17.8 us, 8 x 32^2 384 -> 128 27.0 -> 25.5); 256 x 32, two workgroups on a CU, is better off with 2
  // (64 -> 64 at 256^2 12.4 us, 12.7 with 4)
  constexpr int KD = MODE == 2 && !(MT == 2 && NT == 2 && WM == 8) ? 4 : 2;
  constexpr int PIECES = KS * NB / 8, PB = (PIECES + NTH - 1) / NTH;  // 16-byte pieces of a weight stage, and per thread
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
  bf16_t* const Bs = lds;
  bf16_t* const xs = lds + 2 * KS * LDB;
  const int K = 9 * C, TX = 1 << lgTX, PW = TX + 2, rows = (16 * MT * WM) >> lgTX;
  const int ps = VEC ? ((C >> 3) | 1) * 8 : C;  // LDS elements per patch pixel
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 4, li = lane & 15;
  const int wm = WN == 1 ? w : w / WN, wn = WN == 1 ? 0 : w % WN;
  int t = blockIdx.x;
  const int tx0 = (t % tilesx) << lgTX;
  t /= tilesx;
  const int ty0 = (t % tilesy) * rows, img = t / tilesy;
  const int n0 = blockIdx.y * NB;

  // weights: piece j of this thread holds columns bn.. of row bk + s*KS in stage s
  s16x8 pb[KD][PB];
  const bf16_t* bptr[PB];
  bool bfull[PB];
  int bk[PB], bn[PB], bl[PB];
#pragma unroll
  for (int j = 0; j < PB; ++j) {
    const int q = tid + NTH * j;
    bk[j] = PIECES % NTH == 0 || q < PIECES ? q / (NB / 8) : 1 << 30;
    bn[j] = n0 + (q % (NB / 8)) * 8;
    bl[j] = (q / (NB / 8)) * LDB + (q % (NB / 8)) * 8;
    bptr[j] = B + (long long)(q / (NB / 8)) * sbk + (long long)bn[j] * sbn;
    bfull[j] = sbn == 1 && sbk % 8 == 0 && ((uintptr_t)B & 15) == 0 && bn[j] + 7 < N;
  }
  auto fetch_b = [&](s16x8 (&v)[PB], int k0) {
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      v[j] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
      if (k0 + bk[j] < K) {
        const bf16_t* const p = bptr[j] + (long long)k0 * sbk;
        if (bfull[j]) {
          v[j] = *(const s16x8*)p;
        } else {
          for (int e = 0; e < 8; ++e)
            if (bn[j] + e < N) v[j][e] = (short)p[e * sbn];
        }
      }
    }
  };
  auto store_b = [&](const s16x8 (&v)[PB], int buf) {
#pragma unroll
    for (int j = 0; j < PB; ++j)
      if (PIECES % NTH == 0 || tid + NTH * j < PIECES) *(s16x8*)&Bs[buf * KS * LDB + bl[j]] = v[j];
  };
#pragma unroll
  for (int d = 0; d < KD; ++d) fetch_b(pb[d], d * KS);
  {  // the patch, PU pieces per thread in flight: rows + 2 by TX + 2 pixels, zero outside the image
    constexpr int PU = 4;
    const unsigned cp = VEC ? (unsigned)C >> 3 : (unsigned)C, total = (unsigned)((rows + 2) * PW) * cp;
    const char* const xi = (const char*)(x + (long long)img * H * W * C);  // the launch checks that an image is below 4 GB
    for (unsigned e0 = tid; e0 < total; e0 += PU * NTH) {
      s16x8 v[PU];
      unsigned at[PU];
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        const unsigned e = e0 + NTH * u, p = fdiv(e, cp, cmagic), c = e - p * cp, py = fdiv(p, (unsigned)PW, pmagic);
        const int yy = ty0 + (int)py - 1, xx = tx0 + (int)(p - py * PW) - 1;
        at[u] = p * ps + (VEC ? c * 8 : c);
        v[u] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
        if (e < total && (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W) {
          const char* const src = xi + (size_t)(((unsigned)yy * (unsigned)W + (unsigned)xx) * (unsigned)(2 * C) + c * (VEC ? 16u : 2u));
          if (VEC) v[u] = *(const s16x8*)src;
          else v[u][0] = *(const short*)src;
        }
      }
#pragma unroll
      for (int u = 0; u < PU; ++u)
        if (e0 + NTH * u < total) {
          if (VEC) *(s16x8*)&xs[at[u]] = v[u];
          else xs[at[u]] = (bf16_t)v[u][0];
        }
    }
  }
  store_b(pb[0], 0);
  fetch_b(pb[0], KD * KS);
  int px[MT];  // the patch element where the window of this lane's pixel of M tile i starts
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int q = (wm * MT + i) * 16 + li;
    px[i] = ((q >> lgTX) * PW + (q & (TX - 1))) * ps + (MODE == 2 ? 8 * g : 0);
  }
  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 bv[NT];
  if (EPI != PS_NN_EPI_BF16) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + (wn * NT + j) * 16 + 4 * g + r;
        bv[j][r] = n < N ? bias[n] : 0.f;
      }
  }
  const bf16_t* const bp0 = &Bs[(8 * g + (li >> 2)) * LDB + wn * NT * 16 + 4 * (li & 3)];
  int tap = 0, c0 = 0;  // MODE 2: tap and first channel of the group
  __syncthreads();
  for (int s0 = 0; s0 * KS < K; s0 += KD) {
#pragma unroll
    for (int d = 0; d < KD; ++d) {
      const int s = s0 + d;
      if (s * KS >= K) break;
#pragma unroll
      for (int kk = 0; kk < KS; kk += 32) {
        const int k0 = s * KS + kk;
        if (k0 < K) {
          s16x8 a[NT], b[MT];
          const bf16_t* const bp = bp0 + ((d & 1) * KS + kk) * LDB;
#pragma unroll
          for (int j = 0; j < NT; ++j) a[j] = cat8(lds_tr(bp + 16 * j), lds_tr(bp + 16 * j + 4 * LDB));
          if (MODE == 2) {
            const int ky = (tap * 11) >> 5, off = (ky * PW + (tap - 3 * ky)) * ps + c0;
#pragma unroll
            for (int i = 0; i < MT; ++i) b[i] = *(const s16x8*)&xs[px[i] + off];
            c0 += 32;
            if (c0 == C) {
              c0 = 0;
              ++tap;
            }
          } else if (MODE == 1) {
            const unsigned k = k0 + 8 * g, tp = fdiv(k >> 3, (unsigned)C >> 3, cmagic), ky = (tp * 11u) >> 5;
            const int off = (int)((ky * PW + (tp - 3 * ky)) * ps + (k - tp * C));
            if (k0 + 32 <= K) {
#pragma unroll
              for (int i = 0; i < MT; ++i) b[i] = *(const s16x8*)&xs[px[i] + off];
            } else {  // the last group of a K that is no multiple of 32: zeros behind it
#pragma unroll
              for (int i = 0; i < MT; ++i) {
                b[i] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
                if (k < (unsigned)K) b[i] = *(const s16x8*)&xs[px[i] + off];
              }
            }
          } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const unsigned k = k0 + 8 * g + e, tp = fdiv(k, (unsigned)C, cmagic), ky = (tp * 11u) >> 5;
              const int off = (int)((ky * PW + (tp - 3 * ky)) * ps + (k - tp * C));
              const bool in = k < (unsigned)K;
#pragma unroll
              for (int i = 0; i < MT; ++i) b[i][e] = in ? (short)xs[px[i] + off] : (short)0;
            }
          }
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = mfma(a[j], b[i], acc[i][j]);
        }
      }
      if ((s + 1) * KS < K) {
        // stage s + 1 goes to the buffer that stage s - 1 was read from before the last barrier
        store_b(pb[(d + 1) % KD], (d + 1) & 1);
        fetch_b(pb[(d + 1) % KD], (s + 1 + KD) * KS);
        __syncthreads();
      }
    }
  }
  const bool c_vec = N % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)Y & 7) == 0;
  bf16_t* const yi = Y + (long long)img * H * W * ldc;
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int q = (wm * MT + i) * 16 + li, yy = ty0 + (q >> lgTX), xx = tx0 + (q & (TX - 1));
    if (yy >= H || xx >= W) continue;
    bf16_t* const yp = yi + (size_t)(((unsigned)yy * (unsigned)W + (unsigned)xx) * (unsigned)ldc);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = n0 + (wn * NT + j) * 16 + 4 * g;
      f32x4 v = acc[i][j];
      if (EPI != PS_NN_EPI_BF16) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[r] += bv[j][r];
          if (EPI == PS_NN_EPI_BF16_BIAS_RELU) v[r] = v[r] > 0.f ? v[r] : 0.f;
        }
      }
      const s16x4 o = f2bf4(v);
      if (c_vec) {
        if (n < N) *(s16x4*)(yp + n) = o;
      } else {
        for (int r = 0; r < 4; ++r)
          if (n + r < N) yp[n + r] = (bf16_t)o[r];
      }
    }
  }
}

// ---- weight gradient of a 3x3 convolution: gw[tap*C + c][n] += sum over pixels x(pixel + tap, c) dy(pixel, n)
//
// A workgroup sums a share of the pixel tiles (256 pixels: TX columns wide) for 32 input channels x 32
// output channels x all nine taps: the patch of x and the tile of dy are read from memory once and
// held in LDS as [pixel][channel], the next tile's loads in flight meanwhile. Both MFMA operands need
// 8 consecutive pixels of one channel per lane, which the transposing LDS read takes out of
// [pixel][channel] at any shift. Wavefront w of each half multiplies every fourth group of 32 pixels by
// 16 of the input channels into its own 9 x 2 accumulators (all 32 in one wavefront spilled); they
// are summed in LDS and added to gw with one atomic per element and workgroup. The general product read x nine times, split K over hundreds of
// workgroups of one 64 x 64 tile each, and spent 32 of its 64 columns on padding.
constexpr int WGS = 40;  // LDS elements per pixel: 32 channels, 16 bytes of padding against bank conflicts

template <bool VX, bool VD>  // rows of x, of dy are whole aligned 16-byte pieces
__global__ void __launch_bounds__(512, 2) nn_conv3_wgrad_k(const bf16_t* __restrict__ x, int H, int W, int C, const bf16_t* __restrict__ dy,
                                                           long long sbk, int N, float* __restrict__ gw, long long ldc, int lgTX, int tilesx,
                                                           int tilesy, int ntiles, unsigned pmagic) {
  __shared__ __attribute__((aligned(16))) bf16_t lds[(340 + 256) * WGS];
  constexpr int RS = 36;  // row stride of the FP32 sums [4 wavefronts][2 taps][32][RS]
  static_assert(4 * 2 * 32 * RS * 4 <= (int)sizeof(lds), "the sums reuse the tiles' memory");
  bf16_t* const xs = lds;
  bf16_t* const ds = lds + 340 * WGS;
  const int TX = 1 << lgTX, PW = TX + 2, rows = 256 >> lgTX, npx = (rows + 2) * PW;  // at most 340 patch pixels
  const int tid = threadIdx.x, lane = tid & 63, w = (tid >> 6) & 3, ct = tid >> 8, g = lane >> 4, li = lane & 15;
  const int c0 = blockIdx.x * 32, n0 = blockIdx.y * 32;
  s16x8 rx[3], rd[2];
  auto load = [&](int t) {
    const int tx0 = (t % tilesx) << lgTX, t2 = t / tilesx, ty0 = (t2 % tilesy) * rows, img = t2 / tilesy;
    const long long pb = (long long)img * H * W;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const unsigned e = tid + 512 * j, p = e >> 2, py = __umulhi(p, pmagic);
      const int yy = ty0 + (int)py - 1, xx = tx0 + (int)(p - py * PW) - 1, c = c0 + 8 * (int)(e & 3);
      rx[j] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
      if (p < (unsigned)npx && (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W) {
        const bf16_t* const src = x + (pb + (long long)yy * W + xx) * C + c;
        if (VX) {
          if (c < C) rx[j] = *(const s16x8*)src;
        } else {
          for (int i = 0; i < 8; ++i)
            if (c + i < C) rx[j][i] = (short)src[i];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = tid + 512 * j, p = e >> 2, yy = ty0 + (p >> lgTX), xx = tx0 + (p & (TX - 1)), n = n0 + 8 * (e & 3);
      rd[j] = s16x8{0, 0, 0, 0, 0, 0, 0, 0};
      if (yy < H && xx < W) {
        const bf16_t* const src = dy + (pb + (long long)yy * W + xx) * sbk + n;
        if (VD) {
          if (n < N) rd[j] = *(const s16x8*)src;
        } else {
          for (int i = 0; i < 8; ++i)
            if (n + i < N) rd[j][i] = (short)src[i];
        }
      }
    }
  };
  f32x4 acc[9][2];
#pragma unroll
  for (int a = 0; a < 9; ++a)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[a][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  int t = blockIdx.z;
  load(t);
  while (t < ntiles) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int e = tid + 512 * j;
      if ((e >> 2) < npx) *(s16x8*)&xs[(e >> 2) * WGS + 8 * (e & 3)] = rx[j];
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = tid + 512 * j;
      *(s16x8*)&ds[(e >> 2) * WGS + 8 * (e & 3)] = rd[j];
    }
    __syncthreads();
    const int tx0 = (t % tilesx) << lgTX, ty0 = ((t / tilesx) % tilesy) * rows;
    t += gridDim.z;
    if (t < ntiles) load(t);
    auto products = [&](auto masked) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int q0 = (w + 4 * h) * 32 + 8 * g, q = q0 + (li >> 2), row = q >> lgTX, col = q & (TX - 1);
        s16x8 b[2], keep;
#pragma unroll
        for (int j = 0; j < 2; ++j)
          b[j] = cat8(lds_tr(&ds[q * WGS + 16 * j + 4 * (li & 3)]), lds_tr(&ds[(q + 4) * WGS + 16 * j + 4 * (li & 3)]));
        if (masked) {
          const int left = ty0 + (q0 >> lgTX) < H ? W - tx0 - (q0 & (TX - 1)) : 0;
#pragma unroll
          for (int i = 0; i < 8; ++i) keep[i] = i < left ? (short)-1 : (short)0;
        }
        const bf16_t* const xp = &xs[(row * PW + col) * WGS + 16 * ct + 4 * (li & 3)];
#pragma unroll
        for (int a = 0; a < 9; ++a) {
          const bf16_t* const xa = xp + ((a / 3) * PW + a % 3) * WGS;
          s16x8 v = cat8(lds_tr(xa), lds_tr(xa + 4 * WGS));
          if (masked) v &= keep;
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[a][j] = mfma(v, b[j], acc[a][j]);
        }
      }
    };
    // pixels outside the image take no part (an infinite x there would make a NaN of its zero dy)
    if (tx0 + TX > W || ty0 + rows > H) products(std::true_type{});
    else products(std::false_type{});
    __syncthreads();
  }
  // the four wavefronts' sums meet in LDS, two taps at a time (LDS atomics took 60 us here, one
  // wavefront after the other 25)
  float* const red = (float*)lds;
#pragma unroll
  for (int a0 = 0; a0 < 9; a0 += 2) {
#pragma unroll
    for (int a = a0; a < a0 + 2 && a < 9; ++a)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[((w * 2 + a - a0) * 32 + 16 * ct + 4 * g + r) * RS + 16 * j + li] = acc[a][j][r];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int e = tid + 512 * k, n = e & 31, c = (e >> 5) & 31, a = e >> 10;
      if (a0 + a < 9 && c0 + c < C && n0 + n < N) {
        const float* const p = &red[(a * 32 + c) * RS + n];
        unsafeAtomicAdd(&gw[(long long)((a0 + a) * C + c0 + c) * ldc + n0 + n], (p[0] + p[2 * 32 * RS]) + (p[4 * 32 * RS] + p[6 * 32 * RS]));
      }
    }
    __syncthreads();
  }
}

unsigned grid_for(long long n) { return (unsigned)std::min<long long>((n + 255) / 256, 1 << 20); }

#define GS_LOOP(e, n) for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < (n); e += (long long)gridDim.x * 256)

__global__ void __launch_bounds__(256) nn_im2col_k(const bf16_t* __restrict__ x, int B, int H, int W, int C, bf16_t* __restrict__ col) {
  const long long n = (long long)B * H * W * 9 * C;
  GS_LOOP(e, n) {
    const int c = (int)(e % C);
    const long long t = e / C;
    const int kk = (int)(t % 9);
    const long long p = t / 9;
    const int xx = (int)(p % W);
    const long long t2 = p / W;
    const int yy = (int)(t2 % H), b = (int)(t2 / H);
    const int sy = yy + kk / 3 - 1, sx = xx + kk % 3 - 1;
    col[e] = (sy >= 0 && sy < H && sx >= 0 && sx < W) ? x[(((long long)b * H + sy) * W + sx) * C + c] : (bf16_t)0;
  }
}

// dx[b, y, x, c] = sum over the 3x3 taps of the columns that read (b, y, x, c)
__global__ void __launch_bounds__(256) nn_col2im_k(const bf16_t* __restrict__ dcol, int B, int H, int W, int C, bf16_t* __restrict__ dx) {
  const long long n = (long long)B * H * W * C;
  GS_LOOP(e, n) {
    const int c = (int)(e % C);
    const long long p = e / C;
    const int xx = (int)(p % W);
    const long long t2 = p / W;
    const int yy = (int)(t2 % H), b = (int)(t2 / H);
    float s = 0.f;
    for (int kk = 0; kk < 9; ++kk) {
      const int oy = yy - (kk / 3 - 1), ox = xx - (kk % 3 - 1);  // output pixel whose tap kk reads (yy, xx)
      if (oy < 0 || oy >= H || ox < 0 || ox >= W) continue;
      s += bf2f(dcol[((((long long)b * H + oy) * W + ox) * 9 + kk) * C + c]);
    }
    dx[e] = f2bf(s);
  }
}

// The data movement of the network between its products: V channels (8: 16 bytes, where the channel
// counts and the pointers allow it) per thread. One element per thread was bound by its 64-bit
// index quotients, not by memory: up2 of 1 x 256^2 x 64 took 57.9 us (0.72 TB/s), 8 channels a
// thread 7.1 (5.9 TB/s).
template <int V>
struct Piece {
  bf16_t v[V];
};
template <>
struct __attribute__((aligned(16))) Piece<8> {
  bf16_t v[8];
};

// Low-resolution piece e of (B, H, W, C) and the four pieces of its 2x2 pixels in (B, 2H, 2W, C):
// OP 0 average pooling (four in, one out), 1 its adjoint, 2 nearest upsampling (one in, four out),
// 3 its adjoint. blockIdx.y strides over the B*H rows, x over the pieces of a row.
template <int OP, int V>
__global__ void __launch_bounds__(256) nn_quad_k(const bf16_t* __restrict__ in, long long rows, int W, int C, bf16_t* __restrict__ out) {
  const unsigned cp = (unsigned)C / V;  // pieces of a pixel
  const long long rp = (long long)W * cp;  // and of a low-resolution row
  const Piece<V>* const src = (const Piece<V>*)in;
  Piece<V>* const dst = (Piece<V>*)out;
  GS_LOOP(e, rp) {
    const long long xx = rp <= 0xffffffffLL ? (long long)((unsigned)e / cp) : e / cp, c = e - xx * cp;
    for (long long r = blockIdx.y; r < rows; r += gridDim.y) {
      const long long lo = r * rp + e, hi = 4 * r * rp + 2 * xx * cp + c;  // rows 2r and 2r + 1 hold 2*rp pieces each
      const long long h[4] = {hi, hi + cp, hi + 2 * rp, hi + 2 * rp + cp};
      if (OP == 0 || OP == 3) {
        const Piece<V> a = src[h[0]], b = src[h[1]], d = src[h[2]], f = src[h[3]];
        Piece<V> o;
#pragma unroll
        for (int i = 0; i < V; ++i) {
          const float t = (bf2f(a.v[i]) + bf2f(b.v[i])) + (bf2f(d.v[i]) + bf2f(f.v[i]));
          o.v[i] = f2bf(OP == 0 ? 0.25f * t : t);
        }
        dst[lo] = o;
      } else {
        Piece<V> o = src[lo];
        if (OP == 1) {
#pragma unroll
          for (int i = 0; i < V; ++i) o.v[i] = f2bf(0.25f * bf2f(o.v[i]));
        }
        for (int i = 0; i < 4; ++i) dst[h[i]] = o;
      }
    }
  }
}

// y[p] = (a[p], b[p]) (SPLIT false) or its adjoint (a[p], b[p]) = y[p]; pa, pb: pieces per pixel. I: 32 bits
// where all indices fit (1 + 256 channels at 64 x 16^2, single elements: 11.4 us with both widths in one
// kernel, 6.4 so)
template <int V, bool SPLIT, class I>
__global__ void __launch_bounds__(256) nn_cat_k(bf16_t* __restrict__ a, unsigned pa, bf16_t* __restrict__ b, unsigned pb, I n, bf16_t* __restrict__ y) {
  const unsigned pc = pa + pb;
#pragma clang loop unroll(disable) vectorize(disable) interleave(disable)
  for (I e = (I)blockIdx.x * 256 + threadIdx.x; e < n; e += (I)gridDim.x * 256) {
    const I p = e / pc;
    const unsigned c = (unsigned)(e - p * pc);
    Piece<V>* const o = c < pa ? (Piece<V>*)a + (p * pa + c) : (Piece<V>*)b + (p * pb + (c - pa));
    if (SPLIT) *o = ((const Piece<V>*)y)[e];
    else ((Piece<V>*)y)[e] = *o;
  }
}

template <int V>
__global__ void __launch_bounds__(256) nn_relu_bwd_k(bf16_t* __restrict__ dy, const bf16_t* __restrict__ y, long long n) {
  GS_LOOP(e, n) {
    const Piece<V> a = ((const Piece<V>*)y)[e];
    Piece<V> d = ((Piece<V>*)dy)[e];
#pragma unroll
    for (int i = 0; i < V; ++i)
      if (!(bf2f(a.v[i]) > 0.f)) d.v[i] = 0;
    ((Piece<V>*)dy)[e] = d;
  }
}

// db[n] += sum over rows of dy[m, n] (FP32). Thread t of the T = (256 / units) * units that work sums
// unit t % units (V channels) of every (T / units)-th row of the block's chunk; the partial sums of a
// unit meet in LDS and go to db in one atomic per channel and block. (One thread per channel, as a
// serial loop over 256 rows, took 24 to 60 us for the layers of a
// training step of 8 x 128^2; this one 4.7 to 8.3.)
template <int V>
__global__ void __launch_bounds__(256) nn_bias_grad_k(const bf16_t* __restrict__ dy, long long M, int N, float* __restrict__ db, int chunk) {
  __shared__ float part[256 * V];
  const int units = N / V, u0 = blockIdx.y * 256, nu = min(256, units - u0), groups = 256 / nu, T = groups * nu;
  const int t = threadIdx.x, u = t % nu, grp = t / nu;
  const long long r0 = (long long)blockIdx.x * chunk, r1 = min(M, r0 + chunk);
  float s[V];
#pragma unroll
  for (int i = 0; i < V; ++i) s[i] = 0.f;
  if (t < T) {
#pragma unroll 4
    for (long long m = r0 + grp; m < r1; m += groups) {
      const Piece<V> d = ((const Piece<V>*)dy)[m * units + u0 + u];
#pragma unroll
      for (int i = 0; i < V; ++i) s[i] += bf2f(d.v[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < V; ++i) part[t * V + i] = s[i];
  __syncthreads();
  for (int c = t; c < nu * V; c += 256) {
    float v = 0.f;
    for (int k = 0; k < groups; ++k) v += part[k * nu * V + c];
    atomicAdd(&db[u0 * V + c], v);
  }
}

// ---- products with a thin side (the 1x1 head: 3 output channels). A 64 x 64 MFMA tile would be padding
// for 61 of its 64 columns or 29 of its 32 k; these read each operand once and are bound by that
// (8 x 128^2 x 32 channels: forward 12.3 -> 5.4 us, data gradient 12.8 -> 4.8, weight gradient 63 -> 14.7).
constexpr int THIN = 4, THIN_K = 512;

// C[m, :] = epi(A[m, :] B), N <= THIN: one row per thread, rows of A contiguous 16-byte pieces
template <int EPI>
__global__ void __launch_bounds__(256) nn_thin_n_k(long long M, int N, int K, const bf16_t* __restrict__ A, long long sam, const bf16_t* __restrict__ B,
                                                   long long sbk, long long sbn, bf16_t* __restrict__ C, long long ldc, const float* __restrict__ bias) {
  __shared__ f32x4 b[THIN_K];
  for (int e = threadIdx.x; e < K; e += 256)
    for (int n = 0; n < THIN; ++n) b[e][n] = n < N ? bf2f(B[e * sbk + n * sbn]) : 0.f;
  __syncthreads();
  const long long m = (long long)blockIdx.x * 256 + threadIdx.x;
  if (m >= M) return;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < K; k += 8) {
    const Piece<8> a = *(const Piece<8>*)(A + m * sam + k);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float v = bf2f(a.v[i]);
      for (int n = 0; n < THIN; ++n) acc[n] = fmaf(v, b[k + i][n], acc[n]);
    }
  }
  for (int n = 0; n < THIN; ++n)
    if (n < N) {
      float v = acc[n];
      if (EPI != PS_NN_EPI_BF16) v += bias[n];
      if (EPI == PS_NN_EPI_BF16_BIAS_RELU) v = v > 0.f ? v : 0.f;
      C[m * ldc + n] = f2bf(v);
    }
}

// C[m, n] = sum of K <= THIN products, N in pieces of 8: one piece per thread
__global__ void __launch_bounds__(256) nn_thin_k_k(long long M, int N, int K, const bf16_t* __restrict__ A, long long sam, long long sak,
                                                   const bf16_t* __restrict__ B, long long sbk, long long sbn, bf16_t* __restrict__ C, long long ldc) {
  __shared__ float b[THIN * THIN_K];
  for (int e = threadIdx.x; e < K * N; e += 256) b[e] = bf2f(B[(e / N) * sbk + (e % N) * sbn]);
  __syncthreads();
  const unsigned np = (unsigned)N / 8;
  GS_LOOP(e, M * np) {
    const long long m = M * np <= 0xffffffffLL ? (long long)((unsigned)e / np) : e / np;
    const int n = (int)(e - m * np) * 8;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < K; ++k) {
      const float a = bf2f(A[m * sam + k * sak]);
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i] = fmaf(a, b[k * N + n + i], acc[i]);
    }
    Piece<8> o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o.v[i] = f2bf(acc[i]);
    *(Piece<8>*)(C + m * ldc + n) = o;
  }
}

// C[m, n] += sum over k of A[k][m] B[k][n] (FP32), N <= THIN, M in pieces of 8 (at most 256): each thread
// sums one piece over every (256 / pieces)-th row of the workgroup's chunk
__global__ void __launch_bounds__(256) nn_thin_grad_k(int M, int N, long long K, const bf16_t* __restrict__ A, long long sak, const bf16_t* __restrict__ B,
                                                      long long sbk, float* __restrict__ C, long long ldc, long long chunk) {
  __shared__ float part[256 * 8 * THIN];
  const int units = M / 8, groups = 256 / units, t = threadIdx.x, u = t % units, grp = t / units;
  const long long k0 = (long long)blockIdx.x * chunk, k1 = min(K, k0 + chunk);
  float acc[8][THIN];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int n = 0; n < THIN; ++n) acc[i][n] = 0.f;
  if (grp < groups) {
#pragma unroll 4
    for (long long k = k0 + grp; k < k1; k += groups) {
      const Piece<8> a = *(const Piece<8>*)(A + k * sak + 8 * u);
      float b[THIN];
#pragma unroll
      for (int n = 0; n < THIN; ++n) b[n] = n < N ? bf2f(B[k * sbk + n]) : 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int n = 0; n < THIN; ++n) acc[i][n] = fmaf(bf2f(a.v[i]), b[n], acc[i][n]);
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int n = 0; n < THIN; ++n) part[(i * THIN + n) * 256 + t] = acc[i][n];
  __syncthreads();
  for (int e = t; e < M * THIN; e += 256) {
    const int m = e / THIN, n = e % THIN;
    if (n >= N) continue;
    float v = 0.f;
    for (int k = 0; k < groups; ++k) v += part[((m & 7) * THIN + n) * 256 + k * units + (m >> 3)];
    unsafeAtomicAdd(&C[(long long)m * ldc + n], v);
  }
}

// loss += scale * mask * (pred - target)^2 ; dpred = 2 * scale * mask * (pred - target)
__global__ void __launch_bounds__(256) nn_mse_k(const bf16_t* __restrict__ pred, const float* __restrict__ target, const float* __restrict__ mask,
                                                long long n, float scale, bf16_t* __restrict__ dpred, float* __restrict__ loss) {
  __shared__ float part[256];
  float s = 0.f;
  GS_LOOP(e, n) {
    const float d = bf2f(pred[e]) - target[e];
    const float mk = mask ? mask[e] : 1.f;
    s += scale * mk * d * d;
    dpred[e] = f2bf(2.f * scale * mk * d);
  }
  part[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(loss, part[0]);
}

__global__ void __launch_bounds__(256) nn_adam_k(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                                                 long long n, float lr, float b1, float b2, float eps, float c1, float c2,
                                                 bf16_t* __restrict__ w16) {
  GS_LOOP(e, n) {
    const float ge = g[e];
    const float me = b1 * m[e] + (1.f - b1) * ge;
    const float ve = b2 * v[e] + (1.f - b2) * ge * ge;
    m[e] = me;
    v[e] = ve;
    const float we = w[e] - lr * (me * c1) / (sqrtf(ve * c2) + eps);
    w[e] = we;
    if (w16) w16[e] = f2bf(we);
  }
}

__global__ void __launch_bounds__(256) nn_f32_to_bf16_k(const float* __restrict__ x, long long n, bf16_t* __restrict__ y) {
  GS_LOOP(e, n) y[e] = f2bf(x[e]);
}
__global__ void __launch_bounds__(256) nn_bf16_to_f32_k(const bf16_t* __restrict__ x, long long n, float* __restrict__ y) {
  GS_LOOP(e, n) y[e] = bf2f(x[e]);
}
__global__ void __launch_bounds__(256) nn_fill_f32_k(float* __restrict__ x, long long n, float v) {
  GS_LOOP(e, n) x[e] = v;
}
// the weights of a 3x3 convolution's data gradient: wf[(t*Cout + co)*Cin + ci] = w[((8-t)*Cin + ci)*Cout + co]
// (taps reversed, each tap's Cin x Cout block transposed), so that dx = im2col(dy) . wf
__global__ void __launch_bounds__(256) nn_conv_flip_k(const bf16_t* __restrict__ w, int Cin, int Cout, bf16_t* __restrict__ wf) {
  GS_LOOP(e, 9LL * Cin * Cout) {
    const int ci = (int)(e % Cin);
    const long long r = e / Cin;
    const int co = (int)(r % Cout), t = (int)(r / Cout);
    wf[e] = w[((long long)(8 - t) * Cin + ci) * Cout + co];
  }
}
template <int V>
__global__ void __launch_bounds__(256) nn_add_bf16_k(bf16_t* __restrict__ y, const bf16_t* __restrict__ x, long long n) {
  GS_LOOP(e, n) {
    Piece<V> a = ((Piece<V>*)y)[e];
    const Piece<V> b = ((const Piece<V>*)x)[e];
#pragma unroll
    for (int i = 0; i < V; ++i) a.v[i] = f2bf(bf2f(a.v[i]) + bf2f(b.v[i]));
    ((Piece<V>*)y)[e] = a;
  }
}

int launched(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return ps_internal_fail(PS_EHIP, std::string(what) + ": " + hipGetErrorString(e));
  return 0;
}

}  // namespace

#define NN_BEGIN                                   \
  if (int r_ = ps_internal_require_init()) return r_; \
  hipStream_t st = ps_internal_stream(stream);

namespace {

template <int AM>
int gemm_launch(int M, int N, int K, const void* A, int64_t sam, int64_t sak, const void* B, int64_t sbk, int64_t sbn, void* C, int64_t ldc,
                const float* bias, int epi, int splitk, hipStream_t st, int cH, int cW, int cC) {
  if (M < 0 || N < 0 || K < 0 || splitk < 1) return ps_internal_fail(PS_EARGUMENT, "ps_nn_gemm: negative size or splitk < 1");
  if (M == 0 || N == 0) return 0;
  if ((epi == PS_NN_EPI_BF16_BIAS_RELU || epi == PS_NN_EPI_BF16_BIAS) && !bias) return ps_internal_fail(PS_EARGUMENT, "ps_nn_gemm: bias missing");
  if (splitk > 1 && epi != PS_NN_EPI_F32_ADD) return ps_internal_fail(PS_EARGUMENT, "ps_nn_gemm: split-K needs the accumulating FP32 epilogue");
  // K of a multiple of 72 may be the columns of a 3x3 im2col, whose product is that of the convolution bit for bit
  if (AM == 0 && splitk == 1 && N <= THIN && K <= THIN_K && K % 8 == 0 && K % 72 != 0 && K > 0 && sak == 1 && sam % 8 == 0 && ((uintptr_t)A & 15) == 0 && epi <= PS_NN_EPI_BF16_BIAS &&
      epi >= 0) {
    const dim3 g((unsigned)((M + 255LL) / 256));
#define NN_THIN(E) hipLaunchKernelGGL((nn_thin_n_k<E>), g, dim3(256), 0, st, (long long)M, N, K, (const bf16_t*)A, sam, (const bf16_t*)B, sbk, sbn, (bf16_t*)C, ldc, bias)
    if (epi == PS_NN_EPI_BF16) NN_THIN(PS_NN_EPI_BF16);
    else if (epi == PS_NN_EPI_BF16_BIAS) NN_THIN(PS_NN_EPI_BF16_BIAS);
    else NN_THIN(PS_NN_EPI_BF16_BIAS_RELU);
#undef NN_THIN
    return launched("ps_nn_gemm");
  }
  if (AM == 0 && splitk == 1 && K <= THIN && K > 0 && N <= THIN_K && N % 8 == 0 && ldc % 8 == 0 && ((uintptr_t)C & 15) == 0 && epi == PS_NN_EPI_BF16) {
    hipLaunchKernelGGL(nn_thin_k_k, dim3(grid_for((long long)M * (N / 8))), dim3(256), 0, st, (long long)M, N, K, (const bf16_t*)A, sam, sak, (const bf16_t*)B, sbk,
                       sbn, (bf16_t*)C, ldc);
    return launched("ps_nn_gemm");
  }
  // Not where the split already leaves the MFMA product short sums (64 rows of 600 pixels, split 64: 5.3 us
  // there, 6.3 here, split 2 12.3; 1024 of 16384, split 64: 22 and 28, split 8 69, split 512 55), nor for
  // many rows of few pixels (2048 of 4096: 14 to 66 us there, 116 here).
  if (AM == 0 && splitk > 1 && N <= THIN && M % 8 == 0 && sam == 1 && sak % 8 == 0 && ((uintptr_t)A & 15) == 0 && sbn == 1 &&
      (M <= 256 ? K > 2048 || K > 128LL * splitk : M <= 2048 && K >= 16384 && (K < 64LL * splitk || K > 1024LL * splitk))) {
    // the epilogue is the accumulating one here; about one workgroup per CU, each with 256 rows, or where
    // the pieces of a row leave fewer than 64 of them to be summed at a time, four per thread
    const long long chunk = std::max<long long>(std::min(256, 4 * (256 / (M / 8))), (K + 255LL) / 256);
    hipLaunchKernelGGL(nn_thin_grad_k, dim3((unsigned)((K + chunk - 1) / chunk)), dim3(256), 0, st, M, N, (long long)K, (const bf16_t*)A, sak, (const bf16_t*)B, sbk,
                       (float*)C, ldc, chunk);
    return launched("ps_nn_gemm");
  }
  int kchunk = (K + splitk - 1) / splitk;
  kchunk = ((kchunk + TK - 1) / TK) * TK;
  if (kchunk < TK) kchunk = TK;
  const int nz = (K + kchunk - 1) / kchunk;
  dim3 grid((unsigned)((M + TM - 1) / TM), (unsigned)((N + TN - 1) / TN), (unsigned)std::max(1, nz));
  if (grid.y > 65535 || grid.z > 65535) return ps_internal_fail(PS_EARGUMENT, "ps_nn_gemm: N or split too large");
  const bf16_t* a = (const bf16_t*)A;
  const bf16_t* b = (const bf16_t*)B;
#define NN_GEMM_CASE(E)                                                                                                        \
  case E:                                                                                                                      \
    hipLaunchKernelGGL((nn_gemm_k<E, AM>), grid, dim3(256), 0, st, M, N, K, a, sam, sak, b, sbk, sbn, C, ldc, bias, kchunk, cH, cW, cC); \
    break;
  switch (epi) {
    NN_GEMM_CASE(PS_NN_EPI_BF16)
    NN_GEMM_CASE(PS_NN_EPI_BF16_BIAS_RELU)
    NN_GEMM_CASE(PS_NN_EPI_BF16_BIAS)
    NN_GEMM_CASE(PS_NN_EPI_F32_ADD)
    NN_GEMM_CASE(PS_NN_EPI_F32)
    default: return ps_internal_fail(PS_EARGUMENT, "ps_nn_gemm: unknown epilogue");
  }
#undef NN_GEMM_CASE
  return launched("ps_nn_gemm");
}

// The 3x3 convolution with the patch in LDS (nn_conv3_k), or 1 where the general product serves:
// FP32 results and split K, 8 channels and more that are not whole aligned 16-byte pieces, and
// channel counts whose patch does not fit the LDS.
int conv3_launch(int M, int N, const bf16_t* x, int H, int W, int C, const bf16_t* B, long long sbk, long long sbn, void* Cm, long long ldc,
                 const float* bias, int epi, int splitk, hipStream_t st) {
  const bool vec = C % 8 == 0;
  if (splitk != 1 || (epi != PS_NN_EPI_BF16 && epi != PS_NN_EPI_BF16_BIAS_RELU && epi != PS_NN_EPI_BF16_BIAS)) return 1;
  if (!(vec && ((uintptr_t)x & 15) == 0) && C >= 8) return 1;
  // offsets inside one image are 32-bit
  if ((long long)H * W > 0x7fffffffLL / std::max<long long>(C, std::max<long long>(ldc, N)) || ldc < 0) return 1;
  const int mode = !vec ? 0 : C % 32 == 0 ? 2 : 1;
  const long long imgs = M / ((long long)H * W);
  auto up = [](long long a, long long b) { return (a + b - 1) / b; };
  // pixel tiles 16 columns wide, or 8 where that pads the image less
  auto shape = [&](int pix, int& lg) -> long long {
    const long long w16 = up(W, 16) * up(H, pix / 16), w8 = up(W, 8) * up(H, pix / 8);
    lg = w8 < w16 ? 3 : 4;
    return std::min(w16, w8) * imgs;
  };
  // Tile (pixels x channels, 8 wavefronts each). While the patch leaves room for two workgroups on a
  // CU, 256 x 32: the most workgroups in flight, so that one's loads run under another's products
  // (32 -> 32 at 512^2: 18.6 us; 256 x 64 with the padded channels 25.2, four wavefronts 20.4). Where
  // it does not (C = 128 and above), the patch is better read by fewer workgroups: 256 x 64, then
  // 128 x 64 (192 -> 64 at 256^2: 28.6 us against 41.1 with 256 x 32; 384 -> 128 at 128^2: 34.9
  // against 52.9 with 128 x 32). Tiles that leave CUs without a workgroup give way to smaller ones
  // (256 -> 256 at 64^2: 128 x 32 20.0 us, 128 x 64 24.8). What then bounded the small-C layers was
  // vector instructions around the products (index quotients, masks, rounding): with the patch place
  // of a group of 32 k in scalar registers (MODE 2) and the rounding instruction, 32 -> 32 at 512^2
  // runs 13.8 us, 192 -> 64 26.5, 384 -> 128 31.8.
  struct Tile { int pix, nb; };
  static const Tile tiles[4] = {{256, 64}, {128, 64}, {256, 32}, {128, 32}};
  int lg = 4, pick = -1;
  long long ntile = 0, lds = 0;
  auto fits = [&](int v) {
    const long long ps = vec ? ((C >> 3) | 1) * 8 : C;
    ntile = shape(tiles[v].pix, lg);
    lds = 2LL * (2 * KS * (tiles[v].nb + 8) + ((tiles[v].pix >> lg) + 2) * ((1 << lg) + 2) * ps);
    return lds <= 160 * 1024;
  };
  const bool two = fits(2) && lds <= 80 * 1024;
  for (int v = two ? 2 : 0; v < 4 && pick < 0; ++v)
    if (fits(v) && (v == 3 || ntile * up(N, tiles[v].nb) >= 256)) pick = v;
  if (pick < 0) return 1;
  const int pix = tiles[pick].pix, nb = tiles[pick].nb;
  if (ntile > 0x7fffffffLL || up(N, nb) > 65535) return 1;
  const int tx = 1 << lg, tilesx = (int)up(W, tx), tilesy = (int)up(H, pix / tx);
  const unsigned d = vec ? (unsigned)C >> 3 : (unsigned)C;
  const unsigned cmagic = d == 1 ? 0u : (unsigned)((0x100000000ULL + d - 1) / d), pmagic = (unsigned)((0x100000000ULL + tx + 1) / (tx + 2));
  const dim3 grid((unsigned)ntile, (unsigned)up(N, nb));
#define NN_CONV3(E, MT, NT, WM, WN, MODE)                                                                                                       \
  hipLaunchKernelGGL((nn_conv3_k<E, MT, NT, WM, WN, MODE>), grid, dim3(512), (size_t)lds, st, x, H, W, C, B, sbk, sbn, N, (bf16_t*)Cm, (int)ldc, bias, \
                     lg, tilesx, tilesy, cmagic, pmagic)
#define NN_CONV3_TILE(E, MT, NT, WM, WN)              \
  {                                                   \
    if (mode == 2) NN_CONV3(E, MT, NT, WM, WN, 2);    \
    else NN_CONV3(E, MT, NT, WM, WN, 1);              \
  }
#define NN_CONV3_CASE(E)                              \
  case E:                                             \
    if (pick == 2 && !vec) NN_CONV3(E, 2, 2, 8, 1, 0); \
    else if (!vec) NN_CONV3(E, 1, 2, 8, 1, 0);        \
    else if (pick == 0) NN_CONV3_TILE(E, 2, 4, 8, 1)  \
    else if (pick == 1) NN_CONV3_TILE(E, 2, 2, 4, 2)  \
    else if (pick == 2) NN_CONV3_TILE(E, 2, 2, 8, 1)  \
    else NN_CONV3_TILE(E, 1, 2, 8, 1)                 \
    break;
  switch (epi) {
    NN_CONV3_CASE(PS_NN_EPI_BF16)
    NN_CONV3_CASE(PS_NN_EPI_BF16_BIAS_RELU)
    NN_CONV3_CASE(PS_NN_EPI_BF16_BIAS)
  }
#undef NN_CONV3_CASE
#undef NN_CONV3_TILE
#undef NN_CONV3
  return launched("ps_nn_gemm_im2col");
}

// The weight gradient by nn_conv3_wgrad_k, or 1 where the general product serves: a single K chain
// (splitk 1) keeps its order of summation.
int wgrad_launch(int N, long long K, const bf16_t* x, int H, int W, int C, const bf16_t* dy, long long sbk, long long sbn, void* gw, long long ldc, int epi,
                 int splitk, hipStream_t st) {
  // less than one tile of pixels is all padding to this kernel: 4 x 2 x 2 pixels, 64 -> 128, 7.0 us against 4.3
  if (splitk < 2 || epi != PS_NN_EPI_F32_ADD || sbn != 1 || K < 256) return 1;
  const long long imgs = K / ((long long)H * W);
  auto up = [](long long a, long long b) { return (a + b - 1) / b; };
  // the tile width (32, 16 or 8 pixels of 256) that pads the images least
  int lg = 5;
  long long best = up(W, 32) * up(H, 8);
  for (int l : {4, 3})
    if (up(W, 1 << l) * up(H, 256 >> l) < best) best = up(W, 1 << l) * up(H, 256 >> l), lg = l;
  const int tx = 1 << lg, tilesx = (int)up(W, tx), tilesy = (int)up(H, 256 >> lg);
  const long long nt = best * imgs, gc = up(C, 32), gn = up(N, 32);
  if (nt > 0x7fffffffLL || gn > 65535) return 1;
  // A workgroup ends in 9216 atomics: about 128 workgroups of at least four tiles, 256 from 1024 tiles
  // on (8 x 128^2, 32 -> 32, 512 tiles: 15.3 us with 128 workgroups, 18.1 with 256, 28.8 with 512;
  // 96 -> 32, 1536 tiles: 27.2, 22.7, 30.6; 8 x 32^2, 384 -> 128: 32.7, 19.8, 26.1)
  const long long want = nt * gc * gn < 1024 ? 128 : 256;
  const int S = (int)std::min<long long>(std::min<long long>(nt, 65535), std::max<long long>(1, want / (gc * gn)));
  const unsigned pmagic = (unsigned)((0x100000000ULL + tx + 1) / (tx + 2));
  const dim3 grid((unsigned)gc, (unsigned)gn, (unsigned)S);
  // the first layer's few input channels come one by one, its dy in whole pieces all the same
  const bool vx = C % 8 == 0 && ((uintptr_t)x & 15) == 0, vd = N % 8 == 0 && sbk % 8 == 0 && ((uintptr_t)dy & 15) == 0;
#define NN_WGRAD(VX, VD) \
  hipLaunchKernelGGL((nn_conv3_wgrad_k<VX, VD>), grid, dim3(512), 0, st, x, H, W, C, dy, sbk, N, (float*)gw, ldc, lg, tilesx, tilesy, (int)nt, pmagic)
  if (vx && vd) NN_WGRAD(true, true);
  else if (vx) NN_WGRAD(true, false);
  else if (vd) NN_WGRAD(false, true);
  else NN_WGRAD(false, false);
#undef NN_WGRAD
  return launched("ps_nn_gemm_im2col");
}

}  // namespace

extern "C" int ps_nn_gemm(int M, int N, int K, const void* A, int64_t sam, int64_t sak, const void* B, int64_t sbk, int64_t sbn, void* C,
                          int64_t ldc, const float* bias, int epi, int splitk, void* stream) {
  NN_BEGIN
  return gemm_launch<0>(M, N, K, A, sam, sak, B, sbk, sbn, C, ldc, bias, epi, splitk, st, 1, 1, 1);
}

extern "C" int ps_nn_gemm_im2col(int transpose, int M, int N, int K, const void* x, int H, int W, int Cin, const void* B, int64_t sbk, int64_t sbn,
                                 void* C, int64_t ldc, const float* bias, int epi, int splitk, void* stream) {
  NN_BEGIN
  if (H < 1 || W < 1 || Cin < 1) return ps_internal_fail(PS_EARGUMENT, "ps_nn_gemm_im2col: H, W and C must be positive");
  const long long npix = transpose ? (long long)K : (long long)M, ncol = transpose ? (long long)M : (long long)K;
  if (ncol != 9LL * Cin || npix % ((long long)H * W) != 0)
    return ps_internal_fail(PS_EARGUMENT, "ps_nn_gemm_im2col: the im2col operand is (B*H*W) x (9*C): sizes do not match");
  if (!transpose && M > 0 && N > 0 && (epi == PS_NN_EPI_BF16 || bias)) {
    const int r = conv3_launch(M, N, (const bf16_t*)x, H, W, Cin, (const bf16_t*)B, sbk, sbn, C, ldc, bias, epi, splitk, st);
    if (r <= 0) return r;
  }
  if (transpose && M > 0 && N > 0 && K > 0) {
    const int r = wgrad_launch(N, K, (const bf16_t*)x, H, W, Cin, (const bf16_t*)B, sbk, sbn, C, ldc, epi, splitk, st);
    if (r <= 0) return r;
  }
  return transpose ? gemm_launch<2>(M, N, K, x, 0, 0, B, sbk, sbn, C, ldc, bias, epi, splitk, st, H, W, Cin)
                   : gemm_launch<1>(M, N, K, x, 0, 0, B, sbk, sbn, C, ldc, bias, epi, splitk, st, H, W, Cin);
}

// Element counts are products of the sizes: a pair of negative sizes would make a positive count
// for indices the kernels never expect, so any negative size is refused before the launch.
inline bool nn_negative(std::initializer_list<long long> v) {
  for (long long x : v)
    if (x < 0) return true;
  return false;
}
#define NN_SIZES(what, ...) \
  if (nn_negative({__VA_ARGS__})) return ps_internal_fail(PS_EARGUMENT, what ": negative size");

#define NN_ELEMENTWISE(name, n, ...)                                            \
  NN_BEGIN                                                                      \
  if ((n) <= 0) return 0;                                                       \
  hipLaunchKernelGGL(name, dim3(grid_for(n)), dim3(256), 0, st, __VA_ARGS__); \
  return launched(#name);

extern "C" int ps_nn_im2col(const void* x, int B, int H, int W, int C, void* col, void* stream) {
  NN_SIZES("ps_nn_im2col", B, H, W, C)
  NN_ELEMENTWISE(nn_im2col_k, (long long)B * H * W * 9 * C, (const bf16_t*)x, B, H, W, C, (bf16_t*)col)
}
extern "C" int ps_nn_conv_flip(const void* w, int Cin, int Cout, void* wf, void* stream) {
  NN_SIZES("ps_nn_conv_flip", Cin, Cout)
  NN_ELEMENTWISE(nn_conv_flip_k, 9LL * Cin * Cout, (const bf16_t*)w, Cin, Cout, (bf16_t*)wf)
}
extern "C" int ps_nn_col2im(const void* dcol, int B, int H, int W, int C, void* dx, void* stream) {
  NN_SIZES("ps_nn_col2im", B, H, W, C)
  NN_ELEMENTWISE(nn_col2im_k, (long long)B * H * W * C, (const bf16_t*)dcol, B, H, W, C, (bf16_t*)dx)
}
// 16-byte pieces of 8 elements: whole ones, on aligned pointers
inline bool nn_pieces(std::initializer_list<long long> counts, std::initializer_list<const void*> ptrs) {
  for (long long c : counts)
    if (c % 8) return false;
  for (const void* p : ptrs)
    if ((uintptr_t)p & 15) return false;
  return true;
}

namespace {
// rows = B*H and W of the low-resolution image
template <int OP>
int quad_launch(const char* what, const void* in, long long rows, int W, int C, void* out, hipStream_t st) {
  if (rows <= 0 || W <= 0 || C <= 0) return 0;
  const bool v = nn_pieces({C}, {in, out});
  const long long rp = (long long)W * (v ? C / 8 : C);
  const dim3 grid((unsigned)std::min<long long>((rp + 255) / 256, 1 << 16), (unsigned)std::min<long long>(rows, 32768));
  if (v) hipLaunchKernelGGL((nn_quad_k<OP, 8>), grid, dim3(256), 0, st, (const bf16_t*)in, rows, W, C, (bf16_t*)out);
  else hipLaunchKernelGGL((nn_quad_k<OP, 1>), grid, dim3(256), 0, st, (const bf16_t*)in, rows, W, C, (bf16_t*)out);
  return launched(what);
}
template <bool SPLIT>
int cat_launch(const char* what, const void* a, int Ca, const void* b, int Cb, long long P, const void* y, hipStream_t st) {
  if (P * ((long long)Ca + Cb) <= 0) return 0;
  const bool v = nn_pieces({Ca, Cb}, {a, b, y});
  const unsigned pa = v ? Ca / 8 : Ca, pb = v ? Cb / 8 : Cb;
  const long long n = P * ((long long)pa + pb);
  auto go = [&](auto k, auto m) { hipLaunchKernelGGL(k, dim3(grid_for(n)), dim3(256), 0, st, (bf16_t*)a, pa, (bf16_t*)b, pb, m, (bf16_t*)y); };
  if (n < 0xe0000000LL) {  // e passes n by less than the grid's 2^28 threads
    if (v) go(nn_cat_k<8, SPLIT, unsigned>, (unsigned)n);
    else go(nn_cat_k<1, SPLIT, unsigned>, (unsigned)n);
  } else {
    if (v) go(nn_cat_k<8, SPLIT, unsigned long long>, (unsigned long long)n);
    else go(nn_cat_k<1, SPLIT, unsigned long long>, (unsigned long long)n);
  }
  return launched(what);
}
}  // namespace

// whole pieces of 8 while n and the pointers allow it, else element by element
#define NN_PIECEWISE(kernel, n, p, q)                                                                                        \
  NN_BEGIN                                                                                                                   \
  if ((n) <= 0) return 0;                                                                                                    \
  if (nn_pieces({(long long)(n)}, {p, q}))                                                                                   \
    hipLaunchKernelGGL((kernel<8>), dim3(grid_for((n) / 8)), dim3(256), 0, st, (bf16_t*)p, (const bf16_t*)q, (long long)(n) / 8); \
  else                                                                                                                       \
    hipLaunchKernelGGL((kernel<1>), dim3(grid_for(n)), dim3(256), 0, st, (bf16_t*)p, (const bf16_t*)q, (long long)(n));      \
  return launched(#kernel);

extern "C" int ps_nn_pool2(const void* x, int B, int H, int W, int C, void* y, void* stream) {
  NN_SIZES("ps_nn_pool2", B, H, W, C)
  if ((H | W) & 1) return ps_internal_fail(PS_EARGUMENT, "ps_nn_pool2: H and W must be even");
  NN_BEGIN
  return quad_launch<0>("ps_nn_pool2", x, (long long)B * (H / 2), W / 2, C, y, st);
}
extern "C" int ps_nn_pool2_bwd(const void* dy, int B, int H, int W, int C, void* dx, void* stream) {
  NN_SIZES("ps_nn_pool2_bwd", B, H, W, C)
  if ((H | W) & 1) return ps_internal_fail(PS_EARGUMENT, "ps_nn_pool2_bwd: H and W must be even");
  NN_BEGIN
  return quad_launch<1>("ps_nn_pool2_bwd", dy, (long long)B * (H / 2), W / 2, C, dx, st);
}
extern "C" int ps_nn_up2(const void* x, int B, int H, int W, int C, void* y, void* stream) {
  NN_SIZES("ps_nn_up2", B, H, W, C)
  NN_BEGIN
  return quad_launch<2>("ps_nn_up2", x, (long long)B * H, W, C, y, st);
}
extern "C" int ps_nn_up2_bwd(const void* dy, int B, int H, int W, int C, void* dx, void* stream) {
  NN_SIZES("ps_nn_up2_bwd", B, H, W, C)
  NN_BEGIN
  return quad_launch<3>("ps_nn_up2_bwd", dy, (long long)B * H, W, C, dx, st);
}
extern "C" int ps_nn_concat(const void* a, int Ca, const void* b, int Cb, int64_t P, void* y, void* stream) {
  NN_SIZES("ps_nn_concat", Ca, Cb, P)
  NN_BEGIN
  return cat_launch<false>("ps_nn_concat", a, Ca, b, Cb, P, y, st);
}
extern "C" int ps_nn_split(const void* dy, int Ca, int Cb, int64_t P, void* da, void* db, void* stream) {
  NN_SIZES("ps_nn_split", Ca, Cb, P)
  NN_BEGIN
  return cat_launch<true>("ps_nn_split", da, Ca, db, Cb, P, dy, st);
}
extern "C" int ps_nn_relu_bwd(void* dy, const void* y, int64_t n, void* stream) { NN_PIECEWISE(nn_relu_bwd_k, n, dy, y) }
extern "C" int ps_nn_bias_grad(const void* dy, int64_t M, int N, float* db, void* stream) {
  NN_BEGIN
  if (M <= 0 || N <= 0) return 0;
  const bool v = nn_pieces({N}, {dy});
  const int units = v ? N / 8 : N;
  // about one workgroup per CU, at least 64 rows each: one atomic per channel and workgroup
  const int chunk = (int)std::min<long long>(std::max<long long>(64, (M + 255) / 256), 1 << 30);
  const dim3 grid((unsigned)((M + chunk - 1) / chunk), (unsigned)((units + 255) / 256));
  if (v) hipLaunchKernelGGL((nn_bias_grad_k<8>), grid, dim3(256), 0, st, (const bf16_t*)dy, (long long)M, N, db, chunk);
  else hipLaunchKernelGGL((nn_bias_grad_k<1>), grid, dim3(256), 0, st, (const bf16_t*)dy, (long long)M, N, db, chunk);
  return launched("ps_nn_bias_grad");
}
extern "C" int ps_nn_mse(const void* pred, const float* target, const float* mask, int64_t n, float scale, void* dpred, float* loss,
                         void* stream) {
  NN_BEGIN
  if (n <= 0) return 0;
  // every workgroup ends in one atomic on the loss: a few hundred of them at most (1536 took 22 us)
  hipLaunchKernelGGL(nn_mse_k, dim3(std::min(grid_for(n), 256u)), dim3(256), 0, st, (const bf16_t*)pred, target, mask, (long long)n, scale,
                     (bf16_t*)dpred, loss);
  return launched("ps_nn_mse");
}
extern "C" int ps_nn_adam(float* w, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2, float eps, float c1, float c2,
                          void* w16, void* stream) {
  NN_ELEMENTWISE(nn_adam_k, (long long)n, w, g, m, v, (long long)n, lr, b1, b2, eps, c1, c2, (bf16_t*)w16)
}
extern "C" int ps_nn_f32_to_bf16(const float* x, int64_t n, void* y, void* stream) {
  NN_ELEMENTWISE(nn_f32_to_bf16_k, (long long)n, x, (long long)n, (bf16_t*)y)
}
extern "C" int ps_nn_bf16_to_f32(const void* x, int64_t n, float* y, void* stream) {
  NN_ELEMENTWISE(nn_bf16_to_f32_k, (long long)n, (const bf16_t*)x, (long long)n, y)
}
extern "C" int ps_nn_fill_f32(float* x, int64_t n, float v, void* stream) { NN_ELEMENTWISE(nn_fill_f32_k, (long long)n, x, (long long)n, v) }
extern "C" int ps_nn_add_bf16(void* y, const void* x, int64_t n, void* stream) { NN_PIECEWISE(nn_add_bf16_k, n, y, x) }

extern "C" int ps_nn_alloc(int64_t bytes, void** out) {
  if (int r = ps_internal_require_init()) return r;
  if (bytes < 0) return ps_internal_fail(PS_EARGUMENT, "ps_nn_alloc: negative size");
  hipStream_t st = ps_internal_stream(nullptr);
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  hipError_t e = hipStreamIsCapturing(st, &cs);
  if (e == hipSuccess && cs != hipStreamCaptureStatusNone)
    return ps_internal_fail(PS_EARGUMENT, "ps_nn_alloc: cannot allocate while a graph is being captured on the library stream");
  void* p = nullptr;
  e = hipMalloc(&p, (size_t)std::max<int64_t>(bytes, 256));
  if (e != hipSuccess) return ps_internal_fail(e == hipErrorOutOfMemory ? PS_EOOM : PS_EHIP, std::string("hipMalloc: ") + hipGetErrorString(e));
  // cleared on the library's stream and waited for: a clear on the null stream is not ordered with the
  // library's (non-blocking) streams and could land on what they write next
  e = hipMemsetAsync(p, 0, (size_t)std::max<int64_t>(bytes, 256), st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) {
    (void)hipFree(p);
    return ps_internal_fail(PS_EHIP, std::string("ps_nn_alloc: ") + hipGetErrorString(e));
  }
  *out = p;
  return 0;
}
extern "C" int ps_nn_free(void* p) {
  if (!p) return 0;
  hipError_t e = hipFree(p);
  if (e != hipSuccess) return ps_internal_fail(PS_EHIP, std::string("hipFree: ") + hipGetErrorString(e));
  return 0;
}
extern "C" int ps_nn_h2d(void* dst, const void* src, int64_t bytes, void* stream) {
  NN_BEGIN
  hipError_t e = hipMemcpyAsync(dst, src, (size_t)bytes, hipMemcpyHostToDevice, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return ps_internal_fail(PS_EHIP, std::string("ps_nn_h2d: ") + hipGetErrorString(e));
  return 0;
}
extern "C" int ps_nn_d2h(void* dst, const void* src, int64_t bytes, void* stream) {
  NN_BEGIN
  hipError_t e = hipMemcpyAsync(dst, src, (size_t)bytes, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return ps_internal_fail(PS_EHIP, std::string("ps_nn_d2h: ") + hipGetErrorString(e));
  return 0;
}
extern "C" int ps_nn_d2d(void* dst, const void* src, int64_t bytes, void* stream) {
  NN_BEGIN
  hipError_t e = hipMemcpyAsync(dst, src, (size_t)bytes, hipMemcpyDeviceToDevice, st);
  if (e != hipSuccess) return ps_internal_fail(PS_EHIP, std::string("ps_nn_d2d: ") + hipGetErrorString(e));
  return 0;
}
