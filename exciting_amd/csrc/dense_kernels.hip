// Dense products of the generalized eigensolve (the step after the setup that
// solvewithlapack hands to ZHEGVX, modfvsystem.f90:585-720): the Chebyshev
// filter of the subspace iteration applies the reduced Hermitian matrix C
// (n x n, n ~ 10^4) to a block of a few dozen vectors, about 130 times per
// solve.  At that shape the vendor GEMM reads C at 0.7-1.5 TB/s whatever
// the block width; this kernel splits K over many workgroups instead, so
// that the whole chip streams C once per product on FP64 MFMA.
#include "exh_device.h"

namespace exh {
namespace {

typedef double dx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ dx4 mfma16(double a, double b, dx4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// the value of the neighbouring lane (lane ^ 1), its sign flipped by mask; on
// the integer units, since FP64 multiplies share the matrix cores' pipe
__device__ __forceinline__ double swap_pair(double v, int mask) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, true);
  return __hiloint2double(hi ^ mask, lo);
}

constexpr int CT = 64;    // output rows of a workgroup: 16 per wave
constexpr int CK = 8;     // K slab of X staged in LDS per step
constexpr int CNT = 256;  // 4 waves
constexpr int CNTILE = 8; // column tiles of a workgroup at most

// part[s][i][j] = sum over k in chunk s of conj(A[k][i]) X[k][j] (asign = -1)
// or A[k][i] X[k][j] (asign = 1); chunk s is [s * kchunk, min(K, (s+1) * kchunk)).
// A(k, i) at A[k * lda + i], X(k, j) at X[k * ldx + j], part[s] row-major with
// leading dimension m.
//
// Bound by A's bytes (16 nout K) up to about 16 columns, by the FP64 matrix
// cores beyond.  The columns are taken as the 2m real columns re, im, re, ..
// that X and part hold in memory: out[c] = Re A X[c] +- Im A X[c ^ 1], so m is
// padded to a multiple of 8 and not of 64, and the workgroups' column tiles fit
// m.  The 16 rows of a wave are nobody else's: its A fragments come from memory
// in the MFMA's own lane order (16 lanes read 256 consecutive bytes), without
// LDS, one slab ahead.  X is shared by the waves through two LDS buffers (one
// barrier per slab; row length 16 mod 32 doubles, so that two rows fill the
// banks), its neighbouring column comes from the neighbouring lane.  Rows and
// columns out of range are clamped and not stored, k out of range is zero.
// n = 10364, 64 x 64 tiles of zero-padded columns before, this now (us, with the
// reduction, chunks of K as below): 8 columns 870 -> 333, 24: 870 -> 474, 40:
// 870 -> 681, 56: 886 -> 903 (5.4 TB/s of A at 8, 57 TFLOP/s at 56), 80: 1740 ->
// 1290.  Slabs of 16 K need 171 registers at seven tiles (926 us at 56), 32 rows
// per wave 206 (943).
template <int NT>
__global__ __launch_bounds__(CNT) void cx_part_kernel(int nout, int m, int K, int kchunk,
                                                      const double2 *__restrict__ A,
                                                      long long lda, double asign,
                                                      const double2 *__restrict__ X,
                                                      long long ldx,
                                                      double2 *__restrict__ part) {
  constexpr int W = 16 * NT, LX = W + (W % 32 ? 0 : 16);
  __shared__ double sx[2][CK][LX];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int I0 = blockIdx.x * CT + (tid >> 6) * 16, C0 = blockIdx.y * W, s = blockIdx.z;
  const int k0 = s * kchunk, k1 = min(K, k0 + kchunk), m2 = 2 * m;
  const double2 *ap = A + min(I0 + lr, nout - 1);
  const double *xp = (const double *)X + C0;
  const int flip = (lr & 1 ? asign : -asign) < 0.0 ? (int)0x80000000 : 0;
  constexpr int NX = (CK * W + CNT - 1) / CNT;

  dx4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = dx4{0, 0, 0, 0};
  double2 an[CK / 4];
  double xn[NX];
  auto load = [&](int kb) {
#pragma unroll
    for (int q = 0; q < CK / 4; q++) an[q] = ap[(size_t)min(kb + 4 * q + lk, k1 - 1) * lda];
#pragma unroll
    for (int i = 0; i < NX; i++) {
      const int e = tid + CNT * i;
      xn[i] = xp[(size_t)min(kb + e / W, k1 - 1) * (2 * ldx) + min(e % W, m2 - 1 - C0)];
    }
  };
  load(k0);
  int b = 0;
  for (int kb = k0; kb < k1; kb += CK, b ^= 1) {
    double2 a[CK / 4];
#pragma unroll
    for (int q = 0; q < CK / 4; q++) a[q] = kb + 4 * q + lk < k1 ? an[q] : z2(0.0, 0.0);
#pragma unroll
    for (int i = 0; i < NX; i++) {
      const int e = tid + CNT * i;
      if (CK * W % CNT == 0 || e < CK * W) sx[b][e / W][e % W] = kb + e / W < k1 ? xn[i] : 0.0;
    }
    __syncthreads();
    if (kb + CK < k1) load(kb + CK);
#pragma unroll
    for (int q = 0; q < CK / 4; q++) {
      double x[NT], y[NT];
#pragma unroll
      for (int t = 0; t < NT; t++) x[t] = sx[b][4 * q + lk][16 * t + lr];
#pragma unroll
      for (int t = 0; t < NT; t++) y[t] = swap_pair(x[t], flip);
#pragma unroll
      for (int t = 0; t < NT; t++) acc[t] = mfma16(a[q].x, x[t], acc[t]);
#pragma unroll
      for (int t = 0; t < NT; t++) acc[t] = mfma16(a[q].y, y[t], acc[t]);
    }
  }
  double *ps = (double *)(part + (size_t)s * nout * m);
#pragma unroll
  for (int t = 0; t < NT; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = I0 + lk + 4 * r, c = C0 + 16 * t + lr;
      if (i < nout && c < m2) ps[(size_t)i * m2 + c] = acc[t][r];
    }
}

// One column (m = 1: the matrix-vector products of the Lanczos bound): the
// same partial sums without MFMA, which would spend 63 of 64 columns on
// padding.  One thread per output row i, its reads of A coalesced along i;
// each chunk's x is staged in LDS 256 entries at a time.
constexpr int VT = 256;
__global__ __launch_bounds__(VT) void cx_part_vec_kernel(int nout, int K, int kchunk,
                                                         const double2 *__restrict__ A,
                                                         long long lda, double asign,
                                                         const double2 *__restrict__ X,
                                                         long long ldx,
                                                         double2 *__restrict__ part) {
  const int i = blockIdx.x * VT + threadIdx.x, s = blockIdx.y;
  const int k0 = s * kchunk, k1 = min(K, k0 + kchunk);
  __shared__ double2 sx[VT];
  const double2 *ap = A + min(i, nout - 1);
  double re = 0.0, im = 0.0;
  for (int kb = k0; kb < k1; kb += VT) {
    const int kl = min(VT, k1 - kb);
    __syncthreads();  // the previous block of x is no longer read
    if ((int)threadIdx.x < kl) sx[threadIdx.x] = X[(size_t)(kb + threadIdx.x) * ldx];
    __syncthreads();
#pragma unroll 8
    for (int t = 0; t < kl; t++) {
      const double2 a = ap[(size_t)(kb + t) * lda];
      const double2 x = sx[t];
      const double ai = asign * a.y;  // conj(A): the imaginary part negated
      re = fma(a.x, x.x, re);
      re = fma(-ai, x.y, re);
      im = fma(a.x, x.y, im);
      im = fma(ai, x.x, im);
    }
  }
  if (i < nout) part[(size_t)s * nout + i] = z2(re, im);
}

// Y[i][j] = alpha * sum_s part[s][i][j] (s in order) + beta * Y0[i][j] +
// gamma * Z[i][j]; Y may be Y0 (each element is read before it is written).
__global__ void cx_reduce_kernel(int nout, int m, int S, const double2 *__restrict__ part,
                                 double alpha, double beta, const double2 *y0, long long ld0,
                                 double gamma, const double2 *__restrict__ z, long long ldz,
                                 double2 *y, long long ldy) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t total = (size_t)nout * m;
  if (idx >= total) return;
  const int i = (int)(idx / m), j = (int)(idx % m);
  double sr = 0.0, si = 0.0;
  for (int s = 0; s < S; s++) {
    const double2 v = part[(size_t)s * total + idx];
    sr += v.x;
    si += v.y;
  }
  double yr = alpha * sr, yi = alpha * si;
  if (y0) {
    const double2 v = y0[(size_t)i * ld0 + j];
    yr = fma(beta, v.x, yr);
    yi = fma(beta, v.y, yi);
  }
  if (z) {
    const double2 v = z[(size_t)i * ldz + j];
    yr = fma(gamma, v.x, yr);
    yi = fma(gamma, v.y, yi);
  }
  y[(size_t)i * ldy + j] = z2(yr, yi);
}

}  // namespace
}  // namespace exh

extern "C" int exh_zgemm_cn_device(void *stream, int conj_a, int nout, int m, int k,
                                   const exh_z *a, long long lda, const exh_z *x, long long ldx,
                                   double alpha, double beta, const exh_z *y0, long long ldy0,
                                   double gamma, const exh_z *z, long long ldz, exh_z *y,
                                   long long ldy, int split, exh_z *work) {
  using namespace exh;
  if (nout < 0 || m < 0 || k < 1 || split < 1 || split > 4096) return EXH_EINVAL;
  if (nout == 0 || m == 0) return EXH_OK;
  if (!a || !x || !y || !work || lda < nout || ldx < m || ldy < m) return EXH_EINVAL;
  if ((y0 && ldy0 < m) || (z && ldz < m)) return EXH_EINVAL;
  // chunks of whole slabs, none empty
  int kchunk = (k + split - 1) / split;
  kchunk = (kchunk + CK - 1) / CK * CK;
  const int S = (k + kchunk - 1) / kchunk;
  hipStream_t s = (hipStream_t)stream;
  if (m == 1) {
    const dim3 grid((unsigned)((nout + VT - 1) / VT), (unsigned)S);
    hipLaunchKernelGGL(cx_part_vec_kernel, grid, dim3(VT), 0, s, nout, k, kchunk,
                       (const double2 *)a, lda, conj_a ? -1.0 : 1.0, (const double2 *)x, ldx,
                       (double2 *)work);
  } else {
    // column tiles of 8, spread evenly over the workgroups that share A
    const int tiles = (m + 7) / 8, jb = (tiles + CNTILE - 1) / CNTILE, nt = (tiles + jb - 1) / jb;
    const dim3 grid((unsigned)((nout + CT - 1) / CT), (unsigned)jb, (unsigned)S);
#define LAUNCH(NT)                                                                          \
  case NT:                                                                                  \
    hipLaunchKernelGGL(cx_part_kernel<NT>, grid, dim3(CNT), 0, s, nout, m, k, kchunk,       \
                       (const double2 *)a, lda, conj_a ? -1.0 : 1.0, (const double2 *)x,    \
                       ldx, (double2 *)work);                                               \
    break;
    switch (nt) {
      LAUNCH(1) LAUNCH(2) LAUNCH(3) LAUNCH(4) LAUNCH(5) LAUNCH(6) LAUNCH(7) LAUNCH(8)
    }
#undef LAUNCH
  }
  const size_t total = (size_t)nout * m;
  hipLaunchKernelGGL(cx_reduce_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                     nout, m, S, (const double2 *)work, alpha, beta, (const double2 *)y0, ldy0,
                     gamma, (const double2 *)z, ldz, (double2 *)y, ldy);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? EXH_OK : (int)e;
}
