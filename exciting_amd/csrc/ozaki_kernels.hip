// Modular muffin-tin contraction (Ozaki scheme II on int8 MFMA): exact
// integer products of rounded operands through residues.
//
// The products H_MT = X^H B and O_MT = X^H Y (X = A^T, B = (aa A)^T, Y = X or,
// for iora*, ((1+h1) A)^T; K = every atom's (l, m, io) stacked) are computed
// as follows:
//
//  1. Each G column of an operand gets a power-of-two scale 2^s so that its
//     2-norm is at most 2^(c-1); the scaled values are rounded to integers.
//     This rounding is the only approximation: at most 1/2 of 2^-s per
//     component, i.e. about 2^-c of the column's norm.
//  2. The moduli p_m are products of primes = 1 mod 4, where -1 has a square
//     root I_m.  The Gaussian integer z = zr + i zi then has the two residues
//     z+ = zr + I zi and z- = zr - I zi mod p, which multiply separately:
//     (conj(x) y)+ = x- y+ and (conj(x) y)- = x+ y-.  A complex product costs
//     two real products instead of the three of Karatsuba's scheme modulo
//     arbitrary primes (28.0 -> 18.1 ms at K = 15488, G = 9340, 7 moduli), and
//     two residue arrays per operand instead of three or four.  Residues are
//     int8 in [-p/2, p/2], stored in 16-byte k blocks per G row: the operand
//     format of v_mfma_i32_32x32x32_i8.
//  3. Per modulus and sign, an upper-triangular int8 GEMM accumulates H and O
//     exactly in int32 (K <= kOzMaxK) and stores them modulo p as one signed
//     byte per element (operands streamed global -> LDS by direct DMA loads).
//  4. Re = (P+ + P-)/2 and Im = (P+ - P-)/(2 I) modulo every p are turned
//     back into the exact integers by the Chinese remainder theorem in two-
//     word FP64 (the high words sum without rounding) and rescaled by
//     2^-(s_i+s_j).  The interstitial terms and the conj mirror are added as
//     in the FP64 path.
//
// The integers are Re and Im of x_i^H b_j, bounded by ||x_i|| ||b_j|| <=
// 2^(2c-2) (Cauchy-Schwarz), so n moduli with prod p > 2^(2c-1) recover every
// element exactly.
//
// EXH_SPLIT(n) fixes c as the caller asked (27 bits for n = 7).  Without that
// flag, large bases run here with 15 moduli and c = 56 (oz_fp64): the
// operands keep 55 bits relative to the column norm and nothing else is
// rounded.  Over whole matrices that is closer to the exact products than the
// FP64 MFMA kernels (relative Frobenius error of the contraction alone at 16
// atoms, K = 3872: 2e-16 against 2.4e-15; median element 6e-16 against
// 2.7e-15), whose K-long FP64 accumulation rounds 4 K times per element.
// But the error of element (i, j) is bounded by 2^-55 sqrt(K) ||x_i|| ||b_j||, and
// that of FP64 sums by K 2^-53 sum_k |x_ki| |b_kj|, which does not see how the
// radial functions are normalised.  For H the FP64 products therefore multiply
// X' = 2^t X and B' = 2^-t B with the tables' row exponents t (setup_kernels.hip,
// row_exponents_kernel): the same H, and operands that a change of normalisation
// leaves as they are.  Without them, the io = 1 functions scaled by 2^-10 and
// 2^-20 took H from 1.4e-16 to 8e-14 and 8e-11.  O = X^H Y has its rows unscaled
// (||x_i||^2 is its diagonal), so FP64 has X twice among its operands.  Equal row
// exponents (a flag the tables' kernels leave) make X' and X one.  What is left
// of the difference: two columns that are large in different functions.
//
// Columns whose norm is not finite give NaN rows and columns of H and O, as
// any FP64 sum over them would; zero columns give zeros.
#include <algorithm>
#include <climits>
#include <cmath>

#include "exh_device.h"

namespace exh {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int OZ_T = 128;   // output tile edge
constexpr int OZ_KS = 64;   // k per LDS stage (4 blocks of 16)
constexpr int OZ_N = kOzModuli;
constexpr int OZ_WR = 3;           // 32-row blocks per wave (96 rows)
constexpr int OZ_NWG = 8;          // waves per workgroup
constexpr int OZ_R = 48 * OZ_NWG;  // rows of the row panel per workgroup
constexpr int OZ_W = OZ_R + 2 * OZ_T;  // rows and columns of one LDS stage

// ---------------------------------------------------------------------------
// Moduli: the largest pairwise coprime products of primes = 1 mod 4 below
// 256 (221 = 13*17, 205 = 5*41), and a square root of -1 for each.
// ---------------------------------------------------------------------------
constexpr int kP[OZ_N] = {241, 233, 229, 221, 205, 197, 193, 181,
                          173, 157, 149, 137, 113, 109, 101};

constexpr int sym(long long x, int p) {  // representative in [-p/2, p/2]
  long long r = x % p;
  if (r < 0) r += p;
  return (int)(2 * r > p ? r - p : r);
}
constexpr int root(int p) {
  for (int i = 2; i < p; i++)
    if ((i * i + 1) % p == 0) return sym(i, p);
  return 0;
}
constexpr int inverse(long long a, int p) {
  long long r = ((a % p) + p) % p;
  for (int x = 1; x < p; x++)
    if (r * x % p == 1) return x;
  return 0;
}

// Residue constants of one modulus.  kMagic + r is exact for integers
// |r| < 2^51 and holds r in its low 32 bits; nk cancels it in the quotient.
constexpr double kMagic = 6755399441055744.0;  // 1.5 * 2^52
constexpr int kSplit = 27;                     // y = h 2^27 + l
struct OzMod {
  double p, rp, nk;   // p, 1/p, -kMagic/p
  double c1, c2, im;  // 2^27, 2^27 I, I mod p (symmetric)
};
struct OzMods {
  OzMod m[OZ_N];
};
constexpr OzMods make_mods() {
  OzMods t{};
  for (int k = 0; k < OZ_N; k++) {
    const int p = kP[k], i = root(p);
    t.m[k].p = p;
    t.m[k].rp = 1.0 / p;
    t.m[k].nk = -(kMagic * (1.0 / p));
    t.m[k].c1 = sym(1ll << kSplit, p);
    t.m[k].c2 = sym((1ll << kSplit) * i, p);
    t.m[k].im = i;
  }
  return t;
}
__constant__ const OzMods c_mod = make_mods();

// CRT constants for the first n moduli, P = their product: with s = P+ + P-
// and d = P+ - P- (signed bytes, |s|, |d| <= 2 * 121),
//   Re = sum_m s_m re_m mod P,  Im = sum_m d_m im_m mod P,
//   re_m = (P/p) [(P/p)^-1 / 2 mod p],  im_m = (P/p) [(P/p)^-1 / (2 I) mod p]
// (symmetric), each split into a high word that is a multiple of 2^T and a
// low word |.| < 2^T.  T is such that the sums of high words stay below
// 2^(T+53) and are therefore exact; the low words contribute rounding errors
// of at most 2^(T+13-53), 2^-81 P at n = 15.
struct OzCrt {
  double reh[OZ_N], rel[OZ_N], imh[OZ_N], iml[OZ_N];
  double rP, Ph, Pl;
};
struct OzCrts {
  OzCrt t[OZ_N + 1];
};
typedef __int128 i128;
constexpr int bits_of(i128 x) {
  int n = 0;
  while (x > 0) {
    x >>= 1;
    n++;
  }
  return n;
}
constexpr double to_double(i128 x) {  // exact when x has at most 53 bits after its trailing zeros
  return (double)x;
}
constexpr OzCrts make_crts() {
  OzCrts all{};
  for (int n = 1; n <= OZ_N; n++) {
    OzCrt &c = all.t[n];
    i128 P = 1;
    for (int k = 0; k < n; k++) P *= kP[k];
    // sum |s| |re| <= n * 242 * P/2 < 2^(bits(P) + 11)
    const int T = bits_of(P) + 11 > 53 ? bits_of(P) + 11 - 53 : 0;
    const i128 unit = (i128)1 << T;
    c.rP = 1.0 / to_double(P);
    c.Ph = to_double(P / unit * unit);
    c.Pl = to_double(P % unit);
    for (int k = 0; k < n; k++) {
      const int p = kP[k];
      const i128 Q = P / p;
      const long long qi = inverse((long long)(Q % p), p);
      const long long a = sym(qi * inverse(2, p), p);
      const long long b = sym(qi * inverse(2ll * root(p), p), p);
      const i128 re = Q * a, im = Q * b;
      const i128 reh = re / unit * unit, imh = im / unit * unit;  // truncated toward 0
      c.reh[k] = to_double(reh);
      c.rel[k] = to_double(re - reh);
      c.imh[k] = to_double(imh);
      c.iml[k] = to_double(im - imh);
    }
  }
  return all;
}
__constant__ const OzCrts c_crt = make_crts();

// ---------------------------------------------------------------------------
// Column norms: partial sums of |x|^2, then per column their sum and
// emax[g] = E + 1 with ||x_g|| < 2^E: the scale 2^(c - emax) takes the norm
// below 2^(c-1).  emax = INT_MIN for a zero column, INT_MAX for one that is
// not finite.  bt writes the partial sums of X and B from the values it holds
// (a pass of their own read both operands again: 0.79 of 26 ms at 64 atoms, 7
// moduli); the kernel below does it for operands that bt has not seen (O
// alone, (1+h1)A): part[chunk][g] over 256 k in a fixed order (four k groups
// per workgroup, added in order).  A partial sum whose squares would leave
// FP64's range is marked kNormRecompute, and the final kernel then sums that
// column again from scaled values.
// ---------------------------------------------------------------------------
constexpr int OZ_NCH = 256;      // k per partial sum

__device__ __forceinline__ void colnorm_part_body(const OzK &d, int z) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = blockIdx.x * 64 + lane;
  const int k0 = blockIdx.y * OZ_NCH, k1 = min(d.Ktot, k0 + OZ_NCH);
  if (z >= d.nops || (d.fused >> z & 1) || (int)blockIdx.x * 64 >= d.ngp || k0 >= k1)
    return;  // uniform
  const EXH_G double2 *xp = gptr(d.x[z]) + min(g, d.ngp - 1);
  const long long ldx = d.ld[z];
  EXH_G double *part = gptr(d.part[z]);
  __shared__ double ss[4][64], sm[4][64];
  double s = 0.0, amax = 0.0;
#pragma unroll 8
  for (int k = k0 + w; k < k1; k += 4) {
    const double2 v = ld(xp + (size_t)k * ldx);
    s = fma(v.x, v.x, s);
    s = fma(v.y, v.y, s);
    amax = fmax(amax, fmax(fabs(v.x), fabs(v.y)));
  }
  ss[w][lane] = s;
  sm[w][lane] = amax;
  __syncthreads();
  if (w == 0 && g < d.ngp) {
    amax = fmax(fmax(sm[0][lane], sm[1][lane]), fmax(sm[2][lane], sm[3][lane]));
    part[(size_t)blockIdx.y * d.ldp + g] =
        ((ss[0][lane] + ss[1][lane]) + ss[2][lane]) + ss[3][lane];
    ((EXH_G int *)(part + (size_t)d.nch[z] * d.ldp))[(size_t)blockIdx.y * d.ldp + g] =
        norm_mark(amax);
  }
}

// 64 columns per workgroup, the chunks split over four waves.
__device__ __forceinline__ void colnorm_final_body(const OzK &d, int z) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = blockIdx.x * 64 + lane;
  if (z >= d.nops || (int)blockIdx.x * 64 >= d.ngp) return;  // uniform
  const int nch = d.nch[z], ldp = d.ldp, gc = min(g, d.ngp - 1);
  const EXH_G double *part = gptr((const double *)d.part[z]) + gc;
  const EXH_G int *pe = (const EXH_G int *)(gptr((const double *)d.part[z]) + (size_t)nch * ldp) + gc;
  __shared__ double ss[4][64];
  __shared__ int sm[4][64];
  const int per = (nch + 3) / 4, c0 = w * per, c1 = min(nch, c0 + per);
  double s = 0.0;
  int mark = 0;
#pragma unroll 8
  for (int c = c0; c < c1; c++) {
    s += part[(size_t)c * ldp];
    mark |= pe[(size_t)c * ldp];
  }
  ss[w][lane] = s;
  sm[w][lane] = mark;
  __syncthreads();
  if (w != 0 || g >= d.ngp) return;
  s = ((ss[0][lane] + ss[1][lane]) + ss[2][lane]) + ss[3][lane];
  int em = 0, e = INT_MIN;
  if (sm[0][lane] | sm[1][lane] | sm[2][lane] | sm[3][lane]) {
    // rare: squares out of range; the column again, scaled by its largest entry
    const EXH_G double2 *xp = gptr(d.x[z]) + g;
    const int rs = d.rs[z];
    int top = INT_MIN;
    for (int k = 0; k < d.Ktot; k++) {
      const double2 v = ld(xp + (size_t)k * d.ld[z]);
      const double amax = fmax(fabs(v.x), fabs(v.y));
      if (amax > 0.0) top = max(top, exponent_of(amax) + (rs ? rs * d.rexp[k] : 0));
    }
    em = top;
    s = 0.0;
    for (int k = 0; k < d.Ktot; k++) {
      const double2 v = ld(xp + (size_t)k * d.ld[z]);
      const int sh = (rs ? rs * d.rexp[k] : 0) - em;
      const double a = ldexp(v.x, sh), b = ldexp(v.y, sh);
      s = fma(a, a, s);
      s = fma(b, b, s);
    }
  }
  if (!(s - s == 0.0)) {
    e = INT_MAX;  // Inf or NaN in the column
  } else if (s > 0.0) {
    (void)frexp(sqrt(s), &e);  // norm = f 2^e, f in [0.5, 1): norm < 2^e
    e += 1 + em;
  }
  gptr(d.e[z])[g] = e;
}

// ---------------------------------------------------------------------------
// Residues: one thread per (16-k block, G row), blockIdx.z the operand.
// y = rint(x 2^s) = h 2^27 + l; then per modulus, all in exact FP64 integers,
//   y+- = (hr c1 + lr) +- (hi c2 + li I),   r = y+- - p rint(y+- / p),
// the low byte of kMagic + r being the residue.  |r| <= (1/2 + 2^-9) p.
// Rows ngp..rows-1 and k >= Ktot are written as zeros (no masking
// downstream).  Layout, m counted from m0: Q[(2 m + t) * qstride + (kblk * Gpad + g) * 16 + byte], t = 0 for
// y+, 1 for y-.  About 13 FP64 operations per (element, modulus) beside
// 2 bytes written: bound by HBM and the vector unit alike.
// ROWS: with a row exponent of its own per k (its loads cost 3-7 % where they are
// not needed: 8 k-points of K = 1936, G = 1172, two operands, 361 -> 343 us).
// ---------------------------------------------------------------------------
__device__ __forceinline__ int low_word(double x) { return (int)__double_as_longlong(x); }

// low bytes of the low words of four doubles
__device__ __forceinline__ int pack4(double a, double b, double c, double d) {
  const unsigned x = __builtin_amdgcn_perm((unsigned)low_word(b), (unsigned)low_word(a), 0x0c0c0400);
  const unsigned y = __builtin_amdgcn_perm((unsigned)low_word(d), (unsigned)low_word(c), 0x04000c0c);
  return (int)(x | y);
}

template <bool ROWS>
__device__ __forceinline__ void residue_body(const OzK &d, int z, int m0, int m1) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  const int kb = blockIdx.y;
  const int ngp = d.ngp, Ktot = d.Ktot;
  const int rows = d.nt * OZ_T;  // whole tiles
  if (z >= d.nops || g >= rows || kb >= d.nslab * (OZ_KS / 16)) return;
  const EXH_G double2 *X = gptr(d.x[z]);
  const long long ldx = d.ld[z];
  double hr[16], lr[16], hi[16], li[16];
  int e = INT_MIN;
  if (g < ngp) e = gptr((const int *)d.e[z])[g];
  const bool live = e != INT_MIN && e != INT_MAX;
  const int rs = d.rs[z];
  const EXH_C int *rexp = cptr(d.rexp);
  const int s0 = (live ? d.bits - e : 0) + (!ROWS && rs ? rs * rexp[0] : 0);
#pragma unroll
  for (int t = 0; t < 16; t++) {
    const int k = kb * 16 + t;
    double2 v = z2(0.0, 0.0);
    if (live && k < Ktot) v = exh::ld(X + (size_t)k * ldx + g);
    const int s = ROWS ? s0 + rs * rexp[min(k, Ktot - 1)] : s0;
    const double yr = rint(ldexp(v.x, s)), yi = rint(ldexp(v.y, s));
    constexpr double D = (double)(1ll << kSplit);
    hr[t] = rint(yr * (1.0 / D));
    lr[t] = fma(-D, hr[t], yr) + kMagic;
    hi[t] = rint(yi * (1.0 / D));
    li[t] = fma(-D, hi[t], yi);
  }
  const size_t qstride = d.qstride;
  EXH_G int8_t *out = gptr(d.q) + d.qi[z] * d.q_bytes + ((size_t)kb * d.Gpad + g) * 16;
#pragma unroll 1
  for (int m = m0; m < m1; m++) {
    const double p = c_mod.m[m].p, rp = c_mod.m[m].rp, nk = c_mod.m[m].nk;
    const double c1 = c_mod.m[m].c1, c2 = c_mod.m[m].c2, im = c_mod.m[m].im;
    int wp[4], wm[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      double rpos[4], rneg[4];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const int k = 4 * q + t;
        const double a = fma(hr[k], c1, lr[k]);
        const double b = fma(hi[k], c2, li[k] * im);
        const double u = a + b, v = a - b;
        rpos[t] = fma(-p, rint(fma(u, rp, nk)), u);
        rneg[t] = fma(-p, rint(fma(v, rp, nk)), v);
      }
      wp[q] = pack4(rpos[0], rpos[1], rpos[2], rpos[3]);
      wm[q] = pack4(rneg[0], rneg[1], rneg[2], rneg[3]);
    }
    *(EXH_G v4i *)(out + (size_t)(2 * (m - m0)) * qstride) = v4i{wp[0], wp[1], wp[2], wp[3]};
    *(EXH_G v4i *)(out + (size_t)(2 * (m - m0) + 1) * qstride) = v4i{wm[0], wm[1], wm[2], wm[3]};
  }
}

// ---------------------------------------------------------------------------
// Upper-triangular int8 GEMMs.  One workgroup computes, for one modulus and
// sign, a 384-row panel of the row operand (x- for the sign +, x+ for -) against
// two 128-column blocks: with EXH_SPLIT the block J of H's and of O's column
// operand, which then share the row operand; otherwise (ONE) the blocks 2J and
// 2J + 1 of one matrix, as H's row operand has its rows scaled and O's has not:
//   C[i][j] = sum_k A[k][i] B[k][j]
// (int32, exact), each stored mod p as signed bytes in the 128x128 tiles on
// or above the diagonal.  Each wave owns
// 96 rows x 64 columns of both products (3 x 2 blocks of
// v_mfma_i32_32x32x32_i8 each, 192 accumulator registers) and reads 7 operand
// fragments from LDS per 12 MFMAs; 8 waves form 4 row groups x 2 column
// groups, one workgroup per CU.  (192-row panels, two 4-wave workgroups per
// CU whose barriers fall at different times, gave the same products and
// measured 1 % slower at the 64-atom shape.)
// Operands stream global -> LDS directly (buffer loads to LDS, 16 bytes per
// lane, one 64-row chunk of one k block per instruction), two stages of 64 k
// double-buffered.
// Bound by the power the matrix cores draw: at K = 15488, G = 9340, 14
// products, 16.4 ms = 2.30 POP/s with the cores busy 72 % of the cycles at
// 1.56 GHz; with all-zero operands (same instructions) 13.4 ms.  Reading the
// fragments ahead took it there from 17.9 ms (60 % busy), where both waves of
// a SIMD waited for LDS four times per stage.  A third stage in LDS (16.5 ms)
// and raised wave priority around the MFMAs (16.3-16.4 ms) change nothing.
// Operand lane layout: row/column = lane%32, 16 k bytes from k block
// 2*ks + lane/32; result D[8*(r/4) + 4*(lane/32) + r%4][lane%32].
// ---------------------------------------------------------------------------

#define EXH_LDS(p) ((__attribute__((address_space(3))) void *)(p))
#define EXH_GLB(p) ((const __attribute__((address_space(1))) void *)(p))

// Residues mod p of the 96 x 64 strip of a wave, four consecutive rows packed
// per 32-bit store, into the 128x128 tiles on or above the diagonal.  A tile
// is stored as 16 sub-blocks of 32 x 32 (4 bj + bi) in accumulator order --
// word 64 h + lane holds rows 8 h + 4 (lane/32) .. + 3 of column lane%32 --
// so that each store instruction writes 256 contiguous bytes here and each
// load instruction of the reconstruction reads them.
__device__ __forceinline__ void store_residues(const v16i (&acc)[OZ_WR][2], const OzMod &M,
                                               int rg, int wc, int lane, int IT, int J, int t0,
                                               EXH_G int8_t *Rp) {
  const double p = M.p, rp = M.rp, nk = M.nk;
#pragma unroll
  for (int a = 0; a < OZ_WR; a++) {
    const int row = IT * OZ_R + rg * 32 * OZ_WR + a * 32;
    const int I = row >> 7;
    if (I > J) continue;  // below the diagonal (uniform per wave)
    EXH_G int8_t *out = Rp + ((long long)J * (J + 1) / 2 + I - t0) * (OZ_T * OZ_T) + 4 * lane;
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int h = 0; h < 4; h++) {
        double r[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
          const double x = (double)acc[a][b][4 * h + t] + kMagic;
          r[t] = fma(-p, rint(fma(x, rp, nk)), x);
        }
        const int sub = 4 * (2 * wc + b) + ((row & 127) >> 5);
        *(EXH_G int *)(out + sub * 1024 + h * 256) = pack4(r[0], r[1], r[2], r[3]);
      }
  }
}

// Row panels that columns up to (and including) block j of 128 need.
__host__ __device__ inline int oz_npan(int j) { return (j * OZ_T + OZ_T - 1) / OZ_R + 1; }

// Column steps of one GEMM and the last 128-column block of step j: the
// fused products step by one block, O alone by two (nt blocks in all).
template <bool ONE>
__host__ __device__ inline int oz_steps(int nt) { return ONE ? (nt + 1) / 2 : nt; }
template <bool ONE>
__host__ __device__ inline int oz_last(int j, int nt) {
  const int l = ONE ? 2 * j + 1 : j;
  return l < nt ? l : nt - 1;
}

// Panels per GEMM, of the column steps s0 .. s1 - 1.
template <bool ONE>
__host__ __device__ inline long long oz_panels(int nt, int s0, int s1) {
  long long n = 0;
  for (int j = s0; j < min(s1, oz_steps<ONE>(nt)); j++) n += oz_npan(oz_last<ONE>(j, nt));
  return n;
}

// Tiles of those steps: the first one's number, and how many.
struct OzTiles {
  int t0, n;
};
template <bool ONE>
__host__ __device__ inline OzTiles oz_tiles(int nt, int s0, int s1) {
  const int w = ONE ? 2 : 1, a = min(nt, s0 * w), b = min(nt, min(s1, oz_steps<ONE>(nt)) * w);
  return {a * (a + 1) / 2, max(0, b * (b + 1) / 2 - a * (a + 1) / 2)};
}

// Panel order: super-columns of OZ_SJ column steps, each walked in chunks
// of OZ_SI row panels (4 x 384 rows), so that the workgroups an XCD runs at
// once share a few row panels and column panels in its L2 (the column-major
// order had 32 co-resident workgroups share about 1 column panel and 19 row
// panels); 3.6 % faster at the 64-atom shape, bitwise the same products.
constexpr int OZ_SJ = 8, OZ_SI = 4 * 384 / OZ_R;

// Panel o of one GEMM's steps s0 .. s1 - 1 -> (column step J, row panel IT).
template <bool ONE>
__device__ __forceinline__ void oz_panel_at(int o, int nt, int s0, int s1, int &J, int &IT) {
  const int ns = min(s1, oz_steps<ONE>(nt));
  auto npan = [&](int j) { return oz_npan(oz_last<ONE>(j, nt)); };
  int rem = o, j0 = s0;
  for (;; j0 += OZ_SJ) {
    const int j1 = min(ns, j0 + OZ_SJ);
    int cnt = 0;
    for (int j = j0; j < j1; j++) cnt += npan(j);
    if (rem < cnt) break;
    rem -= cnt;
  }
  const int j1 = min(ns, j0 + OZ_SJ);
  int i0 = 0;
  for (;; i0 += OZ_SI) {
    int cnt = 0;
    for (int j = j0; j < j1; j++) cnt += max(0, min(OZ_SI, npan(j) - i0));
    if (rem < cnt) break;
    rem -= cnt;
  }
  J = j0;
  IT = i0;
  for (int j = j0; j < j1; j++) {
    const int cj = max(0, min(OZ_SI, npan(j) - i0));
    if (rem < cj) {
      J = j;
      IT = i0 + rem;
      return;
    }
    rem -= cj;
  }
}

// Residues of the moduli m0 .. m0 + mc - 1 are in d.q, counted from m0.  ONE: of
// the matrices mat0 .. mat0 + nmat - 1 (H, O).
template <bool ONE>
__device__ __forceinline__ void ozgemm_body(const OzK &d, int m0, int mc, int s0, int s1, int mat0,
                                            int nmat, bool uni, v4i (&sm0)[4][OZ_W],
                                            v4i (&sm1)[4][OZ_W]) {
  const int nt = d.nt, nslab = d.nslab, Gpad = d.Gpad;
  const size_t qstride = d.qstride;
  // XCD-contiguous remap over the k-point's panels (its first block runs on
  // XCD 0: the grid's x extent is a multiple of 8), then ((matrix, sign) * mc + m,
  // panel)
  const int per = (int)oz_panels<ONE>(nt, s0, s1);
  const int bid = blockIdx.x, nb = per * 2 * mc * nmat;
  if (bid >= nb) return;
  const int xcd = bid & 7, i8 = bid >> 3, q8 = nb >> 3, r8 = nb & 7;
  const int t = xcd * q8 + (xcd < r8 ? xcd : r8) + i8;
  const int qm = __builtin_amdgcn_readfirstlane(t / per), o = t - qm * per;
  const int mq = __builtin_amdgcn_readfirstlane(qm / mc);
  const int m = qm - mq * mc, q = mq & 1, mat = mat0 + (mq >> 1);  // q = 0: sign +, 1: -
  int J, IT;
  oz_panel_at<ONE>(o, nt, s0, s1, J, IT);
  // uniform by construction; scalar registers for the addresses that follow
  J = __builtin_amdgcn_readfirstlane(J);
  IT = __builtin_amdgcn_readfirstlane(IT);
  const OzTiles T = oz_tiles<ONE>(nt, s0, s1);
  const int JH = ONE ? 2 * J : J, JO = ONE ? 2 * J + 1 : J;
  const int I0 = IT * OZ_R, H0 = JH * OZ_T;
  // past the last block (odd nt): any valid columns, not stored
  const int O0 = min(JO, nt - 1) * OZ_T;

  const int zr = ONE && !mat && !uni ? d.iA : d.iX, zh = ONE && mat ? d.iY : d.iB;
  const int zo = ONE ? zh : d.iY;
  // in scalar registers: the DMA loads of the loop would otherwise each be a loop
  // over the lanes' (equal) addresses (0.333 -> 0.364 us per workgroup)
  auto operand = [&](int z, int sign) {
    const uintptr_t u = (uintptr_t)(d.q + d.qi[z] * d.q_bytes + (size_t)(2 * m + sign) * qstride);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((int)u);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(u >> 32));
    return (const int8_t *)((uintptr_t)hi << 32 | lo);
  };
  const int8_t *Ab = operand(zr, 1 - q), *Hb = operand(zh, q), *Ob = ONE ? Hb : operand(zo, q);

  // one LDS array per stage: the compiler then sees the DMA into one stage and
  // the reads of the other as disjoint (no wait inserted).  Rows 0..383 hold
  // the row operand, then the two column blocks.
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = w >> 1, wc = w & 1, l32 = lane & 31, lh = lane >> 5;
  v16i ah[OZ_WR][2], ao[OZ_WR][2];
#pragma unroll
  for (int a = 0; a < OZ_WR; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) {
      ah[a][b] = v16i{0};
      ao[a][b] = v16i{0};
    }

  // Chunks of 64 rows x 16 bytes per stage: 4 k blocks x OZ_R/64 row chunks
  // of A (3 per wave), 4 k blocks x 2 of H and of O (one each per wave); each
  // lane moves its 16 bytes to chunk base + 16 lane.  Buffer loads keep the
  // addresses in scalar registers, which leaves the vector registers to the
  // second set of operand fragments below.
  constexpr int RC = OZ_R / 64;
  static_assert(4 * RC == OZ_WR * OZ_NWG && OZ_NWG == 8, "chunking");
  const int voff = lane * 16;
  auto issue = [&](int s, v4i (*st)[OZ_W]) {
    const size_t so = (size_t)s * 4 * Gpad * 16;
    const int span = 4 * Gpad * 16;  // bytes of the stage's four k blocks
    constexpr int kRaw = 0x00020000;
    const auto rA = __builtin_amdgcn_make_buffer_rsrc((void *)(Ab + so), 0, span, kRaw);
    const auto rH = __builtin_amdgcn_make_buffer_rsrc((void *)(Hb + so), 0, span, kRaw);
    const auto rO = __builtin_amdgcn_make_buffer_rsrc((void *)(Ob + so), 0, span, kRaw);
#pragma unroll
    for (int u = 0; u < OZ_WR; u++) {
      const int ci = w * OZ_WR + u;
      const int kk = ci / RC, rc = ci - RC * kk;
      // the last panel may reach past the padded rows: any rows, not stored
      const int row = min(I0 + rc * 64, Gpad - 64);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rA, EXH_LDS(&st[kk][rc * 64]), 16, voff,
                                               (kk * Gpad + row) * 16, 0, 0);
    }
    const int kk = w >> 1, rc = w & 1;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rH, EXH_LDS(&st[kk][OZ_R + rc * 64]), 16, voff,
                                             (kk * Gpad + H0 + rc * 64) * 16, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rO, EXH_LDS(&st[kk][OZ_R + OZ_T + rc * 64]), 16, voff,
                                             (kk * Gpad + O0 + rc * 64) * 16, 0, 0);
  };
  const int ra = rg * 32 * OZ_WR + l32, ca = OZ_R + wc * 64 + l32;
  auto rdA = [&](v4i (*st)[OZ_W], int ks, int a) { return st[2 * ks + lh][ra + a * 32]; };
  auto rdH = [&](v4i (*st)[OZ_W], int ks, int b) { return st[2 * ks + lh][ca + b * 32]; };
  auto rdO = [&](v4i (*st)[OZ_W], int ks, int b) { return st[2 * ks + lh][ca + OZ_T + b * 32]; };
  // four MFMAs of block row a, kept apart from the reads before and after
  auto mm = [&](int a, v4i A, const v4i (&h)[2], const v4i (&o)[2]) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < 2; b++) {
      ah[a][b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, h[b], ah[a][b], 0, 0, 0);
      ao[a][b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, o[b], ao[a][b], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // One stage of 64 k: six groups of four MFMAs.  The fragments of a group
  // are read from LDS one or two groups ahead (h1, o1: the second 32 k; then
  // h0, o0 of the next stage), so the two waves of a SIMD, which the barrier
  // keeps in step, do not both wait for LDS.  At the barrier every read of
  // `cur` has returned (lgkmcnt) and the next stage has landed (vmcnt): `cur`
  // is refilled with stage s + 2, and eight MFMAs whose operands are in
  // registers cover the first reads of `nxt`.  The last two refills repeat
  // the last stage and are not read.
  v4i h0[2], o0[2], h1[2], o1[2], x0, x1, x2;
#define EXH_STAGE_BARRIER(N) \
  asm volatile("s_waitcnt vmcnt(" #N ") lgkmcnt(0)\n\ts_barrier" ::: "memory")
  auto stage = [&](int s, v4i (*cur)[OZ_W], v4i (*nxt)[OZ_W]) {
    x1 = rdA(cur, 0, 1);
    h1[0] = rdH(cur, 1, 0);
    mm(0, x0, h0, o0);
    x2 = rdA(cur, 0, 2);
    h1[1] = rdH(cur, 1, 1);
    o1[0] = rdO(cur, 1, 0);
    mm(1, x1, h0, o0);
    x0 = rdA(cur, 1, 0);
    o1[1] = rdO(cur, 1, 1);
    x1 = rdA(cur, 1, 1);
    mm(2, x2, h0, o0);
    x2 = rdA(cur, 1, 2);
    mm(0, x0, h1, o1);
    EXH_STAGE_BARRIER(0);
    issue(min(s + 2, nslab - 1), cur);
    __builtin_amdgcn_sched_barrier(0);
    h0[0] = rdH(nxt, 0, 0);
    o0[0] = rdO(nxt, 0, 0);
    h0[1] = rdH(nxt, 0, 1);
    mm(1, x1, h1, o1);
    o0[1] = rdO(nxt, 0, 1);
    x0 = rdA(nxt, 0, 0);
    mm(2, x2, h1, o1);
  };
  issue(0, sm0);
  issue(1, sm1);
  EXH_STAGE_BARRIER(5);  // stage 0 has landed, stage 1 (5 loads) may be in flight
  h0[0] = rdH(sm0, 0, 0);
  o0[0] = rdO(sm0, 0, 0);
  h0[1] = rdH(sm0, 0, 1);
  o0[1] = rdO(sm0, 0, 1);
  x0 = rdA(sm0, 0, 0);
  for (int s = 0; s < nslab; s += 2) {
    stage(s, sm0, sm1);
    stage(s + 1, sm1, sm0);
  }
#undef EXH_STAGE_BARRIER
  // the LDS must outlive the last refills
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)

  // planes: (H+, H-, O+, O-) x modulus, or of O alone (O+, O-) x modulus
  const size_t plane = (size_t)T.n * (OZ_T * OZ_T);
  const int pl = 2 * (ONE && d.h ? mat : 0) + q;
  EXH_G int8_t *Rq = gptr(d.r) + (size_t)(pl * d.nmod + m0 + m) * plane;
  const OzMod &M = c_mod.m[m0 + m];
  store_residues(ah, M, rg, wc, lane, IT, JH, T.t0, Rq);
  if (ONE) {
    if (JO < nt) store_residues(ao, M, rg, wc, lane, IT, JO, T.t0, Rq);
  } else {
    store_residues(ao, M, rg, wc, lane, IT, JO, T.t0, Rq + (size_t)2 * d.nmod * plane);
  }
}

// ---------------------------------------------------------------------------
// Residues -> FP64 H and O upper elements (+ interstitial, + mirror).
// One workgroup per 32x32 sub-block of a tile: each thread reconstructs four
// consecutive rows of one column from one 32-bit word per plane, the
// sub-block is staged in LDS and written to the upper triangle (coalesced
// along i) and, transposed and conjugated, to the lower one (coalesced along
// j).  Per value and modulus: one add, one conversion and two FMAs (Garner's
// algorithm needs m multiply-adds and a reduction at step m).  Bound by HBM:
// 4 n bytes read and 64 written per upper element; 2.6 -> 1.26 ms at G = 9340
// with 7 moduli (4.0 GB, 3.2 TB/s), 375 -> 24 us at G = 1166 with 9, where one
// workgroup per 128 x 128 tile left most of the chip idle.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int byte_of(int w, int t) { return (int)((unsigned)w << (24 - 8 * t)) >> 24; }

template <int NM>
__device__ __forceinline__ double crt(double hi, double lo) {
  const OzCrt &C = c_crt.t[NM];
  const double q = rint(hi * C.rP);  // |x| < 0.48 P: the low words cannot change it
  return fma(-q, C.Ph, hi) + fma(-q, C.Pl, lo);
}

template <int NM, bool ONLY_O>
__device__ __forceinline__ void ozcombine_body(const OzK &d, int accumulate, int s0, int s1) {
  const OzTiles T = oz_tiles<NM == OZ_N>(d.nt, s0, s1);  // the products' column steps
  const int sb = blockIdx.x & 15, ngp = d.ngp, bits = d.bits;
  if ((int)(blockIdx.x >> 4) >= T.n) return;
  const int tile = T.t0 + (int)(blockIdx.x >> 4);
  const EXH_G int *ea = gptr((const int *)d.e[d.iA]), *ex = gptr((const int *)d.e[d.iX]);
  const EXH_G int *eb = gptr((const int *)d.e[d.iB]), *ey = gptr((const int *)d.e[d.iY]);
  EXH_G double2 *H = gptr(d.h), *O = gptr(d.o);
  const long long ldh = d.ldh;
  const IstBoxT<const EXH_G int4 *, const EXH_G double *> box{
      gptr(d.box.ivgk), gptr(d.box.vgpc), d.box.T, d.box.lo0, d.box.lo1, d.box.lo2,
      d.box.n0, d.box.n1, d.box.n2};
  int J = (int)((sqrt(8.0 * (double)tile + 1.0) - 1.0) * 0.5);
  while ((J + 1) * (J + 2) / 2 <= tile) J++;
  while (J * (J + 1) / 2 > tile) J--;
  const int I = tile - J * (J + 1) / 2;
  const int i0 = I * OZ_T + (sb & 3) * 32, j0 = J * OZ_T + (sb >> 2) * 32;
  if (i0 > j0 || i0 >= ngp || j0 >= ngp) return;  // below the diagonal or outside
  constexpr int NV = ONLY_O ? 1 : 2;              // matrices
  __shared__ double2 sT[NV][32][33];
  const int tid = threadIdx.x, lane = tid & 63, h = tid >> 6;
  const int il = 8 * h + 4 * (lane >> 5), jl = lane & 31;
  const size_t plane = (size_t)T.n * (OZ_T * OZ_T);
  const EXH_G int8_t *r0 = gptr((const int8_t *)d.r) + (size_t)(tile - T.t0) * (OZ_T * OZ_T) + sb * 1024 + tid * 4;

  double rh[NV][4], rl[NV][4], mh[NV][4], ml[NV][4];
#pragma unroll
  for (int v = 0; v < NV; v++)
#pragma unroll
    for (int t = 0; t < 4; t++) rh[v][t] = rl[v][t] = mh[v][t] = ml[v][t] = 0.0;
  const OzCrt &C = c_crt.t[NM];
#pragma unroll
  for (int k = 0; k < NM; k++)
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const int wp = *(const EXH_G int *)(r0 + (size_t)((2 * v) * NM + k) * plane);
      const int wm = *(const EXH_G int *)(r0 + (size_t)((2 * v + 1) * NM + k) * plane);
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const int a = byte_of(wp, t), b = byte_of(wm, t);
        const double s = (double)(a + b), f = (double)(a - b);
        rh[v][t] = fma(s, C.reh[k], rh[v][t]);
        rl[v][t] = fma(s, C.rel[k], rl[v][t]);
        mh[v][t] = fma(f, C.imh[k], mh[v][t]);
        ml[v][t] = fma(f, C.iml[k], ml[v][t]);
      }
    }

  const int j = j0 + jl;
  if (j < ngp) {
    const int ebj = ONLY_O ? 0 : eb[j], eyj = ey[j];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const int i = i0 + il + t;
      if (i >= ngp || i > j) continue;
      auto value = [&](int v, int exi, int ej) {
        // 2^-(s_i + s_j); a column that is not finite makes the element NaN
        const bool bad = exi == INT_MAX || ej == INT_MAX;
        const int si = exi == INT_MIN ? 0 : bits - exi, sj = ej == INT_MIN ? 0 : bits - ej;
        const int sh = bad ? 0 : -(si + sj);
        const double nan = __builtin_nan("");
        const double re = ldexp(crt<NM>(rh[v][t], rl[v][t]), sh);
        const double im = ldexp(crt<NM>(mh[v][t], ml[v][t]), sh);
        return bad ? z2(nan, nan) : z2(re, im);
      };
      double2 hv = z2(0.0, 0.0), ov = value(NV - 1, ex[i], eyj);
      if (!ONLY_O) hv = value(0, ea[i], ebj);
      ist_add(box, i, j, hv.x, hv.y, ov.x, ov.y);
      if (!ONLY_O) sT[0][jl][il + t] = hv;
      sT[NV - 1][jl][il + t] = ov;
    }
  }
  __syncthreads();
  const int lo = tid & 31, hi8 = tid >> 5;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int c = hi8 + 8 * r, i = i0 + lo, jj = j0 + c;
    if (i >= ngp || jj >= ngp || i > jj) continue;
    const size_t up = (size_t)i + (size_t)jj * ldh;
#pragma unroll
    for (int v = 0; v < NV; v++) {
      EXH_G double2 *M = (!ONLY_O && v == 0) ? H : O;
      double2 x = sT[v][c][lo];
      if (accumulate) {
        const double2 old = ld(M + up);
        x.x += old.x;
        x.y += old.y;
        sT[v][c][lo] = x;
      }
      st(M + up, x);
    }
  }
  if (accumulate) __syncthreads();
  // lower triangle: element (j, i) = conj(upper (i, j)), i < j
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int c = hi8 + 8 * r, jj = j0 + lo, i = i0 + c;
    if (i >= ngp || jj >= ngp || i >= jj) continue;
    const size_t lw = (size_t)jj + (size_t)i * ldh;
#pragma unroll
    for (int v = 0; v < NV; v++) {
      EXH_G double2 *M = (!ONLY_O && v == 0) ? H : O;
      const double2 x = sT[v][lo][c];
      st(M + lw, z2(x.x, -x.y));
    }
  }
}

// Single launches take the k-point by value, grouped ones an array of them;
// blockIdx.z (with the operand) or blockIdx.y selects it.
__global__ __launch_bounds__(256) void colnorm_part_kernel(OzK d) {
  colnorm_part_body(d, blockIdx.z);
}
__global__ __launch_bounds__(256) void colnorm_part_grouped_kernel(const OzK *__restrict__ kd,
                                                                   int nops) {
  colnorm_part_body(kd[blockIdx.z / nops], blockIdx.z % nops);
}
__global__ __launch_bounds__(256) void colnorm_final_kernel(OzK d) {
  colnorm_final_body(d, blockIdx.z);
}
__global__ __launch_bounds__(256) void colnorm_final_grouped_kernel(const OzK *__restrict__ kd,
                                                                   int nops) {
  colnorm_final_body(kd[blockIdx.z / nops], blockIdx.z % nops);
}
// X' comes with X (the column is in the cache), or in the launch of H's operands
// where they are apart.  With equal row exponents X' and X have the same residues:
// one is enough.
__device__ __forceinline__ void residues_of(const OzK &d, int z, int m0, int m1) {
  const bool apart = d.qi[d.iA] == d.qi[d.iX], uni = d.uni && *d.uni;
  if (uni && apart && z == d.iX) return;  // X' lies there
  // the operand with scaled rows, if any, then the one without
  const int zs = uni || !d.uni ? -1 : d.rs[z] ? z : z == d.iX && !apart ? d.iA : -1;
  if (zs >= 0) residue_body<true>(d, zs, m0, m1);
  if (zs != z) residue_body<false>(d, z, m0, m1);
}
__global__ __launch_bounds__(256) void residue_kernel(OzK d, int z0, int m0, int m1) {
  residues_of(d, z0 + blockIdx.z, m0, m1);
}
__global__ __launch_bounds__(256) void residue_grouped_kernel(const OzK *__restrict__ kd, int z0,
                                                              int nz, int m1) {
  residues_of(kd[blockIdx.z / nz], z0 + blockIdx.z % nz, 0, m1);
}
// two waves per SIMD whatever the workgroup size: at most 256 VGPRs
__global__ __launch_bounds__(64 * OZ_NWG) __attribute__((amdgpu_waves_per_eu(2, 2))) void
ozgemm_kernel(OzK d, int m0, int mc, int s0, int s1) {
  __shared__ v4i sm0[4][OZ_W], sm1[4][OZ_W];
  ozgemm_body<false>(d, m0, mc, s0, s1, 0, 1, false, sm0, sm1);
}
__global__ __launch_bounds__(64 * OZ_NWG) __attribute__((amdgpu_waves_per_eu(2, 2))) void
ozgemm_grouped_kernel(const OzK *__restrict__ kd, int mc) {
  __shared__ v4i sm0[4][OZ_W], sm1[4][OZ_W];
  ozgemm_body<false>(kd[blockIdx.y], 0, mc, 0, INT_MAX / 2, 0, 1, false, sm0, sm1);
}
// FP64: steps of two blocks of one matrix, or, where the row exponents are equal
// and O's columns are there beside H's, of one block of both as with EXH_SPLIT
// (at 16 atoms, 148 against 135 workgroups a product pair).
__device__ __forceinline__ void ozgemm64_body(const OzK &d, int m0, int mc, int s0, int s1,
                                              int mat0, int nmat) {
  __shared__ v4i sm0[4][OZ_W], sm1[4][OZ_W];
  const bool uni = d.uni && *d.uni;
  if (uni && (d.qi[d.iB] != d.qi[d.iY])) {
    if (mat0 == 0) ozgemm_body<false>(d, m0, mc, 2 * s0, 2 * s1, 0, 1, true, sm0, sm1);
    return;
  }
  ozgemm_body<true>(d, m0, mc, s0, s1, mat0, nmat, uni, sm0, sm1);
}
__global__ __launch_bounds__(64 * OZ_NWG) __attribute__((amdgpu_waves_per_eu(2, 2))) void
ozgemm64_kernel(OzK d, int m0, int mc, int s0, int s1, int mat0, int nmat) {
  ozgemm64_body(d, m0, mc, s0, s1, mat0, nmat);
}
__global__ __launch_bounds__(64 * OZ_NWG) __attribute__((amdgpu_waves_per_eu(2, 2))) void
ozgemm64_grouped_kernel(const OzK *__restrict__ kd, int mc) {
  ozgemm64_body(kd[blockIdx.y], 0, mc, 0, INT_MAX / 4, 0, 2);
}
template <int NM, bool ONLY_O>
__global__ __launch_bounds__(256) void ozcombine_kernel(OzK d, int accumulate, int s0, int s1) {
  ozcombine_body<NM, ONLY_O>(d, accumulate, s0, s1);
}
template <int NM>
__global__ __launch_bounds__(256) void ozcombine_grouped_kernel(const OzK *__restrict__ kd,
                                                                int accumulate) {
  ozcombine_body<NM, false>(kd[blockIdx.y], accumulate, 0, INT_MAX / 2);
}

inline unsigned cdiv(long long a, long long b) { return (unsigned)((a + b - 1) / b); }

// EXH_SPLIT(n) rounds to the c bits that the product of the n largest primes
// <= 251 would allow, whatever moduli recover the products.
constexpr int kPrimes[kOzMaxMod] = {251, 241, 239, 233, 229, 227, 223, 211, 199, 197, 193, 191};

}  // namespace

OzPlan oz_split(int n) {
  double lm = 0.0;
  for (int k = 0; k < n; k++) lm += std::log2((double)kPrimes[k]);
  // the largest c with 2^(2c) < prod/2 (a hair below guards the log2)
  OzPlan P;
  P.split = true;
  P.bits = (int)std::min(50.0, std::floor((lm - 1.0) * 0.5 - 1e-9));
  // the scaled columns' norms are below 2^(c-1) + sqrt(2K)/2, so the products
  // need prod(p) > 2^(2c-1) (1 + 2^-13 at c = 23)
  double need = 2.0 * P.bits - 1.0 + 1e-3;
  for (P.nmod = 0; need > 0.0; P.nmod++) need -= std::log2((double)kP[P.nmod]);
  return P;
}

// c = 56: norms below 2^55, products below 2^110 < 0.47 prod(p) = 2^111.09.
OzPlan oz_fp64() {
  OzPlan P;
  P.bits = 56;
  P.nmod = OZ_N;
  return P;
}

OzLayout oz_layout(const exh_context *c, const OzPlan &P, bool only_o) {
  return oz_layout_ops(c, P, only_o, P.split ? 2 : 1 + (only_o ? 0 : 2) + (c->have_h1aa ? 1 : 0));
}

OzLayout oz_layout_ops(const exh_context *c, const OzPlan &P, bool only_o, int nops) {
  OzLayout L;
  const int ngkmax = c->ngkmax, Ktot = c->Ktot;
  L.Gpad = (ngkmax + OZ_T - 1) / OZ_T * OZ_T;
  L.Kpad = (Ktot + 2 * OZ_KS - 1) / (2 * OZ_KS) * (2 * OZ_KS);  // an even number of stages
  L.qstride = (size_t)L.Kpad * L.Gpad;
  const int nt = (ngkmax + OZ_T - 1) / OZ_T;  // tile columns of the largest basis
  L.nt = nt;
  L.width = P.split ? 1 : 2;
  L.planes = (only_o ? 2 : 4) * P.nmod;
  L.full = {P.nmod, std::max(1, P.split ? oz_steps<false>(nt) : oz_steps<true>(nt))};
  // per operand: the column exponents, then the partial norms and their marks
  const size_t ng = std::max(ngkmax, 1);
  const int rows = (c->maxaa + kNormRows - 1) / kNormRows;
  L.nch = std::max((Ktot + OZ_NCH - 1) / OZ_NCH, c->natmtot * rows);
  L.e_part_off = (ng * sizeof(int) + 255) / 256 * 256;
  L.e_bytes = (L.e_part_off + (sizeof(double) + sizeof(int)) * L.nch * ng + 255) / 256 * 256;
  L.nops = nops;
  L.panels = 2 * P.nmod * (P.split ? oz_panels<false>(nt, 0, nt) : oz_panels<true>(nt, 0, nt));
  // one matrix's products fill the chip for 32 rounds: the other's residues can
  // take their place afterwards
  L.apart = !P.split && !only_o && L.panels >= 8192;
  if (!P.split && !only_o) L.panels *= 2;
  return L;
}

// The largest part of the products that fits in `bytes` (chunk = 0: none).
// Fewer moduli at a time cost a pass over the operands each; fewer column
// steps cost nothing while the residues of every modulus are there, and
// otherwise all of those passes again, so they come last.
OzFit oz_fit(const OzLayout &L, size_t bytes) {
  auto even = [](int n, int most) {  // n in equal parts of at most `most`
    const int parts = (n + most - 1) / most;
    return (n + parts - 1) / parts;
  };
  auto chunks = [&](size_t room) {
    return (int)std::min<size_t>(L.full.chunk, room / std::max<size_t>(L.q_bytes(1), 1));
  };
  const size_t r = L.r_bytes(L.full.steps);
  OzFit f = L.full;
  if (L.slot_bytes(f) <= bytes) return f;
  if (r < bytes && (f.chunk = chunks(bytes - r)) > 0) {
    f.chunk = even(L.full.chunk, f.chunk);
    return f;
  }
  const int eighth = std::max(1, L.full.steps / 8);
  f.chunk = L.slot_bytes({L.full.chunk, eighth}) <= bytes ? L.full.chunk : 1;
  for (f.steps = L.full.steps; f.steps > 0 && L.slot_bytes(f) > bytes;) f.steps--;
  if (f.steps == 0) return OzFit();
  f.steps = even(L.full.steps, f.steps);
  return f;
}

// bt sums the norms of H's operands and, in passing, of O's X.
NormOut norm_out(const OzK &d) {
  NormOut n;
  n.x = d.part[d.iX];
  n.b = d.part[d.iB];
  if (d.iA != d.iX) {
    n.xs = d.part[d.iA];
    n.rexp = d.rexp;
    n.uni = d.uni;
  }
  n.ld = d.ldp;
  n.nx = d.nch[d.iX];
  n.nb = d.nch[d.iB];
  return n;
}

OzK make_ozk(const exh_context *c, int ngp, const OzPlan &P, const OzLayout &L,
             const OzScratch &w, const double2 *X, long long ldx, const double2 *B,
             const double2 *Y, long long ldb, const IstBox &box, double2 *h, double2 *o,
             int ldh) {
  OzK d{};
  d.ngp = ngp;
  d.Ktot = c->Ktot;
  d.nt = (ngp + OZ_T - 1) / OZ_T;
  d.nslab = L.Kpad / OZ_KS;
  d.Gpad = L.Gpad;
  d.nmod = P.nmod;
  d.bits = P.bits;
  d.ldp = std::max(c->ngkmax, 1);
  d.qstride = L.qstride;
  d.q_bytes = w.fit.chunk * 2 * L.qstride;
  d.rexp = (const int *)c->rexp.p;
  d.uni = h && !P.split ? d.rexp + 3 * (size_t)c->Ktot : nullptr;
  d.q = w.q;
  d.r = w.r;
  d.box = box;
  d.h = h;
  d.o = o;
  d.ldh = ldh;
  const int rows = (c->maxaa + kNormRows - 1) / kNormRows;
  // nch 0: not among bt's norms
  auto add = [&](const double2 *x, long long ld, int rs, int nch) {
    const int n = d.nops++;
    char *e = (char *)w.e + (size_t)n * L.e_bytes;
    d.fused |= nch ? 1u << n : 0u;
    d.nch[n] = nch ? nch : (c->Ktot + OZ_NCH - 1) / OZ_NCH;
    d.x[n] = x;
    d.ld[n] = ld;
    d.rs[n] = rs;
    d.qi[n] = L.apart && n >= 2 ? n - 2 : n;
    d.e[n] = (int *)e;
    d.part[n] = (double *)(e + L.e_part_off);
    return n;
  };
  if (h) {
    d.iA = add(X, ldx, P.split ? 0 : 1, c->natmtot);
    d.iB = add(B, ldb, P.split ? 0 : -1, c->natmtot * rows);
  }
  d.iX = h && P.split ? d.iA : add(X, ldx, 0, h ? c->natmtot : 0);
  d.iY = Y ? add(Y, ldb, 0, 0) : d.iX;
  return d;
}

// One k-point (kd null: by value from d) or the n k-points d[0..n) that kd
// holds in device memory; grouped ones have room for everything at once.
static hipError_t launch_oz(hipStream_t s, const OzK *d, const OzK *kd, int n, const OzFit &fit,
                            int accumulate, const OzRun &run) {
  const bool only_o = d[0].h == nullptr;
  const int nmod = d[0].nmod;
  const bool one = nmod == OZ_N;  // FP64: one matrix per workgroup
  const bool apart = d[0].nops > 2 && d[0].qi[2] == 0;
  int ngp = 0, nch = 0, nops = 0, kb = 0, nt = 0;
  for (int i = 0; i < n; i++) {
    ngp = std::max(ngp, d[i].ngp);
    nops = std::max(nops, d[i].nops);
    for (int z = 0; z < d[i].nops; z++)  // chunks of operands bt has not summed
      if (!(d[i].fused >> z & 1)) nch = std::max(nch, d[i].nch[z]);
    kb = std::max(kb, d[i].nslab * (OZ_KS / 16));
    nt = std::max(nt, d[i].nt);
  }
  if (ngp <= 0) return hipSuccess;
  const unsigned nz = (unsigned)(nops * n);
  auto norms = [&] {
    const dim3 gp(cdiv(ngp, 64), nch, nz), gf(cdiv(ngp, 64), 1, nz);
    if (kd) {
      if (nch) hipLaunchKernelGGL(colnorm_part_grouped_kernel, gp, dim3(256), 0, s, kd, nops);
      hipLaunchKernelGGL(colnorm_final_grouped_kernel, gf, dim3(256), 0, s, kd, nops);
    } else {
      if (nch) hipLaunchKernelGGL(colnorm_part_kernel, gp, dim3(256), 0, s, d[0]);
      hipLaunchKernelGGL(colnorm_final_kernel, gf, dim3(256), 0, s, d[0]);
    }
  };
  auto residues = [&](int z0, int z1, int m0, int m1) {
    const dim3 gr(cdiv(nt * OZ_T, 256), kb, (z1 - z0) * n);
    if (kd) hipLaunchKernelGGL(residue_grouped_kernel, gr, dim3(256), 0, s, kd, z0, z1 - z0, m1);
    else hipLaunchKernelGGL(residue_kernel, gr, dim3(256), 0, s, d[0], z0, m0, m1);
  };
  auto products = [&](int m0, int m1, int s0, int s1, int mat0, int nmat) {
    const int mc = m1 - m0;
    long long nb = one ? oz_panels<true>(nt, s0, s1) * nmat : oz_panels<false>(nt, s0, s1);
    if (one && !only_o) nb = std::max(nb, oz_panels<false>(nt, 2 * s0, 2 * s1));
    const dim3 gg((unsigned)((nb * 2 * mc + 7) / 8 * 8), n), th(64 * OZ_NWG);
    if (kd && one) hipLaunchKernelGGL(ozgemm64_grouped_kernel, gg, th, 0, s, kd, mc);
    else if (kd) hipLaunchKernelGGL(ozgemm_grouped_kernel, gg, th, 0, s, kd, mc);
    else if (one)
      hipLaunchKernelGGL(ozgemm64_kernel, gg, th, 0, s, d[0], m0, mc, s0, s1, mat0, nmat);
    else
      hipLaunchKernelGGL(ozgemm_kernel, gg, th, 0, s, d[0], m0, mc, s0, s1);
  };
  auto combine = [&](int s0, int s1) {
    const OzTiles T = one ? oz_tiles<true>(nt, s0, s1) : oz_tiles<false>(nt, s0, s1);
    const dim3 grid((unsigned)T.n * 16, n);
    if (only_o) {
      if (nmod != OZ_N) return hipErrorInvalidValue;  // EXH_SPLIT is refused for O alone
      hipLaunchKernelGGL((ozcombine_kernel<OZ_N, true>), grid, dim3(256), 0, s, d[0], accumulate,
                         s0, s1);
      return hipGetLastError();
    }
#define EXH_OZC(N)                                                                              \
  case N:                                                                                       \
    if (kd)                                                                                     \
      hipLaunchKernelGGL(ozcombine_grouped_kernel<N>, grid, dim3(256), 0, s, kd, accumulate);   \
    else                                                                                        \
      hipLaunchKernelGGL((ozcombine_kernel<N, false>), grid, dim3(256), 0, s, d[0], accumulate, \
                         s0, s1);                                                               \
    break;
    switch (nmod) {
      EXH_OZC(6)
      EXH_OZC(7)
      EXH_OZC(8)
      EXH_OZC(9)
      EXH_OZC(10)
      EXH_OZC(11)
      EXH_OZC(13)  // EXH_SPLIT(12)
      EXH_OZC(OZ_N)
      default:
        return hipErrorInvalidValue;
    }
#undef EXH_OZC
    return hipGetLastError();
  };
  // operands and matrices whose residues are there together
  struct Pass {
    int z0, z1, mat0, nmat;
  };
  const bool both = one && !only_o;  // X' comes with X
  const Pass all[1] = {{both ? 1 : 0, nops, only_o ? 1 : 0, both ? 2 : 1}};
  const Pass two[2] = {{0, 2, 0, 1}, {2, nops, 1, 1}};
  const Pass *ps = apart ? two : all;
  const int np = apart ? 2 : 1, ns = one ? oz_steps<true>(nt) : oz_steps<false>(nt);
  hipError_t e = hipSuccess;
  for (int s0 = 0; s0 < ns && e == hipSuccess; s0 += fit.steps) {
    const int s1 = std::min(ns, s0 + fit.steps);
    for (int m0 = 0; m0 < nmod && e == hipSuccess; m0 += fit.chunk)
      for (int p = 0; p < np && e == hipSuccess; p++) {
        const int m1 = std::min(nmod, m0 + fit.chunk);
        // residues that an earlier strip has left are still there
        if (s0 == 0 || fit.chunk < nmod || np > 1)
          e = run(EXH_K_OZRES, [&] {
            if (s0 == 0 && m0 == 0 && p == 0) norms();
            residues(ps[p].z0, ps[p].z1, m0, m1);
            return hipGetLastError();
          });
        if (e == hipSuccess)
          e = run(EXH_K_OZGEMM, [&] {
            products(m0, m1, s0, s1, ps[p].mat0, ps[p].nmat);
            return hipGetLastError();
          });
      }
    if (e == hipSuccess) e = run(EXH_K_OZCOMB, [&] { return combine(s0, s1); });
  }
  return e;
}

hipError_t launch_ozaki(hipStream_t s, const OzK &d, const OzFit &fit, int accumulate,
                        const OzRun &run) {
  return launch_oz(s, &d, nullptr, 1, fit, accumulate, run);
}

hipError_t launch_ozaki_grouped(hipStream_t s, const OzK *d, const OzK *kd, int n, int accumulate,
                                const OzRun &run) {
  return launch_oz(s, d, kd, n, {d[0].nmod, INT_MAX / 2}, accumulate, run);
}

}  // namespace exh
