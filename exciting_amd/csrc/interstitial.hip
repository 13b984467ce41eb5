// Interstitial producers on the device: the smooth step function
// (gencfun.f90:13-159), the G components of the effective potential and
// masses (genveffig.f90:13-44, genmeffig.f90:13-61), and the device form of
// exh_set_interstitial.  The closed form, the grid products and the
// grid <-> G maps are kernels of this file; the 3-D transforms are hipFFT
// double-complex plans, batched over the products of one call.
//
// Grid layout: the FFT box of ngrid(1) x ngrid(2) x ngrid(3) points with the
// first index fastest (zfftifc.f90 / genigfft in gengvec.f90:129-167): the G
// vector with integer coordinates (i1,i2,i3) sits at
//   j = j3*n1*n2 + j2*n1 + j1,   j_d = i_d (i_d >= 0) or n_d + i_d,
// which is hipFFT's row-major layout with dimensions (n3, n2, n1).
#include <hipfft/hipfft.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "exh_device.h"

namespace exh {
namespace {

constexpr double kFourPi = 12.566370614359172954;
constexpr double kAlpha = 1.0 / 137.03599911;  // genmeffig.f90:29

// Per-call constants of the closed form.
struct CfunArgs {
  double b[9];   // bvec, column-major (b1, b2, b3)
  double t1;     // 4 pi / omega (gencfun.f90:120)
  double epslat;
  double damp;   // cfdamp / gmaxvr, 0 = no damping
  int n1, n2, n3;
  int lo[3];    // the box holds i_d = lo_d .. lo_d + n_d - 1
  int off[3];   // -lo_d mod n_d
  int nspecies;
};

// position in the box of FFT index j along one axis
__device__ __forceinline__ int box_index(int j, int off, int n) {
  return j + off < n ? j + off : j + off - n;
}

// Phase tables of gencfun.f90:150-155: exp(-i G.tau) is the product over the
// three axes of exp(-i i_d b_d.tau), so the sine and cosine are taken for
// natm (n1 + n2 + n3) arguments instead of natm n1 n2 n3.  tab[atom][j], j the
// FFT index along axis 1, then 2, then 3.  The argument is held in two words
// (b_d.tau to twice the working precision, then the integer multiple), so that
// an entry is good to an ulp however large the phase is.
__global__ __launch_bounds__(256) void phase_table_kernel(CfunArgs a, int natm,
                                                          const double *__restrict__ geo,
                                                          double2 *__restrict__ tab) {
  const int nt = a.n1 + a.n2 + a.n3, e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= natm * nt) return;
  const int ia = e / nt, j = e - ia * nt;
  const int d = j < a.n1 ? 0 : j < a.n1 + a.n2 ? 1 : 2;
  const int n = d == 0 ? a.n1 : d == 1 ? a.n2 : a.n3;
  const int jd = j - (d == 0 ? 0 : d == 1 ? a.n1 : a.n1 + a.n2);
  const double i = a.lo[d] + box_index(jd, a.off[d], n);
  const double *tau = geo + 3 * a.nspecies + 3 * ia;
  double hi = 0.0, low = 0.0;   // b_d . tau
  for (int k = 0; k < 3; k++) {
    const double p = a.b[3 * d + k] * tau[k], ep = fma(a.b[3 * d + k], tau[k], -p);
    const double s = hi + p, v = s - hi;
    low += (hi - (s - v)) + (p - v) + ep;
    hi = s;
  }
  const double ph = i * hi, dl = fma(i, hi, -ph) + i * low;
  double s, c;
  sincos(ph, &s, &c);
  tab[e] = make_double2(c - s * dl, -(s + c * dl));
}

// gencfun.f90:120-157, then :70 (the undamped value at its grid point) and
// :76-82 (damping of cfunig).  One thread per (j1, j2) of the grid and kRows
// consecutive j3: per atom the phase of (j1, j2) is formed once, and each row
// costs one complex multiply-add with a factor that the whole wave shares.
// geo holds per species {rmt, first atom, end atom}, then the positions.
// Per grid point and atom 4 FMA and 4/kRows (10 us for 64 atoms on 80^3), bound
// by the latency of the tables' loads at two waves per SIMD: 93 us with a sincos
// per G vector and atom, 34 now with 2 to 4 rows, 44 with 8; error of cfunig
// against extended precision 4.7e-15 -> 3e-17 (relative norm).
constexpr int kRows = 4;
__global__ __launch_bounds__(256) void cfunig_kernel(CfunArgs a, const int *__restrict__ ivgig,
                                                     const double *__restrict__ geo,
                                                     const double2 *__restrict__ tab,
                                                     double2 *__restrict__ cfunig,
                                                     double2 *__restrict__ zfft) {
  const int plane = a.n1 * a.n2, q = blockIdx.x * blockDim.x + threadIdx.x;
  const int j30 = blockIdx.y * kRows, nt = a.n1 + a.n2 + a.n3;
  if (q >= plane) return;
  const int j2 = q / a.n1, j1 = q - j2 * a.n1;
  const int b1 = box_index(j1, a.off[0], a.n1), b2 = box_index(j2, a.off[1], a.n2);
  const int i1 = a.lo[0] + b1, i2 = a.lo[1] + b2;
  double gc[kRows], re[kRows], im[kRows];
#pragma unroll
  for (int r = 0; r < kRows; r++) {
    const int i3 = a.lo[2] + box_index(min(j30 + r, a.n3 - 1), a.off[2], a.n3);
    double v[3];
#pragma unroll
    for (int d = 0; d < 3; d++)
      v[d] = (double)i1 * a.b[d] + (double)i2 * a.b[3 + d] + (double)i3 * a.b[6 + d];
    gc[r] = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    re[r] = gc[r] > a.epslat ? 0.0 : 1.0;
    im[r] = 0.0;
  }
  for (int is = 0; is < a.nspecies; is++) {
    const double rmt = geo[3 * is];
    const int ia0 = (int)geo[3 * is + 1], ia1 = (int)geo[3 * is + 2];
    if (ia0 == ia1) continue;
    double sr[kRows] = {}, si[kRows] = {};
    for (int ia = ia0; ia < ia1; ia++) {
      const double2 *t = tab + (size_t)ia * nt;
      const double2 x = t[j1], y = t[a.n1 + j2];
      const double px = x.x * y.x - x.y * y.y, py = x.x * y.y + x.y * y.x;
#pragma unroll
      for (int r = 0; r < kRows; r++) {
        const double2 z = t[a.n1 + a.n2 + min(j30 + r, a.n3 - 1)];
        sr[r] += px * z.x - py * z.y;
        si[r] += px * z.y + py * z.x;
      }
    }
#pragma unroll
    for (int r = 0; r < kRows; r++) {
      double ff;
      if (gc[r] > a.epslat) {
        const double t2 = gc[r] * rmt;
        double s, c;
        sincos(t2, &s, &c);
        ff = a.t1 * (s - t2 * c) / (gc[r] * gc[r] * gc[r]);
      } else {
        ff = a.t1 / 3.0 * rmt * rmt * rmt;
      }
      re[r] -= ff * sr[r];
      im[r] -= ff * si[r];
    }
  }
#pragma unroll
  for (int r = 0; r < kRows; r++) {
    const int j3 = j30 + r;
    if (j3 >= a.n3) break;
    zfft[(size_t)j3 * plane + q] = make_double2(re[r], im[r]);
    if (a.damp > 0.0) {
      const double t = a.damp * gc[r], f = exp(-t * t);
      re[r] *= f;
      im[r] *= f;
    }
    const int b3 = box_index(j3, a.off[2], a.n3);
    cfunig[ivgig[b1 + (size_t)a.n1 * (b2 + (size_t)a.n2 * b3)] - 1] = make_double2(re[r], im[r]);
  }
}

// gencfun.f90:74: cfunir = Re(zfft).
__global__ __launch_bounds__(256) void real_part_kernel(int n, const double2 *__restrict__ z,
                                                        double *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = z[i].x;
}

// genveffig.f90:33 and genmeffig.f90:38,50: the selected products, stored as
// consecutive real grids of n values in the order veff, meff, m2eff.
__global__ __launch_bounds__(256) void products_kernel(int n, const double *__restrict__ veffir,
                                                       const double *__restrict__ cfunir,
                                                       int which, double a2,
                                                       double *__restrict__ z) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double v = veffir[i], c = cfunir[i];
  double *p = z + i;
  if (which & EXH_VEFFIG) {
    *p = v * c;
    p += n;
  }
  if (which & (EXH_MEFFIG | EXH_M2EFFIG)) {
    const double d = 1.0 - v * a2;
    if (which & EXH_MEFFIG) {
      *p = c / d;
      p += n;
    }
    if (which & EXH_M2EFFIG) *p = c / (d * d);
  }
}

// genveffig.f90:36-39 (and genmeffig.f90:41-44, :53-56): out_b(ig) = the
// forward transform at G's grid point, times the 1/N of zfftifc.f90:70-77.
// The grids are real, so only j1 <= n1 / 2 is transformed: the other half is
// the conjugate at -j (mod n).  Two products of 80^3: 42 us as complex
// transforms, 32 so, at the same error (2e-16, relative norm).
__global__ __launch_bounds__(256) void gather_kernel(int ngvec, const int *__restrict__ ivg,
                                                     int n1, int n2, int n3, int nb,
                                                     const double2 *__restrict__ z, double scale,
                                                     double2 *o0, double2 *o1, double2 *o2) {
  const int ig = blockIdx.x * blockDim.x + threadIdx.x;
  if (ig >= ngvec) return;
  const int i1 = ivg[3 * ig], i2 = ivg[3 * ig + 1], i3 = ivg[3 * ig + 2];
  int j1 = i1 >= 0 ? i1 : n1 + i1, j2 = i2 >= 0 ? i2 : n2 + i2, j3 = i3 >= 0 ? i3 : n3 + i3;
  const int h1 = n1 / 2 + 1;
  double sy = scale;
  if (j1 >= h1) {
    j1 = n1 - j1;
    j2 = j2 ? n2 - j2 : 0;
    j3 = j3 ? n3 - j3 : 0;
    sy = -scale;
  }
  const size_t n = (size_t)h1 * n2 * n3, j = ((size_t)j3 * n2 + j2) * h1 + j1;
  double2 *outs[3] = {o0, o1, o2};
  for (int b = 0; b < nb; b++) {
    const double2 x = z[b * n + j];
    outs[b][ig] = make_double2(x.x * scale, x.y * sy);
  }
}

int cdiv_i(long long a, int b) { return (int)((a + b - 1) / b); }

void grid_of(const exh_context *c, int *n) {
  for (int d = 0; d < 3; d++) n[d] = c->intgv[3 + d] - c->intgv[d] + 1;
}

// The producers transform the whole G box: every box point is one G vector
// (checked by exh_set_gvectors), so the scatter fills the whole grid and
// every kernel index below stays inside it.
int check_grid(exh_context *c, const char *who) {
  if (!c->have_gvec) return fail(c, EXH_ESTATE, std::string(who) + ": call exh_set_gvectors first");
  if (!c->gvec_full)
    return fail(c, EXH_EINVAL,
                std::string(who) + ": the G set is not the whole FFT grid of the G box "
                                   "(ngrtot = box size, ivgig the inverse of ivg)");
  return 0;
}

const char *fft_error(hipfftResult r) {
  switch (r) {
    case HIPFFT_ALLOC_FAILED: return "allocation failed";
    case HIPFFT_INVALID_VALUE: return "invalid value";
    case HIPFFT_INVALID_SIZE: return "invalid size";
    case HIPFFT_EXEC_FAILED: return "execution failed";
    case HIPFFT_SETUP_FAILED: return "setup failed";
    default: return "error";
  }
}

// Plan over the context's grid: nb = 0 the in-place double-complex transform of
// one grid, nb > 0 the forward transform of nb real grids.
int fft_plan(exh_context *c, int nb, hipfftHandle *out) {
  int n[3];
  grid_of(c, n);
  if (std::memcmp(n, c->fft_grid, sizeof(n)) != 0) {
    interstitial_release(c);
    std::memcpy(c->fft_grid, n, sizeof(n));
  }
  if (!c->fft_plan[nb]) {
    hipfftHandle h = nullptr;
    int dims[3] = {n[2], n[1], n[0]};
    const int dist = c->ngrtot, odist = nb ? (n[0] / 2 + 1) * n[1] * n[2] : dist;
    hipfftResult r = hipfftPlanMany(&h, 3, dims, nullptr, 1, dist, nullptr, 1, odist,
                                    nb ? HIPFFT_D2Z : HIPFFT_Z2Z, std::max(nb, 1));
    if (r != HIPFFT_SUCCESS)
      return fail(c, EXH_ESTATE, std::string("hipfftPlanMany: ") + fft_error(r));
    c->fft_plan[nb] = (void *)h;
  }
  *out = (hipfftHandle)c->fft_plan[nb];
  return 0;
}

// nb = 0: z in place, to the grid; nb > 0: the real grids x into z
int run_fft(exh_context *c, hipStream_t s, int nb, double *x, double2 *z) {
  hipfftHandle h;
  if (int rc = fft_plan(c, nb, &h)) return rc;
  hipfftResult r = hipfftSetStream(h, s);
  hipError_t e = timed(c, EXH_K_IFFT, s, [&] {
    if (r == HIPFFT_SUCCESS)
      r = nb ? hipfftExecD2Z(h, x, (hipfftDoubleComplex *)z)
             : hipfftExecZ2Z(h, (hipfftDoubleComplex *)z, (hipfftDoubleComplex *)z,
                             HIPFFT_BACKWARD);
    return hipSuccess;
  });
  if (r != HIPFFT_SUCCESS) return fail(c, EXH_ESTATE, std::string("hipfftExec: ") + fft_error(r));
  return e == hipSuccess ? 0 : hip_fail(c, e, "fft");
}

// The geometry goes to the device as kernel arguments, kGeoWords at a time: a
// copy from the caller's memory would have to be waited for.
constexpr int kGeoWords = 384;
struct GeoWords {
  double v[kGeoWords];
};
__global__ __launch_bounds__(kGeoWords) void put_words_kernel(GeoWords g, int n,
                                                              double *__restrict__ out) {
  if ((int)threadIdx.x < n) out[threadIdx.x] = g.v[threadIdx.x];
}

template <typename T>
int copy_in(exh_context *c, DevBuf &b, const T *src, size_t n) {
  int rc = ensure(c, b, n * sizeof(T));
  if (rc) return rc;
  hipError_t e = hipMemcpyAsync(b.p, src, n * sizeof(T), hipMemcpyHostToDevice, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  return e == hipSuccess ? 0 : hip_fail(c, e, "upload");
}

int copy_out(exh_context *c, void *dst, const DevBuf &b, size_t bytes) {
  hipError_t e = hipMemcpyAsync(dst, b.p, bytes, hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  return e == hipSuccess ? 0 : hip_fail(c, e, "download");
}

}  // namespace

void interstitial_release(exh_context *c) {
  for (int b = 0; b < 4; b++) {
    if (c->fft_plan[b]) (void)hipfftDestroy((hipfftHandle)c->fft_plan[b]);
    c->fft_plan[b] = nullptr;
  }
  std::memset(c->fft_grid, 0, sizeof(c->fft_grid));
}

}  // namespace exh

using namespace exh;

extern "C" {

int exh_gencfun_device(exh_context *c, void *stream, const double *bvec, const double *atposc,
                       int maxatoms, double epslat, double cfdamp, double gmaxvr,
                       exh_z *cfunig, double *cfunir) {
  if (!c) return EXH_EINVAL;
  if (int rc = wait_done(c)) return rc;
  if (int rc = check_grid(c, "gencfun")) return rc;
  if (!c->have_basis || !c->have_radial)
    return fail(c, EXH_ESTATE, "gencfun: basis and radial data not set");
  if (!bvec || !cfunig || !cfunir || (c->natmtot > 0 && !atposc))
    return fail(c, EXH_EINVAL, "gencfun: null array");
  if (!(epslat >= 0.0) || (cfdamp > 0.0 && !(gmaxvr > 0.0)))
    return fail(c, EXH_EINVAL, "gencfun: epslat < 0, or cfdamp > 0 with gmaxvr <= 0");
  int maxna = 0;
  for (int is = 0; is < c->nspecies; is++) maxna = std::max(maxna, c->natoms[is]);
  if (maxatoms < maxna) return fail(c, EXH_EINVAL, "gencfun: maxatoms below natoms");
  if (hipSetDevice(c->device) != hipSuccess) return fail(c, EXH_ESTATE, "hipSetDevice");
  hipStream_t s = stream ? (hipStream_t)stream : c->stream;

  // geometry: per species {rmt, first, end}, then positions (species-major)
  std::vector<double> geo(3 * (size_t)c->nspecies + 3 * (size_t)c->natmtot);
  size_t k = 3 * (size_t)c->nspecies;
  int ias = 0;
  for (int is = 0; is < c->nspecies; is++) {
    geo[3 * is] = c->rmt[is];
    geo[3 * is + 1] = ias;
    for (int ia = 0; ia < c->natoms[is]; ia++, ias++)
      for (int d = 0; d < 3; d++) geo[k++] = atposc[d + 3 * ((size_t)ia + (size_t)maxatoms * is)];
    geo[3 * is + 2] = ias;
  }
  int rc = ensure(c, c->igeo, geo.size() * sizeof(double));
  if (!rc) rc = ensure(c, c->ifz, (size_t)c->ngrtot * sizeof(double2));
  int n[3];
  grid_of(c, n);
  const size_t ntab = (size_t)c->natmtot * (n[0] + n[1] + n[2]);
  if (!rc) rc = ensure(c, c->iphase, std::max<size_t>(ntab, 1) * sizeof(double2));
  if (rc) return rc;

  CfunArgs a;
  std::memcpy(a.b, bvec, sizeof(a.b));
  a.t1 = kFourPi / c->omega;
  a.epslat = epslat;
  a.damp = cfdamp > 0.0 ? cfdamp / gmaxvr : 0.0;
  grid_of(c, &a.n1);
  for (int d = 0; d < 3; d++) {
    a.lo[d] = c->intgv[d];
    a.off[d] = (int)(((-(long long)a.lo[d]) % n[d] + n[d]) % n[d]);
  }
  a.nspecies = c->nspecies;
  const int ng = c->ngrtot;
  double2 *z = (double2 *)c->ifz.p;
  hipError_t e = timed(c, EXH_K_CFUNIG, s, [&] {
    for (size_t w0 = 0; w0 < geo.size(); w0 += kGeoWords) {
      GeoWords g;
      const int nw = (int)std::min<size_t>(kGeoWords, geo.size() - w0);
      std::memcpy(g.v, geo.data() + w0, nw * sizeof(double));
      hipLaunchKernelGGL(put_words_kernel, dim3(1), dim3(kGeoWords), 0, s, g, nw,
                         (double *)c->igeo.p + w0);
    }
    if (ntab)
      hipLaunchKernelGGL(phase_table_kernel, dim3(cdiv_i(ntab, 256)), dim3(256), 0, s, a,
                         c->natmtot, (const double *)c->igeo.p,
                         (double2 *)c->iphase.p);
    hipLaunchKernelGGL(cfunig_kernel, dim3(cdiv_i((long long)n[0] * n[1], 256), cdiv_i(n[2], kRows)),
                       dim3(256), 0, s, a, (const int *)c->ivgig.p,
                       (const double *)c->igeo.p, (const double2 *)c->iphase.p,
                       (double2 *)cfunig, z);
    return hipGetLastError();
  });
  if (e != hipSuccess) return hip_fail(c, e, "gencfun");
  if ((rc = run_fft(c, s, 0, nullptr, z))) return rc;
  e = timed(c, EXH_K_IGATHER, s, [&] {
    hipLaunchKernelGGL(real_part_kernel, dim3(cdiv_i(ng, 256)), dim3(256), 0, s, ng,
                       (const double2 *)z, cfunir);
    return hipGetLastError();
  });
  if (e == hipSuccess) e = mark_done(c, s);
  return e == hipSuccess ? 0 : hip_fail(c, e, "gencfun");
}

int exh_genveffig_device(exh_context *c, void *stream, const double *veffir,
                         const double *cfunir, int which, exh_z *veffig, exh_z *meffig,
                         exh_z *m2effig) {
  if (!c) return EXH_EINVAL;
  if (int rc = wait_done(c)) return rc;
  if (int rc = check_grid(c, "genveffig")) return rc;
  if (which <= 0 || (which & ~(EXH_VEFFIG | EXH_MEFFIG | EXH_M2EFFIG)))
    return fail(c, EXH_EINVAL, "genveffig: which selects none or unknown outputs");
  if (!veffir || !cfunir || ((which & EXH_VEFFIG) && !veffig) ||
      ((which & EXH_MEFFIG) && !meffig) || ((which & EXH_M2EFFIG) && !m2effig))
    return fail(c, EXH_EINVAL, "genveffig: null array");
  if (hipSetDevice(c->device) != hipSuccess) return fail(c, EXH_ESTATE, "hipSetDevice");
  hipStream_t s = stream ? (hipStream_t)stream : c->stream;
  double2 *outs[3] = {nullptr, nullptr, nullptr};
  int nb = 0;
  if (which & EXH_VEFFIG) outs[nb++] = (double2 *)veffig;
  if (which & EXH_MEFFIG) outs[nb++] = (double2 *)meffig;
  if (which & EXH_M2EFFIG) outs[nb++] = (double2 *)m2effig;
  const int n = c->ngrtot;
  int g[3];
  grid_of(c, g);
  // [nb half grids, complex | nb grids, real]
  const size_t half = (size_t)nb * (g[0] / 2 + 1) * g[1] * g[2];
  if (int rc = ensure(c, c->ifz, half * sizeof(double2) + (size_t)nb * n * sizeof(double)))
    return rc;
  double2 *z = (double2 *)c->ifz.p;
  double *x = (double *)(z + half);
  const double a2 = 0.5 * kAlpha * kAlpha;
  hipError_t e = timed(c, EXH_K_IPROD, s, [&] {
    hipLaunchKernelGGL(products_kernel, dim3(cdiv_i(n, 256)), dim3(256), 0, s, n, veffir,
                       cfunir, which, a2, x);
    return hipGetLastError();
  });
  if (e != hipSuccess) return hip_fail(c, e, "genveffig");
  if (int rc = run_fft(c, s, nb, x, z)) return rc;
  const double scale = 1.0 / (double)n;
  e = timed(c, EXH_K_IGATHER, s, [&] {
    hipLaunchKernelGGL(gather_kernel, dim3(cdiv_i(c->ngvec, 256)), dim3(256), 0, s, c->ngvec,
                       (const int *)c->ivg.p, g[0], g[1], g[2], nb, (const double2 *)z, scale,
                       outs[0], outs[1], outs[2]);
    return hipGetLastError();
  });
  if (e == hipSuccess) e = mark_done(c, s);
  return e == hipSuccess ? 0 : hip_fail(c, e, "genveffig");
}

int exh_gencfun(exh_context *c, const double *bvec, const double *atposc, int maxatoms,
                double epslat, double cfdamp, double gmaxvr, exh_z *cfunig, double *cfunir) {
  if (!c) return EXH_EINVAL;
  if (!cfunig || !cfunir) return fail(c, EXH_EINVAL, "gencfun: null array");
  if (int rc = check_grid(c, "gencfun")) return rc;
  const size_t n = (size_t)c->ngrtot;
  int rc = ensure(c, c->i_out0, n * sizeof(double2));
  if (!rc) rc = ensure(c, c->i_out1, n * sizeof(double));
  if (!rc)
    rc = exh_gencfun_device(c, nullptr, bvec, atposc, maxatoms, epslat, cfdamp, gmaxvr,
                            (exh_z *)c->i_out0.p, (double *)c->i_out1.p);
  if (!rc) rc = copy_out(c, cfunig, c->i_out0, n * sizeof(double2));
  if (!rc) rc = copy_out(c, cfunir, c->i_out1, n * sizeof(double));
  return rc;
}

static int host_products(exh_context *c, const double *veffir, const double *cfunir, int which,
                         exh_z *o0, exh_z *o1, exh_z *o2) {
  if (!veffir || !cfunir) return fail(c, EXH_EINVAL, "genveffig: null array");
  if (int rc = check_grid(c, "genveffig")) return rc;
  const size_t n = (size_t)c->ngrtot, ng = (size_t)c->ngvec;
  int rc = copy_in(c, c->i_in0, veffir, n);
  if (!rc) rc = copy_in(c, c->i_in1, cfunir, n);
  DevBuf *bufs[3] = {&c->i_out0, &c->i_out1, &c->i_out2};
  exh_z *dst[3] = {o0, o1, o2};
  for (int b = 0; b < 3 && !rc; b++)
    if (dst[b]) rc = ensure(c, *bufs[b], ng * sizeof(double2));
  if (rc) return rc;
  rc = exh_genveffig_device(c, nullptr, (const double *)c->i_in0.p, (const double *)c->i_in1.p,
                            which, o0 ? (exh_z *)c->i_out0.p : nullptr,
                            o1 ? (exh_z *)c->i_out1.p : nullptr,
                            o2 ? (exh_z *)c->i_out2.p : nullptr);
  for (int b = 0; b < 3 && !rc; b++)
    if (dst[b]) rc = copy_out(c, dst[b], *bufs[b], ng * sizeof(double2));
  return rc;
}

int exh_genveffig(exh_context *c, const double *veffir, const double *cfunir, exh_z *veffig) {
  if (!c) return EXH_EINVAL;
  if (!veffig) return fail(c, EXH_EINVAL, "genveffig: null array");
  return host_products(c, veffir, cfunir, EXH_VEFFIG, veffig, nullptr, nullptr);
}

int exh_genmeffig(exh_context *c, const double *veffir, const double *cfunir,
                  int valence_rel_none, int iora_star, exh_z *meffig, exh_z *m2effig) {
  if (!c) return EXH_EINVAL;
  if (valence_rel_none) return 0;  // genmeffig.f90:34,46: nothing to produce
  if (!meffig || (iora_star && !m2effig)) return fail(c, EXH_EINVAL, "genmeffig: null array");
  return host_products(c, veffir, cfunir, EXH_MEFFIG | (iora_star ? EXH_M2EFFIG : 0), nullptr,
                       meffig, iora_star ? m2effig : nullptr);
}

int exh_set_interstitial_device(exh_context *c, void *stream, const exh_z *cfunig,
                                const exh_z *veffig, const exh_z *meffig,
                                const exh_z *m2effig, int valence_rel_none, int h1on) {
  if (!c) return EXH_EINVAL;
  if (int rc = wait_done(c)) return rc;
  if (!c->have_gvec) return fail(c, EXH_ESTATE, "set_interstitial: call exh_set_gvectors first");
  if (!cfunig || !veffig || (!valence_rel_none && !meffig) || (h1on && !m2effig))
    return fail(c, EXH_EINVAL, "set_interstitial: null array");
  if (hipSetDevice(c->device) != hipSuccess) return fail(c, EXH_ESTATE, "hipSetDevice");
  hipStream_t s = stream ? (hipStream_t)stream : c->stream;
  hipError_t e = launch_ist_table(s, c, (const double2 *)cfunig, (const double2 *)veffig,
                                  (const double2 *)meffig, (const double2 *)m2effig,
                                  valence_rel_none ? 1 : 0, h1on ? 1 : 0);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return hip_fail(c, e, "set_interstitial");
  c->have_ist = true;
  return 0;
}

}  // extern "C"
