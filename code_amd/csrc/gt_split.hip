// gt_split.hip -- what the first strip kernel (u and v, gt_strip_impl.h)
// leaves to do in the other splits, FP64 in the reference's arithmetic:
//   k_half_u  the closing u half sub-step of the 2-D HALFSPLIT
//             (src/2d/advection.F90:541-552 of getm-model/code);
//   k_full_w  the w sub-step of the 3-D FULLSPLIT
//             (src/3d/advection_3d.F90:426-437, adv_split_w.F90).
// Both are bound by launch latency on small grids and by HBM on large ones
// (a field in and out per cell and per sub-step less than one kernel per
// sub-step): 301 x 203 x 25 FULLSPLIT 156 -> 52 us, one
// 100 x 100 slice 25 -> 16 us (its launches 13 us).
#include "gt_strip_impl.h"

namespace gt {

// A wavefront holds 64 consecutive cells of a row; lanes 2..61 have all the
// neighbours (as the strip kernels).
template <int SCH, bool DIFF>
__global__ __launch_bounds__(256) void k_half_u(Dims d, const double* __restrict__ f2,
                                                const double* __restrict__ d2,
                                                const double* __restrict__ a2, double* f,
                                                double* di, double* adv,
                                                const double* __restrict__ U,
                                                const double* __restrict__ DU,
                                                const uint8_t* __restrict__ flags, double dt,
                                                double dx, double dy, double ard1, double AH) {
  constexpr int isub = SCH == UPSTREAM ? 0 : 1;
  const int lane = threadIdx.x;  // blockDim (64, 4): one row per wavefront
  const int x = blockIdx.x * kStripOut - 2 + lane;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  if (j >= d.NY) return;  // the whole wavefront
  const ColumnBits cb = column_bits(x, lane, d.NX, isub);
  const long c2 = cb.xc + (long)d.NX * j, c = c2 + d.NXY * (long)blockIdx.z;
  const double dth = 0.5 * dt;
  const FaceK ku = face_k(dth, dx, AH);
  DivFull dv;
  const int fl = flags[c2] & cb.xin, fo = (fl | MB_XOUT) & cb.xm;
  const int flm = from_lower_lane(fl), flp = from_upper_lane(fl);
  const double u = U[c];
  FaceC<true> fu;
  face_setup<SCH>(fu, fo & MB_UFLUX, flm & MB_UFLUX, flp & MB_UFLUX, u, DU[c], ku, dv);
  const double um = from_lower_lane(u);
  const bool upd = fo & MB_UUPD;
  const double D0 = d2[c];
  const double D1 = sel(upd, D0 - dth * (u * dy - um * dy) * ard1, D0);
  const double fc = f2[c];
  const double fm1 = from_lower_lane(fc), fp1 = from_upper_lane(fc);
  const double fp2 = from_upper_lane(fp1);
  const double Fu = face_flux<double, SCH, DIFF>(fu, fm1, fc, fp1, fp2, AH, ku, dv);
  const double Fum = from_lower_lane(Fu);
  double advn;
  const double F1 =
      cell_update_exact(upd, D0, dv.den(D1), fc, Fu, Fum, 0.5, dy, ard1, dt, &advn, dv);
  if (fo & MB_XOUT) {
    f[c] = F1;
    if (di) di[c] = D1;
    if (adv) adv[c] = a2[c] + advn;
  }
}

__global__ __launch_bounds__(256) void k_copy3(long n, double* __restrict__ f,
                                               const double* __restrict__ f2, double* di,
                                               const double* __restrict__ d2, double* adv,
                                               const double* __restrict__ a2) {
  const long q = blockIdx.x * 256L + threadIdx.x;
  if (q >= n) return;
  f[q] = f2[q];
  if (di) di[q] = d2[q];
  if (adv) adv[q] = a2[q];
}

// One thread per column and chunk of levels, marching up with the levels
// K-1..K+2 of f2, the heights of K and K+1 and the flux at K-1/2 in
// registers; chunks, because one march per column leaves the chip a few
// hundred wavefronts on a small grid (301 x 203 x 25: 955).
template <int SCH>
__global__ __launch_bounds__(256) void k_full_w(Dims d, const double* __restrict__ f2,
                                                const double* __restrict__ d2,
                                                const double* __restrict__ a2,
                                                const double* __restrict__ ww,
                                                const double* __restrict__ ho,
                                                const uint8_t* __restrict__ flags, double* f,
                                                double* hires, double* advres, double dt,
                                                int kshift, int nchunks, int kc) {
  const int chunk = (int)(blockIdx.x % nchunks);
  const int i = (int)(blockIdx.x / nchunks) * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  const int kmax = d.kmax, K0 = 1 + chunk * kc, K1 = min(K0 + kc - 1, kmax);
  if (i >= d.NX || j >= d.NY || K0 > kmax) return;
  const long NXY = d.NXY, c2 = i + (long)d.NX * j;
  if (chunk == 0) {
    if (hires) hires[c2] = ho[c2];
    if (advres) advres[c2] = 0.0;
  }
  auto at = [&](int K) -> long { return c2 + NXY * (long)K; };
  const bool col = (flags[c2] & MB_WCOL) && i <= d.NX - 2 && j <= d.NY - 2;
  if (!col) {
    for (int K = K0; K <= K1; K++) {
      f[at(K)] = f2[at(K)];
      if (hires) hires[at(K)] = d2[at(K)];
      if (advres) advres[at(K)] = a2[at(K)];
    }
    return;
  }
  DivFull dv;
  auto cap = [&](int K) { return min(max(K, 0), kmax); };
  // the flux at K+1/2 from the levels K-1..K+2 (missing ones repeat an end,
  // which reaches no limiter), the heights and w there
  auto flux = [&](int K, double w, double fm, double f0, double fp, double fpp, double Dlo,
                  double Dhi) -> double {
    WFace<true> wf;
    wface_setup<SCH>(wf, w, dt, Dlo, Dhi, true, dv);
    return wflux_exact<SCH>(wf, SCH != UPSTREAM && K > 1 - kshift, SCH != UPSTREAM && K < kmax - 1,
                            fm, f0, fp, fpp, dv);
  };
  double fm = f2[at(K0 - 1)], f0 = f2[at(K0)], fp = f2[at(cap(K0 + 1))], fpp = f2[at(cap(K0 + 2))];
  double D0 = d2[at(K0)], Dp = d2[at(cap(K0 + 1))];
  double wm = ww[at(K0 - 1)], w0 = ww[at(K0)];
  double Fm = K0 > 1 || kshift
                  ? flux(K0 - 1, wm, f2[at(cap(K0 - 2))], fm, f0, fp, d2[at(K0 - 1)], D0)
                  : 0.0;
  for (int K = K0; K <= K1; K++) {
    // the next level's operands, ahead of this one's divisions
    const double fn = f2[at(cap(K + 3))], Dn = d2[at(cap(K + 2))], wp = ww[at(cap(K + 1))];
    const double F = K <= kmax - 1 ? flux(K, w0, fm, f0, fp, fpp, D0, Dp) : 0.0;
    double r = f0, h = D0, aw = 0.0;
    if (K <= kmax - kshift) {
      h = D0 - dt * (w0 - wm);
      aw = 1.0 * (F - Fm);
      r = (D0 * f0 - dt * aw) / h;
    }
    f[at(K)] = r;
    if (hires) hires[at(K)] = h;
    if (advres) advres[at(K)] = a2[at(K)] + aw;
    fm = f0; f0 = fp; fp = fpp; fpp = fn;
    D0 = Dp; Dp = Dn;
    wm = w0; w0 = wp;
    Fm = F;
  }
}

#define GT_SCHEMES(X)                                                        \
  switch (scheme) {                                                          \
    case P2_PDM: X(P2_PDM); break;                                           \
    case SUPERBEE: X(SUPERBEE); break;                                       \
    case MUSCL: X(MUSCL); break;                                             \
    case P2: X(P2); break;                                                   \
    case UPSTREAM: X(UPSTREAM); break;                                       \
    default: return hipErrorInvalidValue;                                    \
  }

hipError_t launch_half_u(hipStream_t st, Dims d, int ns, const double* f2, const double* d2,
                         const double* a2, double* f, double* di, double* adv, const double* U,
                         const double* DU, const uint8_t* flags, double dt, double dx, double dy,
                         double ard1, int scheme, double AH) {
  const dim3 g((d.NX + kStripOut - 1) / kStripOut, (d.NY + 3) / 4, ns), b(64, 4);
#define GT_X(S)                                                                                  \
  if (AH > 0.0)                                                                                  \
    hipLaunchKernelGGL((k_half_u<S, true>), g, b, 0, st, d, f2, d2, a2, f, di, adv, U, DU, flags, \
                       dt, dx, dy, ard1, AH);                                                    \
  else                                                                                           \
    hipLaunchKernelGGL((k_half_u<S, false>), g, b, 0, st, d, f2, d2, a2, f, di, adv, U, DU,      \
                       flags, dt, dx, dy, ard1, AH)
  GT_SCHEMES(GT_X)
#undef GT_X
  return hipGetLastError();
}

hipError_t launch_copy3(hipStream_t st, long n, double* f, const double* f2, double* di,
                        const double* d2, double* adv, const double* a2) {
  hipLaunchKernelGGL(k_copy3, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, f, f2, di,
                     d2, adv, a2);
  return hipGetLastError();
}

hipError_t launch_full_w(hipStream_t st, Dims d, const double* f2, const double* d2,
                         const double* a2, const double* ww, const double* ho,
                         const uint8_t* flags, double* f, double* hires, double* advres,
                         double dt, int scheme, int kshift) {
  // chunks of at least 4 levels until the columns give 8 wavefronts per SIMD
  const long waves = (long)((d.NX + 63) / 64) * d.NY;
  int nch = 1;
  while (waves * nch < 8192 && d.kmax / (nch + 1) >= 4) nch++;
  const int kc = (d.kmax + nch - 1) / nch, nchunks = (d.kmax + kc - 1) / kc;
  const dim3 g((unsigned)(((d.NX + 63) / 64) * nchunks), (d.NY + 3) / 4), b(64, 4);
#define GT_X(S)                                                                                \
  hipLaunchKernelGGL((k_full_w<S>), g, b, 0, st, d, f2, d2, a2, ww, ho, flags, f, hires,       \
                     advres, dt, kshift, nchunks, kc)
  GT_SCHEMES(GT_X)
#undef GT_X
  return hipGetLastError();
}

}  // namespace gt
