// gt_substeps.hip -- the HALFSPLIT step one sub-step at a time, in both
// arithmetic flavours of the strip kernels, and the transpose of each
// sub-step: the reverse mode of the advection.
//
// There is no counterpart in getm-model/code; the forward operator is the
// HALFSPLIT composition of advection_3d.F90:439-547 (u/2, v/2, w, v/2, u/2)
// with the sub-steps of adv_split_u.F90, adv_split_v.F90 and
// adv_split_w.F90.
//
// Forward: one kernel per sub-step, built from the strip kernels' device
// functions (gt_strip_impl.h) with the same operands, so every intermediate
// state is the one the strip kernels hold at that point and the final state
// equals theirs bit for bit.  TF = double: the reference's expressions
// (EXACT); TF = float: the batched FP32 arithmetic.  The layer heights D1..D5
// depend on the velocities only and are formed once (k_heights), in FP64
// with the sub-steps' expressions.
//
// Reverse: with velocities and layer heights held fixed each sub-step is a
// piecewise linear map of the tracer,
//   f_new(i) = a(i) f(i) - s(i) (F(i) - F(i-1)),
//   F(X)     = vel(X) rec(fuu, fu, fd) - kA(X) (f(X+1) - f(X)),
// with a = Dio/Dn and s = dt*splitfac*dlen*ard1/Dn (FP32: 1+am1 and b, the
// factors of cell_update_fast).  The transpose is formed face by face, every
// face once: along i a lane owns a face and the cells collect their faces'
// terms by cross-lane moves; along j and k a thread marches rows or levels
// with a four-deep window in registers and stores each output when no
// further face reaches it (no atomics).  The limiter's derivative is that of
// the branch the forward took (one-sided at ties and kinks).
#include "gt_strip_impl.h"
#include "gt_substeps.h"

namespace gt {

// ---- layer heights ---------------------------------------------------------------
// D1..D5 from D0 = ho: adv_split_u.F90:275 (Di = Dio - dti*(U(i)*dy -
// U(i-1)*dy)*ard1), adv_split_v.F90 likewise with dx, adv_split_w.F90:288
// (hi = hio - dti*(ww(k) - ww(k-1))), where the sub-step updates the cell;
// level 0 keeps ho
__global__ void k_heights(Dims d, const uint8_t* __restrict__ flags, const double* __restrict__ ho,
                          const double* __restrict__ uu, const double* __restrict__ vv,
                          const double* __restrict__ ww, double* __restrict__ D1,
                          double* __restrict__ D2, double* __restrict__ D3,
                          double* __restrict__ D4, double* __restrict__ D5, double dt, double dx,
                          double dy, double ard1, int isub, int kshift) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  const int k = blockIdx.z;
  if (i >= d.NX || j >= d.NY || k > d.kmax) return;
  const long c2 = i + (long)d.NX * j, c = c2 + d.NXY * (long)k;
  const double D0 = ho[c];
  if (k == 0) {
    D1[c] = D0; D2[c] = D0; D3[c] = D0; D4[c] = D0; D5[c] = D0;
    return;
  }
  const int fl = flags[c2];
  const double dth = 0.5 * dt;
  const bool updu = (fl & MB_UUPD) && i >= 1 + isub && i <= d.NX - 2 - isub;
  const bool updv = (fl & MB_VUPD) && j >= 1 + isub && j <= d.NY - 2 - isub;
  const bool wupd = (fl & MB_WCOL) && i <= d.NX - 2 && j <= d.NY - 2 && k <= d.kmax - kshift;
  const double du = updu ? uu[c] * dy - uu[c - 1] * dy : 0.0;
  const double dv = updv ? vv[c] * dx - vv[c - d.NX] * dx : 0.0;
  const double h1 = updu ? D0 - dth * du * ard1 : D0;
  const double h2 = updv ? h1 - dth * dv * ard1 : h1;
  const double h3 = wupd ? h2 - dt * (ww[c] - ww[c - d.NXY]) : h2;
  const double h4 = updv ? h3 - dth * dv * ard1 : h3;
  const double h5 = updu ? h4 - dth * du * ard1 : h4;
  D1[c] = h1; D2[c] = h2; D3[c] = h3; D4[c] = h4; D5[c] = h5;
}

// ---- shared pieces -------------------------------------------------------------
template <typename TF>
constexpr bool kExact = sizeof(TF) == 8;
// tracers per thread of the row and column marches
template <typename TF>
constexpr int kGroup = sizeof(TF) == 8 ? 1 : 6;
// output rows per wavefront of the v marches (FP64 carries one tracer, so
// shorter marches for more wavefronts)
template <typename TF>
constexpr int kVRows = sizeof(TF) == 8 ? 8 : 16;
// most output rows per wavefront of the u and v transposes (marches of 16 and
// 32 rows recompute six rows each): the launcher halves them where that leaves
// the chip short of wavefronts.  256 x 256 x 30, one FP64 tracer, 8 / 16 / 24
// rows: 69 + 62, 57 + 54, 61 + 64 us; 18 FP32 tracers at 320 x 256 x 30,
// 16 / 32 rows: 351 + 316, 331 + 312 us.
template <typename TF>
constexpr int kUVRows = sizeof(TF) == 8 ? 16 : 32;
constexpr long kUVWaves = 2048;  // ... and how many wavefronts they aim for (2 per SIMD)
constexpr long kWaveTarget = 8192;  // wavefronts a column march aims for (8 per SIMD)
constexpr int kUOutF = 60;  // outputs per wavefront of the u forward
constexpr int kUOutA = 58;  // ... and of the u transpose

// geometry of one sweep: dir 0 = u (faces along i, stride 1), 1 = v (NX)
struct Sweep {
  long st;
  int n;
  uint8_t mflux, mupd;
};
__device__ __forceinline__ Sweep sweep(const Dims& d, int dir) {
  return dir == 0 ? Sweep{1, d.NX, MB_UFLUX, MB_UUPD} : Sweep{(long)d.NX, d.NY, MB_VFLUX, MB_VUPD};
}

// the constants of face X (between cells X and X+1 of the sweep) as the strip
// kernels form them; X in 0..n-2, x2 its column index, o its level offset
template <int SCH, bool EXACT>
__device__ __forceinline__ FaceC<EXACT> face_at(const Sweep& s, int X, long x2, long o,
                                                const uint8_t* flags, const double* vel,
                                                const double* Dv, const FaceK& k) {
  constexpr int isub = SCH == UPSTREAM ? 0 : 1;
  const bool active = X >= isub && X <= s.n - 2 - isub && (flags[x2] & s.mflux);
  const bool lim_l = SCH != UPSTREAM && X >= 1 && (flags[x2 - s.st] & s.mflux);
  const bool lim_r = SCH != UPSTREAM && (flags[x2 + s.st] & s.mflux);
  FaceC<EXACT> fc;
  DivFull dv;
  face_setup<SCH>(fc, active, lim_l, lim_r, vel[o + x2], Dv[o + x2], k, dv);
  return fc;
}

// a face that carries no flux (outside the sweep's face range)
template <bool EXACT>
__device__ __forceinline__ FaceC<EXACT> no_face() {
  return FaceC<EXACT>{};
}

// the loads of row Y of a v march: face Y's transport, layer height and
// flux-mask bytes (rows Y-1..Y+1) and cell Y's heights before and after,
// read one row ahead of their use (rows outside 0..NY-1 read a clamped row;
// the face and the update are switched off there by Y itself)
struct VRaw {
  double vel, Dv, Dio, Dn;
  uint8_t fm, f0, fp;
};
__device__ __forceinline__ VRaw vraw(const Dims& d, int x, long o, int Y,
                                     const uint8_t* flags, const double* vel,
                                     const double* Dv, const double* Dio, const double* Dn) {
  const int NX = d.NX, Yc = min(max(Y, 0), d.NY - 1);
  const long x2 = x + (long)NX * Yc;
  VRaw r;
  r.vel = vel[o + x2];
  r.Dv = Dv[o + x2];
  r.Dio = Dio[o + x2];
  r.Dn = Dn[o + x2];
  r.f0 = flags[x2];
  r.fm = flags[x + (long)NX * max(Yc - 1, 0)];
  r.fp = flags[x + (long)NX * min(Yc + 1, d.NY - 1)];
  return r;
}
// face Y of the v sweep from its loads, as face_at forms it (0 <= Y <= NY-2)
template <int SCH, bool EXACT>
__device__ __forceinline__ FaceC<EXACT> vface(const Dims& d, int Y, const VRaw& r,
                                              const FaceK& k) {
  constexpr int isub = SCH == UPSTREAM ? 0 : 1;
  const bool active = Y >= isub && Y <= d.NY - 2 - isub && (r.f0 & MB_VFLUX);
  const bool lim_l = SCH != UPSTREAM && Y >= 1 && (r.fm & MB_VFLUX);
  const bool lim_r = SCH != UPSTREAM && (r.fp & MB_VFLUX);
  FaceC<EXACT> fc;
  DivFull dv;
  face_setup<SCH>(fc, active, lim_l, lim_r, r.vel, r.Dv, k, dv);
  return fc;
}

// the update of one cell: f_new = (Dio f - dt advn)/Dn (EXACT, the
// reference's expression) or f + f am1 - (Fc - Fm) b (FP32), and its
// linearisation: diag (d f_new / d f) and mu (d f_new / d Fc, = -d/d Fm)
template <bool EXACT>
struct CellOp;
template <>
struct CellOp<false> {
  float am1 = 0.0f, b = 0.0f;
  // dtc = dt*splitfac*dlen*ard1 (dt for w)
  __device__ static CellOp make(double Dio, double Dn, double dtc) {
    const CellK k = cell_factors(Dio, Dn, dtc);
    CellOp c;
    c.am1 = k.am1;
    c.b = k.b;
    return c;
  }
  __device__ float h_step(float fo, float Fc, float Fm, double, double, double) const {
    return cell_update_fast(true, CellK{am1, b}, fo, Fc, Fm);
  }
  __device__ float w_step(float fo, float wk, float wprev, double) const {
    return cell_update_fast(true, CellK{am1, b}, fo, wk, wprev);
  }
  __device__ float diag(float l) const { return __builtin_fmaf(l, am1, l); }
  __device__ float mu(float l, double, double) const { return -b * l; }
};
template <>
struct CellOp<true> {
  double Dio = 1.0, Dn = 1.0;
  __device__ static CellOp make(double Dio, double Dn, double) {
    CellOp c;
    c.Dio = Dio;
    c.Dn = Dn;
    return c;
  }
  // adv_split_u.F90:267-286 in the reference's order (dlen: the face length)
  __device__ double h_step(double fo, double Fc, double Fm, double dt, double dlen,
                           double ard1) const {
    double advn;
    DivFull dv;
    return cell_update_exact(true, Dio, dv.den(Dn), fo, Fc, Fm, 0.5, dlen, ard1, dt, &advn, dv);
  }
  // adv_split_w.F90:287-294
  __device__ double w_step(double fo, double wk, double wprev, double dt) const {
    const double aw = 1.0 * (wk - wprev);
    return (Dio * fo - dt * aw) / Dn;
  }
  __device__ double diag(double l) const { return l * Dio / Dn; }
  // fac = splitfac*dlen*ard1 (splitfac for w)
  __device__ double mu(double l, double dt, double fac) const { return l * (-dt / Dn) * fac; }
};

// ---- derivatives of the reconstruction --------------------------------------------
template <typename T>
struct RecG {
  T duu, du, dd;
};

// (Both flavours form every operand and select, as the forward does: returning
// early for the faces without a limiter cut the marches into blocks in which
// nothing overlapped.  320 x 256 x 30 x 18 FP32 tracers: w transpose 245 ->
// 225 us, u and v transposes 364 + 338 -> 351 + 316 us, with fewer registers.)

// the reference arithmetic (reconstruct_bf): rec = fu + (1-cfl)/2 phi(r)
// deltaf, r = deltafu/deltaf, the branch of phi that the forward's min / max
// selected; E = 2/(1-cfl) as the face holds it; lim: the limiter applies
template <int SCH>
__device__ __forceinline__ RecG<double> rec_grad_exact(bool lim, double cfl, double E, double fuu,
                                                       double fu, double fd) {
  const double g = 0.5 * (1.0 - cfl);
  const double deltaf = fd - fu, deltafu = fu - fuu;
  if constexpr (SCH == UPSTREAM) {
    return {0.0, 1.0, 0.0};
  } else if constexpr (SCH == P2) {  // linear on both branches
    const double x = (1.0 / 6.0) * (1.0 - 2.0 * cfl);
    return {lim ? -g * (0.5 - x) : 0.0, lim ? 1.0 - g * (0.5 + x) + g * (0.5 - x) : 1.0,
            lim ? g * (0.5 + x) : 0.0};
  } else {
    const bool on = lim & (deltaf * deltafu > 0.0);
    const double r = deltafu / deltaf;
    double phi, dphi;
    if constexpr (SCH == P2_PDM) {
      const double x = (1.0 / 6.0) * (1.0 - 2.0 * cfl);
      const double a = 2.0 * r / (cfl + 1.e-10), b = (0.5 + x) + (0.5 - x) * r;
      const double m = a < b ? a : b;
      const double dm = a < b ? 2.0 / (cfl + 1.e-10) : (0.5 - x);
      phi = E < m ? E : m;
      dphi = E < m ? 0.0 : dm;
    } else if constexpr (SCH == SUPERBEE) {
      const bool a1 = 2.0 * r < 1.0, b1 = r < 2.0;
      const double a = a1 ? 2.0 * r : 1.0, da = a1 ? 2.0 : 0.0;
      const double b = b1 ? r : 2.0, db = b1 ? 1.0 : 0.0;
      phi = a > b ? a : b;
      dphi = a > b ? da : db;
    } else {  // MUSCL
      const double a = 2.0 * r, b = 0.5 * (1.0 + r);
      const double m = a < b ? a : b, dm = a < b ? 2.0 : 0.5;
      phi = 2.0 < m ? 2.0 : m;
      dphi = 2.0 < m ? 0.0 : dm;
    }
    // d/dfuu = -g dphi, d/dfu = 1 + g (dphi (1 + r) - phi), d/dfd = g (phi - dphi r)
    return {on ? -g * dphi : 0.0, on ? 1.0 + g * (dphi * (1.0 + r) - phi) : 1.0,
            on ? g * (phi - dphi * r) : 0.0};
  }
}

// the FP32 arithmetic (rec_fast): rec = fu + g t, t the branch term the
// forward's min / max selected, each term linear in du = fu-fuu, df = fd-fu;
// the identity where the limiter does not apply (g = 0) or deltaf*deltafu <=
// 0.  The terms are compared over the magnitudes, as the forward takes them.
template <int SCH>
__device__ __forceinline__ RecG<float> rec_grad_fast(float fuu, float fu, float fd, float g,
                                                     float A, float al, float E) {
  if constexpr (SCH == UPSTREAM) {
    return {0.0f, 1.0f, 0.0f};
  } else {
    const float df = fd - fu, du = fu - fuu;
    bool on = g != 0.0f;
    float tu, tf;  // d t / d du, d t / d df
    if constexpr (SCH == P2) {
      tu = 1.0f - al;
      tf = al;
    } else {
      on &= df * du > 0.0f;
      const float adf = __builtin_fabsf(df), adu = __builtin_fabsf(du);
      if constexpr (SCH == P2_PDM) {
        const float t1 = A * adu, t2 = __builtin_fmaf(al, adf - adu, adu), t3 = E * adf;
        const bool s2 = t2 < t1;
        const bool s3 = t3 < (s2 ? t2 : t1);
        tu = s3 ? 0.0f : (s2 ? 1.0f - al : A);
        tf = s3 ? E : (s2 ? al : 0.0f);
      } else if constexpr (SCH == SUPERBEE) {
        // max(min(2du, df), min(du, 2df))
        const float a2 = 2.0f * adu, b2 = 2.0f * adf;
        const bool inner_a = adf < a2;  // first pair: picks df
        const bool inner_b = b2 < adu;  // second pair: picks 2df
        const bool outer_b = (inner_b ? b2 : adu) > (inner_a ? adf : a2);
        tu = outer_b ? (inner_b ? 0.0f : 1.0f) : (inner_a ? 0.0f : 2.0f);
        tf = outer_b ? (inner_b ? 2.0f : 0.0f) : (inner_a ? 1.0f : 0.0f);
      } else {  // MUSCL: min(min(2du, h), 2df), h = (df+du)/2
        const float a2 = 2.0f * adu, b2 = 2.0f * adf, h = 0.5f * (adf + adu);
        const bool s2 = h < a2;
        const bool s3 = b2 < (s2 ? h : a2);
        tu = s3 ? 0.0f : (s2 ? 0.5f : 2.0f);
        tf = s3 ? 2.0f : (s2 ? 0.5f : 0.0f);
      }
    }
    return {on ? -g * tu : 0.0f, on ? 1.0f + g * (tu - tf) : 1.0f, on ? g * tf : 0.0f};
  }
}

// partials of face_flux with respect to the cells X-1..X+2
template <typename TF, int SCH, bool DIFF>
__device__ __forceinline__ void face_flux_grad(const FaceC<kExact<TF>>& fc, TF fm1, TF f0, TF fp1,
                                               TF fp2, double AH, double dlen, TF out[4]) {
  RecG<TF> r;
  bool left;
  TF vel;  // 0 for a face that carries no flux (not limited either)
  if constexpr (kExact<TF>) {
    left = fc.left;
    vel = fc.active ? fc.vel : 0.0;
    r = rec_grad_exact<SCH>(fc.lim, fc.cfl, fc.E, left ? fm1 : fp2, left ? f0 : fp1,
                            left ? fp1 : f0);
  } else {
    left = !fc.right;
    vel = fc.vel;
    r = rec_grad_fast<SCH>(left ? fm1 : fp2, left ? f0 : fp1, left ? fp1 : f0, fc.g, fc.A, fc.al,
                           fc.E);
  }
  const TF duu = vel * r.duu, du = vel * r.du, dd = vel * r.dd;
  out[0] = left ? duu : TF(0);
  out[1] = left ? du : dd;
  out[2] = left ? dd : du;
  out[3] = left ? TF(0) : duu;
  if constexpr (DIFF) {
    TF k;
    if constexpr (kExact<TF>) k = fc.active ? AH * fc.Dv / dlen : 0.0;
    else k = fc.kA;
    out[1] += k;
    out[2] -= k;
  }
  (void)AH; (void)dlen;
}

// the w flux at face K (K+1/2) from the levels K-1..K+2, and its partials;
// lim_up / lim_dn: whether the limiter applies going up / down
template <typename TF, int SCH>
__device__ __forceinline__ TF w_flux(const WFace<kExact<TF>>& wf, bool lim_up, bool lim_dn,
                                     TF fkm1, TF fk, TF fk1, TF fk2) {
  if constexpr (kExact<TF>) {
    DivFull dv;
    return wflux_exact<SCH>(wf, lim_up, lim_dn, fkm1, fk, fk1, fk2, dv);
  } else {
    return wflux_fast<SCH>(wf, lim_up, lim_dn, fkm1, fk, fk1, fk2);
  }
}

template <typename TF, int SCH>
__device__ __forceinline__ void w_flux_grad(const WFace<kExact<TF>>& wf, bool lim_up, bool lim_dn,
                                            TF fkm1, TF fk, TF fk1, TF fk2, TF out[4]) {
  const bool up = wf.w > 0;
  const TF fu = up ? fk : fk1, fuu = up ? fkm1 : fk2, fd = up ? fk1 : fk;
  const bool lim = up ? lim_up : lim_dn;
  RecG<TF> r;
  if constexpr (kExact<TF>) {
    r = rec_grad_exact<SCH>(lim, wf.cfl, wf.E, fuu, fu, fd);
  } else {
    r = rec_grad_fast<SCH>(fuu, fu, fd, lim ? wf.g : 0.0f, wf.A, wf.al, wf.E);
  }
  const TF w = TF(wf.w);
  const TF duu = w * r.duu, du = w * r.du, dd = w * r.dd;
  out[0] = up ? duu : TF(0);
  out[1] = up ? du : dd;
  out[2] = up ? dd : du;
  out[3] = up ? TF(0) : duu;
}

// ---- the u half sub-step ---------------------------------------------------------
// A wavefront holds 64 consecutive cells of a row; lane L forms the flux of
// face x from the cells x-1..x+2 (cross-lane moves) and cell x takes the flux
// of face x-1 from lane L-1, as the strip kernels do: lanes 2..61 are
// complete.  Level 0 and cells the sub-step leaves alone are copied.
template <typename TF, int SCH, bool DIFF>
__global__ __launch_bounds__(256) void k_sub_u(Dims d, int ntr, long ts,
                                               const TF* __restrict__ fin, TF* __restrict__ fout,
                                               const double* __restrict__ Dio,
                                               const double* __restrict__ Dn,
                                               const double* __restrict__ uu,
                                               const double* __restrict__ hu,
                                               const uint8_t* __restrict__ flags, double dt,
                                               double dx, double dy, double ard1, double AH) {
  constexpr bool EX = kExact<TF>;
  constexpr int isub = SCH == UPSTREAM ? 0 : 1;
  const int lane = threadIdx.x;  // blockDim (64, 4): one row per wavefront
  const int x = blockIdx.x * kUOutF - 2 + lane;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  const int k = blockIdx.z;
  if (j >= d.NY) return;  // the whole wavefront
  const bool xin = x >= 0 && x < d.NX;
  const long c2 = (long)min(max(x, 0), d.NX - 1) + (long)d.NX * j;
  const long o = d.NXY * (long)k, c = o + c2;
  const bool out = xin && lane >= 2 && lane <= 61;
  if (k == 0) {
    if (out)
      for (int t = 0; t < ntr; t++) fout[t * ts + c] = fin[t * ts + c];
    return;
  }
  const FaceK fk = face_k(0.5 * dt, dx, AH);
  DivFull dv;
  FaceC<EX> fc = no_face<EX>();
  if (xin && x <= d.NX - 2)
    fc = face_at<SCH, EX>(sweep(d, 0), x, c2, o, flags, uu, hu, fk);
  const bool upd = xin && x >= 1 + isub && x <= d.NX - 2 - isub && (flags[c2] & MB_UUPD);
  CellOp<EX> cu;
  if (upd) cu = CellOp<EX>::make(Dio[c], Dn[c], dt * (0.5 * dy * ard1));
  for (int t = 0; t < ntr; t++) {
    const TF fx = fin[t * ts + c];
    const TF fm1 = from_lower_lane(fx), fp1 = from_upper_lane(fx);
    const TF fp2 = from_upper_lane(fp1);
    const TF Fc = face_flux<TF, SCH, DIFF>(fc, fm1, fx, fp1, fp2, AH, fk, dv);
    const TF Fm = from_lower_lane(Fc);
    const TF u = cu.h_step(fx, Fc, Fm, dt, dy, ard1);
    if (out) fout[t * ts + c] = upd ? u : fx;
  }
}

// ---- the v half sub-step: a row march -------------------------------------------
// A wavefront holds 64 columns and marches the faces Y = y0-1 .. y1-1 for a
// group of tracers, with the rows Y-1..Y+2 and the flux of face Y-1 in
// registers; row Y is updated after face Y.
template <typename TF, int SCH, bool DIFF>
__global__ __launch_bounds__(64) void k_sub_v(Dims d, int ntr, long ts, const TF* __restrict__ fin,
                                              TF* __restrict__ fout,
                                              const double* __restrict__ Dio,
                                              const double* __restrict__ Dn,
                                              const double* __restrict__ vv,
                                              const double* __restrict__ hv,
                                              const uint8_t* __restrict__ flags, double dt,
                                              double dx, double dy, double ard1, double AH,
                                              int ngroups) {
  constexpr bool EX = kExact<TF>;
  constexpr int isub = SCH == UPSTREAM ? 0 : 1;
  constexpr int G = kGroup<TF>;
  const int x = blockIdx.x * 64 + threadIdx.x;
  const int y0 = blockIdx.y * kVRows<TF>;
  const int k = blockIdx.z / ngroups, t0 = (blockIdx.z % ngroups) * G;
  if (x >= d.NX) return;  // no cross-lane moves here
  const int NX = d.NX, NY = d.NY;
  const long o = d.NXY * (long)k;
  const int y1 = min(y0 + kVRows<TF>, NY);
  long tb[G];
#pragma unroll
  for (int g = 0; g < G; g++) tb[g] = (long)min(t0 + g, ntr - 1) * ts;
  if (k == 0) {
    for (int y = y0; y < y1; y++)
#pragma unroll
      for (int g = 0; g < G; g++)
        if (t0 + g < ntr) fout[tb[g] + x + (long)NX * y] = fin[tb[g] + x + (long)NX * y];
    return;
  }
  const FaceK fk = face_k(0.5 * dt, dy, AH);
  DivFull dv;
  const double dtc = dt * (0.5 * dx * ard1);
  auto row = [&](int y) -> long { return o + x + (long)NX * (y >= 0 && y < NY ? y : 0); };
  TF w[G][4], Fp[G];
#pragma unroll
  for (int g = 0; g < G; g++) {
    Fp[g] = TF(0);
#pragma unroll
    for (int q = 0; q < 4; q++) w[g][q] = fin[tb[g] + row(y0 - 2 + q)];
  }
  VRaw rn = vraw(d, x, o, y0 - 1, flags, vv, hv, Dio, Dn);
  for (int Y = y0 - 1; Y < y1; Y++) {
    const VRaw r = rn;
    rn = vraw(d, x, o, Y + 1, flags, vv, hv, Dio, Dn);
    FaceC<EX> fc = no_face<EX>();
    if (Y >= 0 && Y <= NY - 2) fc = vface<SCH, EX>(d, Y, r, fk);
    const bool st = Y >= y0;
    const long cY = o + x + (long)NX * (Y >= 0 ? Y : 0);
    const bool upd = st && Y >= 1 + isub && Y <= NY - 2 - isub && (r.f0 & MB_VUPD);
    CellOp<EX> cu;
    if (upd) cu = CellOp<EX>::make(r.Dio, r.Dn, dtc);
#pragma unroll
    for (int g = 0; g < G; g++) {
      const TF F = face_flux<TF, SCH, DIFF>(fc, w[g][0], w[g][1], w[g][2], w[g][3], AH, fk, dv);
      if (st && t0 + g < ntr) {
        const TF u = cu.h_step(w[g][1], F, Fp[g], dt, dx, ard1);
        fout[tb[g] + cY] = upd ? u : w[g][1];
      }
      Fp[g] = F;
      w[g][0] = w[g][1];
      w[g][1] = w[g][2];
      w[g][2] = w[g][3];
      w[g][3] = fin[tb[g] + row(Y + 3)];
    }
  }
}

// ---- the vertical sub-step (adv_ver_iterations = 1) ------------------------------
// One thread per column, group of tracers and chunk of levels, marching up with
// the levels K-1..K+2 of each tracer, K..K+3 of D2, D3 and ww and the flux
// at K-1/2 in registers (kmax >= 2).  At level K, as the strip kernels set them
// (adv_split_w.F90:249-300): the flux at K+1/2 exists below kmax, the one at
// K-1/2 above level 1 (or at level 1 with kshift); level K is updated up to
// kmax-kshift; the limiter applies above level 1-kshift going up and below
// kmax-1 going down.
template <typename TF, int SCH>
__global__ __launch_bounds__(256) void k_sub_w(Dims d, int ntr, long ts, const TF* __restrict__ fin,
                                               TF* __restrict__ fout,
                                               const double* __restrict__ D2,
                                               const double* __restrict__ D3,
                                               const double* __restrict__ ww,
                                               const uint8_t* __restrict__ flags, double dt,
                                               int kshift, int ngroups, int nchunks, int kc) {
  constexpr bool EX = kExact<TF>;
  constexpr int G = kGroup<TF>;
  // blockIdx.x = column block * nz + z, z = chunk * ngroups + group: the
  // groups and chunks of one column block run together, so the FP64 fields
  // they all read meet in the cache
  const int nz = ngroups * nchunks, bz = (int)(blockIdx.x % nz);
  const int i = (int)(blockIdx.x / nz) * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  const int t0 = (bz % ngroups) * G;
  const int kmax = d.kmax;
  // this thread's levels K0..K1 (chunk bz / ngroups of kc levels; the first
  // chunk also carries level 0)
  const int K0 = 1 + (bz / ngroups) * kc, K1 = min(K0 + kc - 1, kmax);
  if (i >= d.NX || j >= d.NY || t0 >= ntr || K0 > kmax) return;
  const long NXY = d.NXY, c2 = i + (long)d.NX * j;
  long tb[G];
#pragma unroll
  for (int g = 0; g < G; g++) tb[g] = (long)min(t0 + g, ntr - 1) * ts;
  const bool wcol = (flags[c2] & MB_WCOL) && i <= d.NX - 2 && j <= d.NY - 2;
  if (!wcol) {
    for (int K = K0 == 1 ? 0 : K0; K <= K1; K++)
#pragma unroll
      for (int g = 0; g < G; g++)
        if (t0 + g < ntr) fout[tb[g] + c2 + NXY * K] = fin[tb[g] + c2 + NXY * K];
    return;
  }
  TF n[G][5];  // n[1..4]: levels K-1..K+2 (entries past kmax unused)
  TF fKm2[G];  // level K0-2 (zero below level 0), for the flux at K0-1/2
#pragma unroll
  for (int g = 0; g < G; g++) {
    const TF* f = fin + tb[g];
    fKm2[g] = K0 >= 2 ? f[c2 + NXY * (K0 - 2)] : TF(0);
    n[g][1] = f[c2 + NXY * (K0 - 1)];
    n[g][2] = f[c2 + NXY * K0];
    n[g][3] = K0 + 1 <= kmax ? f[c2 + NXY * (K0 + 1)] : TF(0);
    n[g][4] = K0 + 2 <= kmax ? f[c2 + NXY * (K0 + 2)] : TF(0);
    if (K0 == 1 && t0 + g < ntr) fout[tb[g] + c2] = n[g][1];  // level 0
  }
  // D2, D3 and ww of levels K..K+3 in registers, each loaded three levels
  // ahead of its use (levels past kmax read level kmax, never used)
  auto lv = [&](int L) -> long { return c2 + NXY * (long)min(L, kmax); };
  double d2r[4], d3r[4], wr[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    d2r[q] = D2[lv(K0 + q)];
    d3r[q] = D3[lv(K0 + q)];
    wr[q] = ww[lv(K0 + q)];
  }
  // The flux at K-1/2 that level K reads is the flux at K+1/2 of level K-1,
  // so each face is evaluated once and carried up (pc).  The operands agree
  // except the one past kmax that the strip kernels substitute, which is the
  // upwind-upwind level of a downward face with the limiter off: not read.
  DivFull dv;
  TF pc[G];
  {
    const int F = K0 - 1;  // the face below level K0
    WFace<EX> wf0;
    wface_setup<SCH>(wf0, ww[c2 + NXY * F], dt, D2[c2 + NXY * F], d2r[0], true, dv);
    const bool lim_up = SCH != UPSTREAM && F > 1 - kshift;
    const bool lim_dn = SCH != UPSTREAM && F < kmax - 1;
#pragma unroll
    for (int g = 0; g < G; g++)
      pc[g] = w_flux<TF, SCH>(wf0, lim_up, lim_dn, fKm2[g], n[g][1], n[g][2],
                              K0 + 1 <= kmax ? n[g][3] : n[g][2]);
  }
  for (int K = K0; K <= K1; K++) {
    const long cK = c2 + NXY * K;
    const bool wk_on = K <= kmax - 1, wp_on = K > 1 || kshift, kdo = K <= kmax - kshift;
    const bool limk_up = SCH != UPSTREAM && K > 1 - kshift;
    const bool limk_dn = SCH != UPSTREAM && K < kmax - 1;
    const double dk = d2r[0], dp = d2r[1];  // D2 at K, K+1
    WFace<EX> wfk;
    wface_setup<SCH>(wfk, wr[0], dt, dk, K + 1 <= kmax ? dp : dk, true, dv);
    const CellOp<EX> cw = CellOp<EX>::make(dk, d3r[0], dt);
    const bool nxt = K + 3 <= kmax;
    const long cn = c2 + NXY * (nxt ? K + 3 : kmax);
#pragma unroll
    for (int g = 0; g < G; g++) {
      // the operands of the strip kernels: levels past kmax are replaced by
      // level K
      const TF fKm1 = n[g][1], fK = n[g][2];
      const TF fKp1 = K + 1 <= kmax ? n[g][3] : fK, fKp2 = K + 2 <= kmax ? n[g][4] : fK;
      const TF q = w_flux<TF, SCH>(wfk, limk_up, limk_dn, fKm1, fK, fKp1, fKp2);
      const TF wprev = wp_on ? pc[g] : TF(0), wk = wk_on ? q : TF(0);
      const TF r = kdo ? cw.w_step(fK, wk, wprev, dt) : fK;
      if (t0 + g < ntr) fout[tb[g] + cK] = r;
      pc[g] = q;
      n[g][1] = n[g][2];
      n[g][2] = n[g][3];
      n[g][3] = n[g][4];
      n[g][4] = nxt ? fin[tb[g] + cn] : TF(0);
    }
#pragma unroll
    for (int q = 0; q < 3; q++) {
      d2r[q] = d2r[q + 1];
      d3r[q] = d3r[q + 1];
      wr[q] = wr[q + 1];
    }
    d2r[3] = D2[lv(K + 4)];
    d3r[3] = D3[lv(K + 4)];
    wr[3] = ww[lv(K + 4)];
  }
}

// ---- transpose of a u and a v sub-step, in either order: a row march -----------
// UF: u first (the last two sub-steps of HALFSPLIT, reversed), else v first
// (the first two).  A wavefront marches the rows of a strip of kUOutA output
// columns; fu, fv: the states before the u and the v sub-step; lam_in: the
// adjoint of the later one's output; lam_out: of the earlier one's input.
//
// v: the faces Y = y0-2 .. y1 (those of the output rows); before face Y the
// window holds rows Y-1..Y+2 of the lane's column: each row enters with its
// diagonal part and mu, collects the terms of the faces whose stencil holds
// it, and leaves when it is complete (row Y-1 after face Y).
// u: lane L owns cell x and face x (between x and x+1).  Face x reads the
// cells x-1..x+2 and its flux enters the updates of cells x and x+1; cell x
// collects the faces x-2..x+1 (lanes L-2..L+1).  Lanes 3..60 are complete.
// A row passes the u transpose when it enters the window (UF) or when it
// leaves it, so the adjoint between the two sub-steps stays in registers.
// The set is read and written once for two sub-steps.  Against a kernel each:
// 256 x 256 x 30, one FP64 tracer, 28 + 35 -> 59 (u first) and 54 us (v
// first), bound by the latency of each row's chain; 320 x 256 x 30, 18 FP32
// tracers, 157 + 223 -> 323 and 312 us, 708 MB each, bound by issue at three
// wavefronts per SIMD.  The four rows before the first face go through the
// same loop: unrolled ahead of it they took 60 registers of scratch.
template <typename TF, int SCH, bool DIFF, bool UF>
__global__ __launch_bounds__(64, kExact<TF> ? 4 : 3) void k_sub_uv_adj(
    Dims d, int ntr, long ts, const TF* __restrict__ fu, const TF* __restrict__ fv,
    const TF* __restrict__ lam_in, TF* __restrict__ lam_out, const double* __restrict__ Du0,
    const double* __restrict__ Du1, const double* __restrict__ Dv0,
    const double* __restrict__ Dv1, const double* __restrict__ uu,
    const double* __restrict__ hu, const double* __restrict__ vv, const double* __restrict__ hv,
    const uint8_t* __restrict__ flags, double dt, double dx, double dy, double ard1, double AH,
    int ngroups, int rows) {
  constexpr bool EX = kExact<TF>;
  constexpr int isub = SCH == UPSTREAM ? 0 : 1;
  constexpr int G = kGroup<TF>;
  // whether the u loads of a row are issued a row ahead: where the registers
  // hold them (FP32, v first: 104 bytes of scratch and 689 us; 12 with
  // diffusion) and it pays
  // (FP64, u first: 59 us either way)
  constexpr bool AHEAD = EX ? !UF : UF && !DIFF;
  const int lane = threadIdx.x;
  const int x = blockIdx.x * kUOutA - 3 + lane;
  const int y0 = blockIdx.y * rows;
  const int k = blockIdx.z / ngroups, t0 = (blockIdx.z % ngroups) * G;
  const int NX = d.NX, NY = d.NY;
  const bool xin = x >= 0 && x < NX, out = xin && lane >= 3 && lane <= 60;
  const int xc = min(max(x, 0), NX - 1);
  const long o = d.NXY * (long)k;
  const int y1 = min(y0 + rows, NY);
  long tb[G];
#pragma unroll
  for (int g = 0; g < G; g++) tb[g] = (long)min(t0 + g, ntr - 1) * ts;
  if (k == 0) {
    for (int y = y0; y < y1; y++)
#pragma unroll
      for (int g = 0; g < G; g++)
        if (out && t0 + g < ntr) lam_out[tb[g] + x + (long)NX * y] = lam_in[tb[g] + x + (long)NX * y];
    return;
  }
  const FaceK fku = face_k(0.5 * dt, dx, AH), fkv = face_k(0.5 * dt, dy, AH);
  const double facu = 0.5 * dy * ard1, facv = 0.5 * dx * ard1;
  auto row_of = [&](int y) -> long { return o + xc + (long)NX * (y >= 0 && y < NY ? y : 0); };

  // the u transpose of row y: its loads, and l -> its adjoint in place
  struct URaw {
    TF f[G];
    double D0, D1, vel, Dv;
    uint8_t fm, fc, fp;
  };
  auto fetch_u = [&](int y) -> URaw {
    const long c = row_of(y);
    URaw r;
    r.D0 = Du0[c];
    r.D1 = Du1[c];
    r.vel = uu[c];
    r.Dv = hu[c];
    r.fc = flags[c - o];
    r.fm = flags[c - o - (xc > 0)];
    r.fp = flags[c - o + (xc < NX - 1)];
#pragma unroll
    for (int g = 0; g < G; g++) r.f[g] = fu[tb[g] + c];
    return r;
  };
  auto u_adj = [&](const URaw& r, TF (&l)[G]) {
    FaceC<EX> fc = no_face<EX>();
    if (xin && x <= NX - 2) {
      const bool active = x >= isub && x <= NX - 2 - isub && (r.fc & MB_UFLUX);
      const bool lim_l = SCH != UPSTREAM && x >= 1 && (r.fm & MB_UFLUX);
      const bool lim_r = SCH != UPSTREAM && (r.fp & MB_UFLUX);
      DivFull dv;
      face_setup<SCH>(fc, active, lim_l, lim_r, r.vel, r.Dv, fku, dv);
    }
    const bool upd = xin && x >= 1 + isub && x <= NX - 2 - isub && (r.fc & MB_UUPD);
    CellOp<EX> cu;
    if (upd) cu = CellOp<EX>::make(r.D0, r.D1, dt * facu);
#pragma unroll
    for (int g = 0; g < G; g++) {
      const TF fx = r.f[g], lx = l[g];
      const TF fm1 = from_lower_lane(fx), fp1 = from_upper_lane(fx);
      const TF fp2 = from_upper_lane(fp1);
      const TF mu = upd ? cu.mu(lx, dt, facu) : TF(0);  // d(out x)/d F(x) times lam
      const TF Fbar = mu - from_upper_lane(mu);
      TF q[4];
      face_flux_grad<TF, SCH, DIFF>(fc, fm1, fx, fp1, fp2, AH, dx, q);
      TF acc = upd ? cu.diag(lx) : lx;
      acc += Fbar * q[1];                                   // face x
      acc += from_upper_lane(Fbar * q[0]);                  // face x+1
      acc += from_lower_lane(Fbar * q[2]);                  // face x-1
      acc += from_lower_lane(from_lower_lane(Fbar * q[3])); // face x-2
      l[g] = acc;
    }
  };

  struct Row {
    TF f, acc, mu;
  };
  Row w[G][4] = {};
  // the loads of a row entering the window, read one face ahead
  struct ERaw {
    TF l[G], f[G];
    double D0, D1;
    uint8_t fl;
  };
  auto fetch = [&](int y) -> ERaw {
    const long c = row_of(y);
    ERaw r;
    r.D0 = Dv0[c];
    r.D1 = Dv1[c];
    r.fl = flags[c - o];
#pragma unroll
    for (int g = 0; g < G; g++) {
      r.l[g] = lam_in[tb[g] + c];
      r.f[g] = fv[tb[g] + c];
    }
    return r;
  };
  // row y enters the window (UF: through its u transpose)
  auto enter = [&](int y, ERaw r, const URaw& ur) {
    if constexpr (UF) u_adj(ur, r.l);
    const bool yin = xin && y >= 0 && y < NY;
    const bool upd = yin && y >= 1 + isub && y <= NY - 2 - isub && (r.fl & MB_VUPD);
    CellOp<EX> cu;
    if (upd) cu = CellOp<EX>::make(r.D0, r.D1, dt * facv);
#pragma unroll
    for (int g = 0; g < G; g++) {
      const TF l = r.l[g];
      w[g][3].f = r.f[g];
      w[g][3].acc = upd ? cu.diag(l) : l;
      w[g][3].mu = upd ? cu.mu(l, dt, facv) : TF(0);
    }
  };
  // four rows enter before the first face
  ERaw en = fetch(y0 - 3);
  URaw un{};  // UF: of the next row to enter; else of the next to leave
  if constexpr (AHEAD) un = fetch_u(UF ? y0 - 3 : y0);
  VRaw rn = vraw(d, xc, o, y0 - 2, flags, vv, hv, Dv0, Dv1);
  for (int Y = y0 - 6; Y <= y1; Y++) {
    const ERaw e = en;
    en = fetch(Y + 4);
    URaw ur = un;
    if constexpr (UF) {
      if constexpr (AHEAD) un = fetch_u(Y + 4);
      else ur = fetch_u(Y + 3);
    }
    if (Y >= y0 - 2) {
      const VRaw r = rn;
      rn = vraw(d, xc, o, Y + 1, flags, vv, hv, Dv0, Dv1);
      FaceC<EX> fc = no_face<EX>();
      if (Y >= 0 && Y <= NY - 2) fc = vface<SCH, EX>(d, Y, r, fkv);
#pragma unroll
      for (int g = 0; g < G; g++) {
        const TF Fbar = w[g][1].mu - w[g][2].mu;
        TF gr[4];
        face_flux_grad<TF, SCH, DIFF>(fc, w[g][0].f, w[g][1].f, w[g][2].f, w[g][3].f, AH, dy, gr);
#pragma unroll
        for (int q = 0; q < 4; q++) w[g][q].acc += Fbar * gr[q];
      }
      const int yd = Y - 1;  // complete
      if (yd >= y0 && yd < y1) {
        TF l[G];
#pragma unroll
        for (int g = 0; g < G; g++) l[g] = w[g][0].acc;
        if constexpr (!UF) {
          if constexpr (AHEAD) un = fetch_u(yd + 1);
          else ur = fetch_u(yd);
          u_adj(ur, l);
        }
#pragma unroll
        for (int g = 0; g < G; g++)
          if (out && t0 + g < ntr) lam_out[tb[g] + o + x + (long)NX * yd] = l[g];
      }
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
      w[g][0] = w[g][1];
      w[g][1] = w[g][2];
      w[g][2] = w[g][3];
    }
    enter(Y + 3, e, ur);
  }
}

// ---- transpose of the vertical sub-step ----------------------------------------
// One thread per column and group of tracers.  Marching over the faces
// K' = 0..kmax-1, the window holds levels K'-1..K'+2 (the flux at K'+1/2
// reads them): each level enters with its diagonal part and mu, collects the
// face terms, and is stored when it leaves.  A face is the wk of level K' and
// the wprev of level K'+1 (K' >= 1, or K' = 0 with kshift).
template <typename TF, int SCH>
__global__ __launch_bounds__(256) void k_sub_w_adj(Dims d, int ntr, long ts,
                                                   const TF* __restrict__ f,
                                                   const TF* __restrict__ lam_in,
                                                   TF* __restrict__ lam_out,
                                                   const double* __restrict__ D2,
                                                   const double* __restrict__ D3,
                                                   const double* __restrict__ ww,
                                                   const uint8_t* __restrict__ flags, double dt,
                                                   int kshift, int ngroups, int nchunks, int kc) {
  constexpr bool EX = kExact<TF>;
  constexpr int G = kGroup<TF>;
  // blockIdx.x = column block * nz + z, z = chunk * ngroups + group: the
  // groups and chunks of one column block run together, so the FP64 fields
  // they all read meet in the cache
  const int nz = ngroups * nchunks, bz = (int)(blockIdx.x % nz);
  const int i = (int)(blockIdx.x / nz) * blockDim.x + threadIdx.x;
  const int j = blockIdx.y * blockDim.y + threadIdx.y;
  const int t0 = (bz % ngroups) * G;
  const int kmax = d.kmax;
  // this thread stores levels L0..L1 (chunk bz / ngroups of kc levels); it
  // marches the faces L0-2..L1+1 that reach them, in the order of the whole
  // column, so every stored sum is formed in the same order
  const int L0 = (bz / ngroups) * kc, L1 = min(L0 + kc - 1, kmax);
  if (i >= d.NX || j >= d.NY || t0 >= ntr || L0 > kmax) return;
  const int Fs = max(L0 - 2, 0), Fe = min(L1 + 1, kmax - 1);
  const long NXY = d.NXY, c2 = i + (long)d.NX * j;
  long tb[G];
#pragma unroll
  for (int g = 0; g < G; g++) tb[g] = (long)min(t0 + g, ntr - 1) * ts;
  const bool wcol = (flags[c2] & MB_WCOL) && i <= d.NX - 2 && j <= d.NY - 2;
  if (!wcol) {
    for (int K = L0; K <= L1; K++)
#pragma unroll
      for (int g = 0; g < G; g++)
        if (t0 + g < ntr) lam_out[tb[g] + c2 + NXY * K] = lam_in[tb[g] + c2 + NXY * K];
    return;
  }
  struct Lev {
    TF f, acc, mu;
  };
  Lev w[G][4];
  // a level's loads (read two faces before it enters the window; levels past
  // kmax read level kmax, whose slot is never stored)
  struct Raw {
    TF l[G], f[G];
    double d2, d3;
  };
  auto lv = [&](int L) -> long { return c2 + NXY * (long)min(L, kmax); };
  auto fetch = [&](int L, Raw& r) {
    const long cL = lv(L);
    r.d2 = D2[cL];
    r.d3 = D3[cL];
#pragma unroll
    for (int g = 0; g < G; g++) {
      r.l[g] = lam_in[tb[g] + cL];
      r.f[g] = f[tb[g] + cL];
    }
  };
  auto enter = [&](int L, int q, const Raw& r) {
    const bool kdo = L <= kmax && L >= 1 && L <= kmax - kshift;
    CellOp<EX> cw;
    if (kdo) cw = CellOp<EX>::make(r.d2, r.d3, dt);
#pragma unroll
    for (int g = 0; g < G; g++) {
      const TF l = r.l[g];
      w[g][q].f = r.f[g];
      w[g][q].acc = kdo ? cw.diag(l) : l;
      w[g][q].mu = kdo ? cw.mu(l, dt, 1.0) : TF(0);
    }
  };
  // the window at face Fs holds levels Fs-1..Fs+2 (level -1 is zero)
  {
    Raw r0, r1, r2, r3;
    fetch(max(Fs - 1, 0), r0);
    fetch(Fs, r1);
    fetch(Fs + 1, r2);
    fetch(Fs + 2, r3);
    if (Fs >= 1) {
      enter(Fs - 1, 0, r0);
    } else {
#pragma unroll
      for (int g = 0; g < G; g++) w[g][0] = Lev{TF(0), TF(0), TF(0)};
    }
    enter(Fs, 1, r1);
    enter(Fs + 1, 2, r2);
    enter(Fs + 2, 3, r3);
  }
  Raw rq0, rq1;  // levels K'+3, K'+4
  fetch(Fs + 3, rq0);
  fetch(Fs + 4, rq1);
  // D2 at K', K'+1, K'+2 and ww at K', K'+1, K'+2, loaded two faces ahead
  double dq[3], wq[3];
#pragma unroll
  for (int q = 0; q < 3; q++) {
    dq[q] = D2[lv(Fs + q)];
    wq[q] = ww[lv(Fs + q)];
  }
  for (int Kf = Fs; Kf <= Fe; Kf++) {
    // level 0 is never updated (mu = 0), so at K' = 0 Fbar is -mu(1) with
    // kshift and 0 without
    const bool used = Kf >= 1 || kshift;
    WFace<EX> wf;
    DivFull dv;
    wface_setup<SCH>(wf, wq[0], dt, dq[0], dq[1], true, dv);
    const bool lim_up = SCH != UPSTREAM && Kf > 1 - kshift;
    const bool lim_dn = SCH != UPSTREAM && Kf < kmax - 1;
#pragma unroll
    for (int g = 0; g < G; g++) {
      const TF Fbar = used ? w[g][1].mu - w[g][2].mu : TF(0);
      const TF fkm1 = Kf >= 1 ? w[g][0].f : TF(0), fk = w[g][1].f, fk1 = w[g][2].f;
      const TF fk2 = Kf + 2 <= kmax ? w[g][3].f : fk;
      TF gr[4];
      w_flux_grad<TF, SCH>(wf, lim_up, lim_dn, fkm1, fk, fk1, fk2, gr);
      // (a slot past either end of the column is never stored)
#pragma unroll
      for (int q = 0; q < 4; q++) w[g][q].acc += Fbar * gr[q];
    }
    if (Kf - 1 >= L0 && Kf - 1 <= L1) {
#pragma unroll
      for (int g = 0; g < G; g++)
        if (t0 + g < ntr) lam_out[tb[g] + c2 + NXY * (Kf - 1)] = w[g][0].acc;
    }
#pragma unroll
    for (int g = 0; g < G; g++) {
      w[g][0] = w[g][1];
      w[g][1] = w[g][2];
      w[g][2] = w[g][3];
    }
    enter(Kf + 3, 3, rq0);
    rq0 = rq1;
    fetch(Kf + 5, rq1);
#pragma unroll
    for (int q = 0; q < 2; q++) {
      dq[q] = dq[q + 1];
      wq[q] = wq[q + 1];
    }
    dq[2] = D2[lv(Kf + 3)];
    wq[2] = ww[lv(Kf + 3)];
  }
  // after the last face, levels kmax-1 and kmax are complete
  if (Fe == kmax - 1) {
#pragma unroll
    for (int g = 0; g < G; g++) {
      if (t0 + g < ntr) {
        if (kmax - 1 >= L0 && kmax - 1 <= L1) lam_out[tb[g] + c2 + NXY * (kmax - 1)] = w[g][0].acc;
        if (L1 == kmax) lam_out[tb[g] + c2 + NXY * kmax] = w[g][1].acc;
      }
    }
  }
}

// ---- launchers --------------------------------------------------------------------
hipError_t launch_heights(hipStream_t st, Dims d, const uint8_t* flags, const double* ho,
                          const double* uu, const double* vv, const double* ww,
                          double* const D[5], double dt, double dx, double dy, double ard1,
                          int scheme, int kshift) {
  hipLaunchKernelGGL(k_heights, dim3((d.NX + 63) / 64, (d.NY + 3) / 4, d.kmax + 1), dim3(64, 4),
                     0, st, d, flags, ho, uu, vv, ww, D[0], D[1], D[2], D[3], D[4], dt, dx, dy,
                     ard1, scheme == UPSTREAM ? 0 : 1, kshift);
  return hipGetLastError();
}

// f(scheme, diffusion) with both as compile-time constants
#define GT_H(S) (AH > 0.0 ? GT_H1(S, true) : GT_H1(S, false))
#define GT_H_SCHEMES()                        \
  switch (scheme) {                           \
    case UPSTREAM: GT_H(UPSTREAM); break;     \
    case P2: GT_H(P2); break;                 \
    case SUPERBEE: GT_H(SUPERBEE); break;     \
    case MUSCL: GT_H(MUSCL); break;           \
    case P2_PDM: GT_H(P2_PDM); break;         \
    default: return hipErrorInvalidValue;     \
  }                                           \
  return hipGetLastError()

template <typename TF, int SCH, bool DIFF>
static void launch_h_one(hipStream_t st, Dims d, int dir, int ntr, long ts, const TF* fin,
                         TF* fout, const double* Dio, const double* Dn, const double* vel,
                         const double* Dv, const uint8_t* flags, double dt, double dx, double dy,
                         double ard1, double AH) {
  const int ng = (ntr + kGroup<TF> - 1) / kGroup<TF>;
  const dim3 gv((d.NX + 63) / 64, (d.NY + kVRows<TF> - 1) / kVRows<TF>, (d.kmax + 1) * ng);
  if (dir == 0)
    hipLaunchKernelGGL((k_sub_u<TF, SCH, DIFF>),
                       dim3((d.NX + kUOutF - 1) / kUOutF, (d.NY + 3) / 4, d.kmax + 1),
                       dim3(64, 4), 0, st, d, ntr, ts, fin, fout, Dio, Dn, vel, Dv, flags, dt, dx,
                       dy, ard1, AH);
  else
    hipLaunchKernelGGL((k_sub_v<TF, SCH, DIFF>), gv, dim3(64), 0, st, d, ntr, ts, fin, fout, Dio,
                       Dn, vel, Dv, flags, dt, dx, dy, ard1, AH, ng);
}

template <typename TF, int SCH, bool DIFF>
static void launch_uv_adj_one(hipStream_t st, Dims d, bool ufirst, int ntr, long ts, const TF* fu,
                              const TF* fv, const TF* lam_in, TF* lam_out, const double* Du0,
                              const double* Du1, const double* Dv0, const double* Dv1,
                              const double* uu, const double* hu, const double* vv,
                              const double* hv, const uint8_t* flags, double dt, double dx,
                              double dy, double ard1, double AH) {
  const int ng = (ntr + kGroup<TF> - 1) / kGroup<TF>;
  const int nsx = (d.NX + kUOutA - 1) / kUOutA;
  int rows = kUVRows<TF>;
  while (rows > 4 && (long)nsx * ((d.NY + rows - 1) / rows) * d.kmax * ng < kUVWaves) rows /= 2;
  const dim3 g(nsx, (d.NY + rows - 1) / rows, (d.kmax + 1) * ng);
  if (ufirst)
    hipLaunchKernelGGL((k_sub_uv_adj<TF, SCH, DIFF, true>), g, dim3(64), 0, st, d, ntr, ts, fu,
                       fv, lam_in, lam_out, Du0, Du1, Dv0, Dv1, uu, hu, vv, hv, flags, dt, dx, dy,
                       ard1, AH, ng, rows);
  else
    hipLaunchKernelGGL((k_sub_uv_adj<TF, SCH, DIFF, false>), g, dim3(64), 0, st, d, ntr, ts, fu,
                       fv, lam_in, lam_out, Du0, Du1, Dv0, Dv1, uu, hu, vv, hv, flags, dt, dx, dy,
                       ard1, AH, ng, rows);
}

template <typename TF, bool ADJ, int SCH>
static void launch_w_one(hipStream_t st, Dims d, int ntr, long ts, const TF* a, const TF* b,
                         TF* out, const double* D2, const double* D3, const double* ww,
                         const uint8_t* flags, double dt, int kshift) {
  // A column march has one wavefront per 64 columns and tracer group; where
  // that leaves the chip short of wavefronts (one FP64 tracer on a small
  // grid) the columns are cut into up to four chunks of at least 8 levels.
  const int ng = (ntr + kGroup<TF> - 1) / kGroup<TF>;
  const long waves = (long)((d.NX + 63) / 64) * d.NY * ng;
  int nch = 1;
  while (nch < 4 && waves * nch < kWaveTarget && d.kmax / (nch + 1) >= 8) nch++;
  const int nlev = ADJ ? d.kmax + 1 : d.kmax;  // levels split: 0..kmax, resp. 1..kmax
  const int kc = (nlev + nch - 1) / nch;
  const int nchunks = (nlev + kc - 1) / kc;
  const dim3 g((unsigned)(((d.NX + 63) / 64) * ng * nchunks), (d.NY + 3) / 4, 1);
  if constexpr (ADJ) {
    hipLaunchKernelGGL((k_sub_w_adj<TF, SCH>), g, dim3(64, 4), 0, st, d, ntr, ts, a, b, out, D2,
                       D3, ww, flags, dt, kshift, ng, nchunks, kc);
  } else {
    (void)b;
    hipLaunchKernelGGL((k_sub_w<TF, SCH>), g, dim3(64, 4), 0, st, d, ntr, ts, a, out, D2, D3, ww,
                       flags, dt, kshift, ng, nchunks, kc);
  }
}

template <typename TF, bool ADJ>
static hipError_t launch_w(hipStream_t st, Dims d, int ntr, long ts, const TF* a, const TF* b,
                           TF* out, const double* D2, const double* D3, const double* ww,
                           const uint8_t* flags, double dt, int scheme, int kshift) {
  switch (scheme) {
    case UPSTREAM: launch_w_one<TF, ADJ, UPSTREAM>(st, d, ntr, ts, a, b, out, D2, D3, ww, flags, dt, kshift); break;
    case P2: launch_w_one<TF, ADJ, P2>(st, d, ntr, ts, a, b, out, D2, D3, ww, flags, dt, kshift); break;
    case SUPERBEE: launch_w_one<TF, ADJ, SUPERBEE>(st, d, ntr, ts, a, b, out, D2, D3, ww, flags, dt, kshift); break;
    case MUSCL: launch_w_one<TF, ADJ, MUSCL>(st, d, ntr, ts, a, b, out, D2, D3, ww, flags, dt, kshift); break;
    case P2_PDM: launch_w_one<TF, ADJ, P2_PDM>(st, d, ntr, ts, a, b, out, D2, D3, ww, flags, dt, kshift); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <typename TF>
hipError_t launch_sub_h(hipStream_t st, Dims d, int dir, int ntr, long ts, const TF* fin, TF* fout,
                        const double* Dio, const double* Dn, const double* vel, const double* Dv,
                        const uint8_t* flags, double dt, double dx, double dy, double ard1,
                        int scheme, double AH) {
#define GT_H1(S, DF)                                                                          \
  launch_h_one<TF, S, DF>(st, d, dir, ntr, ts, fin, fout, Dio, Dn, vel, Dv, flags, dt, dx, dy, \
                          ard1, AH)
  GT_H_SCHEMES();
#undef GT_H1
}

template <typename TF>
hipError_t launch_sub_uv_adj(hipStream_t st, Dims d, bool ufirst, int ntr, long ts, const TF* fu,
                             const TF* fv, const TF* lam_in, TF* lam_out, const double* Du0,
                             const double* Du1, const double* Dv0, const double* Dv1,
                             const double* uu, const double* hu, const double* vv,
                             const double* hv, const uint8_t* flags, double dt, double dx,
                             double dy, double ard1, int scheme, double AH) {
#define GT_H1(S, DF)                                                                            \
  launch_uv_adj_one<TF, S, DF>(st, d, ufirst, ntr, ts, fu, fv, lam_in, lam_out, Du0, Du1, Dv0,  \
                               Dv1, uu, hu, vv, hv, flags, dt, dx, dy, ard1, AH)
  GT_H_SCHEMES();
#undef GT_H1
}
#undef GT_H
#undef GT_H_SCHEMES

template <typename TF>
hipError_t launch_sub_w(hipStream_t st, Dims d, int ntr, long ts, const TF* fin, TF* fout,
                        const double* D2, const double* D3, const double* ww,
                        const uint8_t* flags, double dt, int scheme, int kshift) {
  return launch_w<TF, false>(st, d, ntr, ts, fin, nullptr, fout, D2, D3, ww, flags, dt, scheme,
                             kshift);
}

template <typename TF>
hipError_t launch_sub_w_adj(hipStream_t st, Dims d, int ntr, long ts, const TF* f,
                            const TF* lam_in, TF* lam_out, const double* D2, const double* D3,
                            const double* ww, const uint8_t* flags, double dt, int scheme,
                            int kshift) {
  return launch_w<TF, true>(st, d, ntr, ts, f, lam_in, lam_out, D2, D3, ww, flags, dt, scheme,
                            kshift);
}

#define GT_INST(TF)                                                                            \
  template hipError_t launch_sub_h<TF>(hipStream_t, Dims, int, int, long, const TF*, TF*,      \
                                       const double*, const double*, const double*,            \
                                       const double*, const uint8_t*, double, double, double,  \
                                       double, int, double);                                   \
  template hipError_t launch_sub_uv_adj<TF>(                                                   \
      hipStream_t, Dims, bool, int, long, const TF*, const TF*, const TF*, TF*, const double*, \
      const double*, const double*, const double*, const double*, const double*,               \
      const double*, const double*, const uint8_t*, double, double, double, double, int,       \
      double);                                                                                 \
  template hipError_t launch_sub_w<TF>(hipStream_t, Dims, int, long, const TF*, TF*,           \
                                       const double*, const double*, const double*,            \
                                       const uint8_t*, double, int, int);                      \
  template hipError_t launch_sub_w_adj<TF>(hipStream_t, Dims, int, long, const TF*, const TF*, \
                                           TF*, const double*, const double*, const double*,   \
                                           const uint8_t*, double, int, int);
GT_INST(float)
GT_INST(double)
#undef GT_INST

}  // namespace gt
