// gt_strip_impl.h -- the HALFSPLIT transport step as two strip kernels.
//
// The step u/2 + v/2 + w + v/2 + u/2 (src/3d/advection_3d.F90:439-547 of
// getm-model/code) is cut after the first v/2:
//   k_strip_uv   u/2 then v/2 at one level; writes the tracers f2 and the
//                layer heights d2 after them (work fields in HBM);
//   k_strip_wvu  w at one level from f2 at the levels K-2..K+2, then v/2 and
//                u/2; writes the result and hires.
// Neither kernel carries state from level to level, so every (strip, level,
// tracer group) is an independent work item.
//
// A work item is one wavefront.  Lane l owns column x = 60*sx - 2 + l; the
// wavefront marches up a strip of rows, one row per step, so
//   * i-neighbours (the u sub-steps) come from the adjacent lanes through DPP
//     wave shifts, and lanes 2..61 have all four ghost columns the two-cell
//     stencil of a flux and the two fluxes of an update need;
//   * j-neighbours (the v sub-steps) are earlier rows of the march, kept in a
//     four-row register window;
//   * k-neighbours (w) are loads of the neighbouring levels of f2.
// There is no LDS and no barrier.  Work shared by the tracers of a group is
// done once per row: the layer-height trajectory (FP64), and per face the
// upwind direction, whether the limiter applies (masks), the Courant number
// and the limiter constants that depend on it.
//
// Two arithmetic flavours:
//   EXACT (TF=double): the reference's expressions in the reference's order,
//     so results are bit-identical to the per-sub-step kernels and the CPU
//     restatement.
//   fast (TF=float): tracer and flux arithmetic in FP32 with a division-free
//     form of each limiter (phi(r)*deltaf as a min/max of products, the sign
//     of deltaf choosing min or max) and reciprocals for the face constants;
//     the layer heights stay FP64 and the cell update (Dio*f - dt*advn)/Di is
//     f + [f*(Dio-Di)/Di - dF*(dt*c/Di)] with the two factors formed once per
//     cell (Dio-Di in FP64, the rest in FP32, as the Courant numbers) and
//     shared by the tracers.
//
// Which cells each sub-step updates follows the reference exactly (the isub /
// jsub bounds of adv_split_u/v.F90 and the column range of adv_split_w.F90),
// so cells the reference leaves alone pass through unchanged.
#pragma once

#include <type_traits>

#include "gt_batched.h"

namespace gt {

// 1/x to about one FP64 ulp: hardware estimate and one Newton step (fast path)
__device__ __forceinline__ double rcp_nr(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double e = __builtin_fma(-x, r, 1.0);
  return __builtin_fma(r, e, r);
}

// ---- the divisions of the exact flavour ----------------------------------------
// The compiler's a/b is v_div_scale (twice), v_rcp, two Newton steps for
// y = 1/b, q0 = a*y, r = a - b*q0, q = q0 + r*y (v_div_fmas) and v_div_fixup:
// 11 instructions.  Where nothing needs scaling the scale and fixup steps
// pass their operands through, so the Newton steps and the last three
// operations alone give the same bits, and y is formed once for every
// quotient over the same b (the cell updates of the tracers, P2-PDM's
// 2r/(cfl+1e-10), the division by dx).  They need a remainder that is exact
// and a quotient that is normal; DivNewton tests for what takes that away and
// gives a strip up where it fires (asked after the first row, the fourth and
// every four), which is then marched again with DivFull:
//   * a numerator below 2^-969, zero aside: its remainder ends in the
//     denormals, rounded, or flushed to a zero that looks exact (a < 2^-1021
//     over |b| < 1);
//   * an infinity, a NaN, a zero b or an overflow (q infinite or NaN), and a
//     denormal q (rounded twice).
// What is known of a quotient (Quot) saves part of the test.  Not covered: |b|
// of 2^1022 or more, Courant numbers beyond 2^50, and a quotient within one
// rounding of 2^-1075.
// A zero numerator gives +0 where the full sequence keeps its sign.
// Cost and reach (400 x 400 x 40, two tracers, P2-PDM): 380 us where nothing
// fires (375 with the remainder's class as the only test, 455 with full
// divisions alone); tails of a tracer that fade out below 1e-292 fire it
// (look_ahead has their figures), a field that lies there as a whole takes 441
// (469 with full divisions alone).
struct Den {
  double b, y;
};
// what is known of a quotient.  kNonzero: its numerator is not zero where it is
// used.  kFace: a Courant number, whose last bits vanish in 1 - c, 1 - 2c and
// c + 1e-10 where it is tiny.  kRatio: twice a tested quotient on top, so a
// numerator of 2^-1021 or more, whose remainder tells the rest (one that rounds
// to zero leaves q0 the nearest).  kBound: P2-PDM's 2/(1-c), tested with c, and
// NaN for c = 1, which the min takes for the infinity it stands for.
enum Quot { kAny, kNonzero, kFace, kRatio, kBound };
struct DivFull {
  static constexpr bool kTests = false;
  __device__ __forceinline__ Den den(double b) const { return {b, 0.0}; }
  template <Quot Q = kAny>
  __device__ __forceinline__ double over(double a, const Den& d, bool) const {
    return a / d.b;
  }
  template <Quot Q = kAny>
  __device__ __forceinline__ double div(double a, double b, bool) const {
    return a / b;
  }
  __device__ __forceinline__ void pin() const {}
  __device__ __forceinline__ bool stop() const { return false; }
};
struct DivNewton {
  uint64_t bad = 0;    // the lanes it fired on, up to the last pin()
  bool fired = false;  // and since
  static constexpr bool kTests = true;
  // below 2^-969 and not zero: by the bits past the sign, less one, which
  // makes a zero the largest
  static __device__ __forceinline__ bool tiny(double a) {
    const uint64_t m = (__builtin_bit_cast(uint64_t, a) << 1) - 1;
    return (uint32_t)(m >> 32) < (1023 - 969) << 21;
  }
  __device__ __forceinline__ Den den(double b) const {
    double y = __builtin_amdgcn_rcp(b);
    y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
    y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
    return {b, y};
  }
  // a/b; used: whether this lane's quotient reaches a result
  template <Quot Q = kAny>
  __device__ __forceinline__ double over(double a, const Den& d, bool used) {
    constexpr int kNanInfDenorm = 0x1 | 0x2 | 0x4 | 0x10 | 0x80 | 0x200;
    const double q0 = a * d.y;
    const double r = __builtin_fma(-d.b, q0, a);
    const double q = __builtin_fma(r, d.y, q0);
    if constexpr (Q == kNonzero) {
      fired |= used & ((__builtin_fabs(a) < 0x1p-969) | __builtin_amdgcn_class(q, kNanInfDenorm));
    } else if constexpr (Q == kAny) {
      fired |= used & (tiny(a) | __builtin_amdgcn_class(q, kNanInfDenorm));
    } else if constexpr (Q != kBound) {
      fired |= used & __builtin_amdgcn_class(r, kNanInfDenorm);
    }
    return q;
  }
  template <Quot Q = kAny>
  __device__ __forceinline__ double div(double a, double b, bool used) {
    return over<Q>(a, den(b), used);
  }
  // fires for a tracer value that a quotient will fire for, from its high word
  // (values below 2^-1042 pass)
  __device__ __forceinline__ void look(uint32_t hi, bool used) {
    fired |= used & ((hi << 1) - 1 < (1023 - 969) << 21);
  }
  // ends a section of the row: the tests of the section's quotients stay in
  // it (left to the compiler they gather at the row's end and keep every
  // remainder in registers until there)
  __device__ __forceinline__ void pin() {
    bad |= __builtin_amdgcn_ballot_w64(fired);
    asm volatile("" : "+s"(bad));
    fired = false;
  }
  __device__ __forceinline__ bool stop() const { return bad != 0; }
};

// ---- one face of a sweep -----------------------------------------------------

template <bool EXACT>
struct FaceC;
// EXACT: the values the reference's flux expression reads
template <>
struct FaceC<true> {
  double vel, cfl, Dv, E;  // E = 2/(1-cfl), P2-PDM's third bound, formed once
  Den c1;                  // cfl + 1e-10, the denominator of its first
  bool active, left, lim;  // carries a flux, goes right (upwind cell on the left), is limited
};
// fast: vel = 0 for an inactive face, g = 0 where the limiter does not apply
template <>
struct FaceC<false> {
  float vel, g, A, al, E, kA;
  bool right;
};

// the sweep's constants: dti = splitfac*dt, the face length dlen, and for
// the fast path dti/dlen and AH/dlen (0 without diffusion)
struct FaceK {
  double dti, dlen, cscale, kscale;
  Den len;  // dlen as a denominator
};
__device__ __forceinline__ FaceK face_k(double dti, double dlen, double AH) {
  return {dti, dlen, dti / dlen, AH > 0.0 ? AH / dlen : 0.0, DivNewton{}.den(dlen)};
}

// face constants from the transport (vel), layer height (Dv) and masks;
// lim_l/lim_r: the flux mask of the upwind neighbour allows the limiter
// (adv_split_u.F90:219-265, adv_split_v.F90:77-119)
template <int SCH, typename Div>
__device__ __forceinline__ void face_setup(FaceC<true>& fc, bool active, bool lim_l, bool lim_r,
                                           double vel, double Dv, const FaceK& k, Div& dv) {
  // The exact path is branch-free like the fast one: every operand is formed
  // and the result selected, so the division chains of neighbouring faces and
  // tracers share one basic block and interleave; a lane whose value is not
  // selected may compute inf or NaN, which is never used.  One division
  // chain serves both directions: the reference's vel/Dv*dti/dlen going
  // right, -vel/Dv*dti/dlen going left, with the operand selected first.
  fc.vel = vel;
  fc.Dv = Dv;
  const bool left = vel > 0.0;
  const bool lim = active & (SCH != UPSTREAM) & (left ? lim_l : lim_r);
  fc.active = active;
  fc.left = left;
  fc.lim = lim;
  const double c =
      dv.template over<kFace>(dv.template div<kFace>(left ? vel : -vel, Dv, lim) * k.dti, k.len, lim);
  fc.cfl = lim ? c : 0.0;
  if constexpr (SCH == P2_PDM) {
    fc.E = dv.template div<kBound>(2.0, 1.0 - fc.cfl, lim);
    fc.c1 = dv.den(fc.cfl + 1.e-10);
  } else {
    fc.E = 0.0;
    fc.c1 = {1.0, 1.0};
  }
}

// adv_interfacial_reconstruction (src/2d/advection.F90:806-845), branch-free:
// every operation of reconstruct() in its order, P2-PDM's 2/(1-cfl) taken
// from the face (E) instead of formed per tracer.  Returns the limited value
// and sets take where the reference returns it (lim, the limiter applies,
// and deltaf*deltafu > 0 for the TVD schemes, lim for P2, never for upstream)
// -- fu otherwise -- so the caller folds this choice into its own select of
// the face's value
template <int SCH, typename Div>
__device__ __forceinline__ double reconstruct_bf(double cfl, double E, const Den& c1, double fuu,
                                                 double fu, double fd, bool lim, bool& take,
                                                 Div& dv) {
  const double deltaf = fd - fu;
  const double deltafu = fu - fuu;
  if constexpr (SCH == UPSTREAM) {
    (void)E; (void)cfl; (void)c1; (void)lim; (void)dv;
    take = false;
    return fu;
  } else if constexpr (SCH == P2) {
    (void)E; (void)c1; (void)dv;
    take = lim;
    return reconstruct_p2<double>(cfl, fu, deltafu, deltaf);
  } else {
    // The reference's min/max are the hardware's: where the result is
    // selected (deltaf*deltafu > 0) the ratio is positive and, with
    // cfl >= 0, no operand is NaN and no two are zeros of opposite sign, so
    // v_min_f64 / v_max_f64 pick the operand the comparison form picks
    take = lim & (deltaf * deltafu > 0.0);
    const double ratio = dv.template div<kNonzero>(deltafu, deltaf, take);
    double limiter;
    if constexpr (SCH == P2_PDM) {
      const double one6th = 1.0 / 6.0;
      const double x = one6th * (1.0 - 2.0 * cfl);
      limiter = (0.5 + x) + (0.5 - x) * ratio;
      limiter = __builtin_fmin(__builtin_fmin(dv.template over<kRatio>(2.0 * ratio, c1, take), limiter), E);
    } else if constexpr (SCH == SUPERBEE) {
      (void)E;
      limiter = __builtin_fmax(__builtin_fmin(2.0 * ratio, 1.0), __builtin_fmin(ratio, 2.0));
    } else {  // MUSCL
      (void)E;
      limiter = __builtin_fmin(__builtin_fmin(2.0 * ratio, 0.5 * (1.0 + ratio)), 2.0);
    }
    return fu + 0.5 * limiter * (1.0 - cfl) * deltaf;
  }
}

template <int SCH, typename Div>
__device__ __forceinline__ void face_setup(FaceC<false>& fc, bool active, bool lim_l, bool lim_r,
                                           double vel, double Dv, const FaceK& k, Div&) {
  const bool right = !(vel > 0.0);
  const bool lim = active & (SCH != UPSTREAM) & (right ? lim_r : lim_l);
  // the Courant number feeds FP32 arithmetic only: formed in FP32
  const float c0 =
      __builtin_fabsf((float)vel) * (float)k.cscale * __builtin_amdgcn_rcpf((float)Dv);
  const float c = lim ? c0 : 0.0f;
  fc.right = right;
  fc.vel = active ? (float)vel : 0.0f;
  fc.g = lim ? 0.5f * (1.0f - c) : 0.0f;
  fc.A = 2.0f * __builtin_amdgcn_rcpf(c + 1.e-10f);
  fc.al = 0.5f + (1.0f / 6.0f) * (1.0f - 2.0f * c);
  fc.E = 2.0f * __builtin_amdgcn_rcpf(1.0f - c);
  fc.kA = active ? (float)(k.kscale * Dv) : 0.0f;
}

// the limiter, division-free FP32 form.  With deltaf = fd-fu,
// deltafu = fu-fuu, r = deltafu/deltaf and g = (1-c)/2 the reference returns
// fu + g*phi(r)*deltaf when deltaf*deltafu > 0 (else fu); phi(r)*deltaf is
// the min (deltaf > 0) or max (deltaf < 0) of the branch terms times deltaf.
// P2-PDM: A = 2/(c+1e-10), al = 1/2 + (1-2c)/6, E = 2/(1-c).
// (adv_interfacial_reconstruction, src/2d/advection.F90:785-879)
// On the lanes that take the limited value deltaf and deltafu share a sign,
// and the branch terms of deltaf < 0 are those of |deltaf|, |deltafu|
// negated, each rounding alike, so the max there is minus the min over the
// magnitudes: one min (abs taken as operand modifiers) whose sign is flipped
// where deltaf is negative (one three-operand bit operation) gives bit for
// bit the min/max selected by the sign.  (Not a copied sign: P2-PDM's terms
// are negative above Courant number 1.)  No divergent branch; fused
// multiply-adds are written out where they shorten the chain.
template <int SCH>
__device__ __forceinline__ float rec_fast(float fuu, float fu, float fd, float g, float A,
                                          float al, float E) {
  const float df = fd - fu, du = fu - fuu;
  if constexpr (SCH == P2) {
    // al*df + (1-al)*du = du + al*(df-du)
    return __builtin_fmaf(g, __builtin_fmaf(al, df - du, du), fu);
  } else if constexpr (SCH == UPSTREAM) {
    return fu;
  } else {
    const float adf = __builtin_fabsf(df), adu = __builtin_fabsf(du);
    float m;
    if constexpr (SCH == P2_PDM) {
      m = __builtin_fminf(__builtin_fminf(A * adu, __builtin_fmaf(al, adf - adu, adu)),
                          E * adf);
    } else if constexpr (SCH == SUPERBEE) {
      const float a2 = 2.0f * adu, b2 = 2.0f * adf;
      m = __builtin_fmaxf(__builtin_fminf(a2, adf), __builtin_fminf(adu, b2));
    } else {  // MUSCL
      const float a2 = 2.0f * adu, b2 = 2.0f * adf, h = 0.5f * (adf + adu);
      m = __builtin_fminf(__builtin_fminf(a2, h), b2);
    }
    const uint32_t ms = __builtin_bit_cast(uint32_t, m) ^
                        (__builtin_bit_cast(uint32_t, df) & 0x80000000u);
    const float r = __builtin_fmaf(g, __builtin_bit_cast(float, ms), fu);
    return df * du > 0.0f ? r : fu;
  }
}

// flux through the face between cells X and X+1 of a sweep, from the cells
// X-1, X, X+1, X+2 (fm1, f0, fp1, fp2)
// DIFF: horizontal diffusion on (AH > 0), fixed at compile time
template <typename TF, int SCH, bool DIFF, typename Div>
__device__ __forceinline__ TF face_flux(const FaceC<true>& fc, TF fm1, TF f0, TF fp1, TF fp2,
                                        double AH, const FaceK& k, Div& dv) {
  // upwind operands selected first, then one reconstruction for both
  // directions (left: fm1, f0, fp1; right: fp2, fp1, f0; branch-free, see
  // face_setup)
  const TF fuu = fc.left ? fm1 : fp2, fd = fc.left ? fp1 : f0;
  const TF fu0 = fc.left ? f0 : fp1;
  bool take;
  const TF rr = reconstruct_bf<SCH>(fc.cfl, fc.E, fc.c1, fuu, fu0, fd, fc.lim, take, dv);
  TF fl = fc.vel * (take ? rr : fu0);
  if constexpr (DIFF) fl = fl - dv.over(AH * fc.Dv * (fp1 - f0), k.len, fc.active);
  return fc.active ? fl : TF(0);
}

template <typename TF, int SCH, bool DIFF, typename Div>
__device__ __forceinline__ TF face_flux(const FaceC<false>& fc, TF fm1, TF f0, TF fp1, TF fp2,
                                        double /*AH*/, const FaceK&, Div&) {
  const TF fuu = fc.right ? fp2 : fm1;
  const TF fu0 = fc.right ? fp1 : f0;
  const TF fd = fc.right ? f0 : fp1;
  const TF fu = rec_fast<SCH>(fuu, fu0, fd, fc.g, fc.A, fc.al, fc.E);
  TF fl = fc.vel * fu;
  if constexpr (DIFF) fl = __builtin_fmaf(-fc.kA, fp1 - f0, fl);
  return fl;
}

// the tracer update of one cell of a horizontal sub-step: the reference's
// (Dio*fo - dt*advn)/Dn, advn = frac*(Fc*dlen - Fm*dlen)*ard1 (frac: splitfac)
// (adv_split_u.F90:267-286), in the reference's order (EXACT); computed on
// every lane and selected by upd (advn_out is 0 where the cell is not
// updated)
template <typename Div>
__device__ __forceinline__ double cell_update_exact(bool upd, double Dio, const Den& Dn, double fo,
                                                    double Fc, double Fm, double frac,
                                                    double dlen, double ard1, double dt,
                                                    double* advn_out, Div& dv) {
  const double advn = frac * (Fc * dlen - Fm * dlen) * ard1;
  *advn_out = upd ? advn : 0.0;
  const double fn = dv.over(Dio * fo - dt * advn, Dn, upd);
  return upd ? fn : fo;
}

// fast: the same as fo + [fo*(Dio-Dn)/Dn - (Fc-Fm)*(dt*splitfac*dlen*ard1/Dn)]:
// the two factors are formed once per cell in FP32 from the FP64 layer
// heights (Dio-Dn taken in FP64, then rounded) and shared by the tracers
// (CellK); the bracket is a small correction, so their few FP32 roundings
// are far below the final rounding of fo + correction.
// A cell that is not updated is selected, not given zero factors: a NaN or an
// infinity times zero is NaN, which would walk through land a cell per sub-step.
struct CellK {
  float am1, b;
};
__device__ __forceinline__ CellK cell_factors(double Dio, double Dn, double dtc) {
  const float r = __builtin_amdgcn_rcpf((float)Dn);
  return {(float)(Dio - Dn) * r, (float)dtc * r};
}
__device__ __forceinline__ float cell_update_fast(bool upd, const CellK& k, float fo, float Fc,
                                                  float Fm) {
  const float fn = fo + __builtin_fmaf(fo, k.am1, -(Fc - Fm) * k.b);
  return upd ? fn : fo;
}

// ---- vertical faces (adv_split_w.F90:249-277) --------------------------------
template <bool EXACT>
struct WFace;
template <>
struct WFace<true> {
  double w, cfl, E;
  Den c1;  // as in FaceC
};
template <>
struct WFace<false> {
  float w, g, A, al, E;
};

// face k+1/2 of a column: w = ww(k), cfl from the layer heights either side
// (used: whether the face carries a flux that reaches a result)
template <int SCH, typename Div>
__device__ __forceinline__ void wface_setup(WFace<true>& wf, double w, double dt, double Dlo,
                                            double Dhi, bool used, Div& dv) {
  wf.w = w;
  wf.cfl = dv.template div<kFace>(__builtin_fabs(w) * dt, 0.5 * (Dlo + Dhi), used);
  if constexpr (SCH == P2_PDM) {
    wf.E = dv.template div<kBound>(2.0, 1.0 - wf.cfl * 1.0, used);
    wf.c1 = dv.den(wf.cfl * 1.0 + 1.e-10);
  } else {
    wf.E = 0.0;
    wf.c1 = {1.0, 1.0};
  }
}
template <int SCH, typename Div>
__device__ __forceinline__ void wface_setup(WFace<false>& wf, double w, double dt, double Dlo,
                                            double Dhi, bool, Div&) {
  const float c =
      __builtin_fabsf((float)w) * (float)(2.0 * dt) * __builtin_amdgcn_rcpf((float)(Dlo + Dhi));
  wf.w = (float)w;
  wf.g = 0.5f * (1.0f - c);
  wf.A = 2.0f * __builtin_amdgcn_rcpf(c + 1.e-10f);
  wf.al = 0.5f + (1.0f / 6.0f) * (1.0f - 2.0f * c);
  wf.E = 2.0f * __builtin_amdgcn_rcpf(1.0f - c);
}

// flux at face k+1/2 from the levels k-1..k+2; lim_up / lim_dn: whether the
// limiter applies going up / down at this face (above level 1-kshift, below
// kmax-1).  Branch-free, as the horizontal faces
template <int SCH, typename Div>
__device__ __forceinline__ double wflux_exact(const WFace<true>& wf, bool lim_up, bool lim_dn,
                                              double fkm1, double fk, double fk1, double fk2,
                                              Div& dv) {
  const bool up = wf.w > 0.0;
  const double fu = up ? fk : fk1, fuu = up ? fkm1 : fk2, fd = up ? fk1 : fk;
  bool take;
  const double rr = reconstruct_bf<SCH>(wf.cfl * 1.0, wf.E, wf.c1, fuu, fu, fd,
                                        up ? lim_up : lim_dn, take, dv);
  return wf.w * (take ? rr : fu);
}

// the same in FP32, the limiter switched off by g = 0
template <int SCH>
__device__ __forceinline__ float wflux_fast(const WFace<false>& wf, bool lim_up, bool lim_dn,
                                            float fkm1, float fk, float fk1, float fk2) {
  const bool up = wf.w > 0.0f;
  const float fu = up ? fk : fk1, fuu = up ? fkm1 : fk2, fd = up ? fk1 : fk;
  const bool lim = up ? lim_up : lim_dn;
  return wf.w * rec_fast<SCH>(fuu, fu, fd, lim ? wf.g : 0.0f, wf.A, wf.al, wf.E);
}

template <typename T>
__device__ __forceinline__ T sel(bool c, T a, T b) {
  return c ? a : b;
}

// ---- work items ------------------------------------------------------------------
struct StripItem {
  int dom, lev, sx, sy, grp;
};

// Blocks of 4 wavefronts, one work item per wavefront.  Consecutive blocks
// are dealt round-robin to the 8 XCDs, so block b is given the work of
// block (b%8)*per + b/8: each XCD takes a contiguous run of items.  Items of
// the w kernel are numbered tracer group fastest, then level, then strip, so
// the groups of one strip-level (which read the same layer heights,
// transports and masks) and then the neighbouring levels (which read the same
// tracer levels in the w sub-step) run side by side and meet in that XCD's
// L2.
template <int P, typename TF>
__device__ __forceinline__ bool strip_item(const FusedArgs<TF>& A, StripItem& it) {
  const long nblk = (A.nitems[P] + 3) / 4;
  const long per = (nblk + 7) / 8;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const long item = ((long)(blockIdx.x % 8) * per + blockIdx.x / 8) * 4 + wave;
  if (item >= A.nitems[P]) return false;
  int di = 0;
  while (di + 1 < A.ndom && A.doms[di + 1].item_begin[P] <= item) di++;
  const FusedDomain<TF>& a = A.doms[di];
  long loc = item - a.item_begin[P];
  it.dom = di;
  it.grp = (int)(loc % A.ngroups);
  loc /= A.ngroups;
  if constexpr (P == 0) {
    // u/v kernel: no coupling across levels; the strips of one column of
    // strips run side by side instead, so the four ghost rows a strip reads
    // below and above are the rows its neighbours read at the same time
    it.sy = (int)(loc % a.nsy[0]);
    loc /= a.nsy[0];
    it.sx = (int)(loc % a.nsx);
    it.lev = 1 + (int)(loc / a.nsx);
  } else {
    it.lev = 1 + (int)(loc % a.d.kmax);
    loc /= a.d.kmax;
    it.sx = (int)(loc % a.nsx);
    it.sy = (int)(loc / a.nsx);
  }
  return true;
}

template <int R>
using Slot = std::integral_constant<int, R>;

// Per-lane column data, kept in vector registers: xc = x (0 outside the
// array, so an address is always valid), xin = 0xff inside the array (else
// 0, masks the flags), xm = the MB_* bits the column's i-bounds allow
// (adv_split_u.F90 isub bounds; the w column stops at NX-2) plus MB_XOUT on
// the 60 columns a strip writes.
struct ColumnBits {
  int xc, xin, xm;
};
__device__ __forceinline__ ColumnBits column_bits(int x, int lane, int NX, int isub) {
  const bool in = x >= 0 && x < NX;
  int xm = MB_VFLUX | MB_VUPD;
  // (the u faces and updates of the outermost lanes reach no written column,
  // and what they would read beyond the wavefront is zero)
  const bool inner = lane >= 1 && lane <= 62;
  if (inner && x >= isub && x <= NX - 2 - isub) xm |= MB_UFLUX;
  if (inner && x >= 1 + isub && x <= NX - 2 - isub) xm |= MB_UUPD;
  if (x <= NX - 2) xm |= MB_WCOL;
  if (lane >= 2 && lane < 2 + kStripOut) xm |= MB_XOUT;
  return {in ? x : 0, in ? 0xff : 0, in ? xm : 0};
}

// load / store at a wave-uniform base plus a 32-bit byte offset: the base
// stays in scalar registers and the address costs one vector register (the
// saddr form of global_load/store).  A field of one tracer must stay below
// 4 GiB, which the launch plan checks.
template <typename T>
__device__ __forceinline__ T ldo(const T* base, uint32_t off) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}
template <typename T>
__device__ __forceinline__ void sto(T* base, uint32_t off, T v) {
  *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off) = v;
}

// The row march is unrolled four times: the four-row windows rotate by
// renaming (logical row q of step s lives in slot (s+q)&3).  Loads read
// valid addresses everywhere (cell 0 outside the array, the group's last
// tracer past its end, level K for a missing level); only the flags are
// masked, since every other value of a cell outside the array, or of a
// missing level, reaches discarded results only.

// FP64 loads a row's inputs while the row before it is computed, each tracer
// into the registers its sub-step has just read and the shared fields once
// the row's faces are set up, so the lookahead costs no second buffer (400 x
// 400 x 40 x 2 tracers: 376 us against 387 with two row buffers in the u/v
// kernel and the shared fields loaded where a row starts).  FP32 loads where
// the row starts: its kernels issue VALU instructions in three of four cycles
// and the longer live ranges only cost them a wavefront or spills (18 tracers
// on eight subdomains: 2.55 ms, against 3.2 ms with the lookahead).  All of
// the row's loads are issued before anything else of it: left to the compiler,
// the largest variants fetch a tracer at a time and wait for each (9 tracers
// with budgets and diffusion, 700 x 600 x 30: 1492 us, 1185 with the barrier).
// One tracer is better left alone (100 x 100 x 20: 20.4 us, 22.3 with it).
template <typename TF>
constexpr bool kRowAhead = sizeof(TF) == 8;

// The momentum variants (MOM; FP64, one tracer): the tracer is the velocity
// of the U (MOM = 1) or V (2) control volumes and the transports, w and layer
// heights are averaged onto those volumes (uv_advect_3d.F90:70-92, 238-256)
// where a row is read, instead of in a kernel of their own that writes six
// work fields and has them read back (400 x 400 x 40, both parts: 606 us, 920
// with the averaging kernels).
// The caller's arrays come as uu, vv, ww, ho, hn, hu = hun and hv = hvn.  The
// averages go to the next column (a lane move; the last column is zero) or
// the next row (loaded; the last row of the V part starts from the U part's
// result there, as the routine's work array does: mrow).  Only advres is
// wanted: the second kernel leaves out the result and its last division but
// on that row.
enum { MOM_NONE = 0, MOM_U = 1, MOM_V = 2 };

// The state variants (ST) also store the tracers after each sub-step, which
// the reverse mode reads: f1 after u/2 beside f2, f3 after w and f4 after v/2
// beside the result (fout may be NULL).  They are the states the sub-step
// kernels leave, in two launches that form the layer heights on the way
// instead of five that read them (256 x 256 x 30, one FP64 tracer: 83 us
// against 117; 320 x 256 x 30 x 18 FP32: 695 against 773).

// Five rows spread over a strip's nsteps are looked at before the march, so
// that a strip in a tail (which runs over several rows) takes the full
// divisions at once and not after a part of the short march: 400 x 400 x 40,
// two tracers, 40 patches in an empty basin after 60 steps 441 us against 481
// (449 with full divisions alone); nothing tiny, 383 against 380.  Three rows
// find fewer (478).  4-row strips lose little and are bound by latency: not
// there.  load(s, g, fl): the high word of tracer g in the row of step s, fl
// the cell's masks.
template <int G, typename Div, typename Load>
__device__ __forceinline__ void look_ahead(Div& dv, int nsteps, Load load) {
  constexpr int N = 5;
  const int stride = nsteps / N;
  uint32_t f[N][G];
  int fl[N];
#pragma unroll
  for (int q = 0; q < N; q++)
#pragma unroll
    for (int g = 0; g < G; g++) f[q][g] = load(stride / 2 + q * stride, g, fl[q]);
#pragma unroll
  for (int q = 0; q < N; q++)
#pragma unroll
    for (int g = 0; g < G; g++) dv.look(f[q][g], (fl[q] & MB_WCOL) != 0);
  dv.pin();
}

// ---- kernel 1: u/2 then v/2 at level L ------------------------------------------------
// Div: the divisions of the exact flavour; dv tells whether one left their
// range
template <typename TF, int SCH, int G, bool EXACT, bool ADV, bool DIFF, int MOM, bool ST,
          typename Div>
__device__ __forceinline__ void strip_uv(const FusedArgs<TF>& A, Div& dv) {
  StripItem it;
  if (!strip_item<0>(A, it)) return;
  const FusedDomain<TF>& a = A.doms[it.dom];
  const int lane = threadIdx.x & 63;
  const int NX = a.d.NX, NY = a.d.NY;
  const long NXY = a.d.NXY;
  const int x = it.sx * kStripOut - 2 + lane;
  const int y0 = it.sy * A.rows[0];
  const int t0 = it.grp * G;
  const int ntr = min(G, A.ntracers - t0);
  constexpr int isub = SCH == UPSTREAM ? 0 : 1;
  const ColumnBits cb = column_bits(x, lane, NX, isub);
  const bool xout = (cb.xm & MB_XOUT) != 0;
  const double dt = A.dt, dx = a.dx, dy = a.dy, ard1 = a.ard1, AH = A.AH;
  const double fracu = EXACT ? A.fracu : 0.5, fracv = EXACT ? A.fracv : 0.5;
  const double dtu = fracu * dt, dtv = fracv * dt;
  const double dtcu = dt * (0.5 * dy * ard1), dtcv = dt * (0.5 * dx * ard1);
  const FaceK ku = face_k(dtu, dx, AH), kv = face_k(dtv, dy, AH);
  const long oL = NXY * (long)it.lev;
  const long ts = a.tstride;
  const TF* fin_g[G];
  TF* f2_g[G];
#pragma unroll
  for (int g = 0; g < G; g++) {
    const long tg = (long)(t0 + min(g, ntr - 1)) * ts + oL;
    fin_g[g] = a.fin + tg;
    f2_g[g] = a.f2 + tg;
  }
  const double *ho = a.ho + oL, *uu = a.uu + oL, *hu = a.hu + oL, *vv = a.vv + oL,
               *hv = a.hv + oL;
  double* d2 = a.d2 + oL;
  double* a2 = ADV ? a.a2 + oL : nullptr;
  const uint8_t* flags = a.flags;
  const int nsteps = A.rows[0] + 4;
  auto cell = [&](int y) -> uint32_t {
    return (y >= 0 && y < NY) ? (uint32_t)(cb.xc + NX * y) : (uint32_t)cb.xc;
  };

  // inputs of the step of row y: the u/2 row y and the v face of row y-2 (the
  // momentum variants: the fields they are averaged from)
  struct Row {
    int fl;
    double ho, uu, hu, vv, hv;
    double hn, uun, hun, vvc, vvn;  // MOM
    TF f[G];
  };
  [[maybe_unused]] const double* hn = MOM ? a.hn + oL : nullptr;
  auto load_shared = [&](int y, Row& r) {
    const uint32_t c = cell(y), c2 = cell(y - 2);
    const uint32_t b8 = c * 8u, b82 = c2 * 8u;
    r.fl = flags[c];
    r.uu = ldo(uu, b8);
    r.hu = ldo(hu, b8);
    r.vv = ldo(vv, b82);
    if constexpr (MOM == MOM_V) {
      const uint32_t n = cell(y + 1) * 8u, n2 = cell(y - 1) * 8u;
      r.hv = ldo(hv, b8);
      r.uun = ldo(uu, n);
      r.hun = ldo(hu, n);
      const bool last = y == NY - 1;
      r.vvc = ldo(last ? a.mrow + (long)NX * it.lev : vv, last ? (uint32_t)cb.xc * 8u : b8);
      r.vvn = ldo(vv, n2);
      r.ho = ldo(ho, n2);
      r.hn = ldo(hn, n2);
    } else {
      r.ho = ldo(ho, b8);
      r.hv = ldo(hv, b82);
      if constexpr (MOM == MOM_U) r.hn = ldo(hn, b8);
    }
  };
  auto load_f = [&](int y, Row& r, int g) {
    if constexpr (!MOM) r.f[g] = ldo(fin_g[g], cell(y) * (uint32_t)sizeof(TF));
  };
  // the row's transports and heights, and (momentum) its velocity
  struct Fields {
    double ho, uu, hu, vv, hv;
  };
  auto fields = [&](int y, Row& r) -> Fields {
    if constexpr (MOM == MOM_U) {
      r.f[0] = x <= NX - 2 ? r.uu / r.hu : 0.0;
      return {r.hu, 0.5 * (r.uu + from_upper_lane(r.uu)), from_upper_lane(0.5 * (r.ho + r.hn)),
              0.5 * (r.vv + from_upper_lane(r.vv)), 0.5 * (r.hv + from_upper_lane(r.hv))};
    } else if constexpr (MOM == MOM_V) {
      const double q = r.vvc / r.hv;
      r.f[0] = y == NY - 1 ? r.vvc : q;
      return {r.hv, 0.5 * (r.uu + r.uun), 0.5 * (r.hu + r.hun), 0.5 * (r.vv + r.vvn),
              0.5 * (r.ho + r.hn)};
    } else {
      return {r.ho, r.uu, r.hu, r.vv, r.hv};
    }
  };
  auto load_row = [&](int y, Row& r) {
    load_shared(y, r);
#pragma unroll
    for (int g = 0; g < G; g++) load_f(y, r, g);
  };

  int flw[4] = {0, 0, 0, 0};
  double d1w[4] = {1, 1, 1, 1};
  double a1w[ADV ? 4 : 1][G];
  TF f1w[G][4];
  TF fvp[G];  // v flux through the face below the row being updated
  double vvp = 0.0;  // the v transport there
#pragma unroll
  for (int g = 0; g < G; g++) {
    fvp[g] = TF(0);
#pragma unroll
    for (int q = 0; q < 4; q++) f1w[g][q] = TF(0);
  }
  if constexpr (ADV) {
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int g = 0; g < G; g++) a1w[q][g] = 0.0;
  }

  // one row of the march; VF / VR: whether the v face and the v row of the
  // step exist (they start with the fourth and fifth row).  Known at compile
  // time, and every store waits for the end of the row, so the row is one
  // basic block in which the tracers' chains interleave
  auto step = [&](auto slot, auto vfc, auto vrc, Row& buf, int s) {
    constexpr int R = decltype(slot)::value;
    constexpr bool VF = decltype(vfc)::value, VR = decltype(vrc)::value;
    constexpr int w0 = R & 3, w1 = (R + 1) & 3, w2 = (R + 2) & 3, w3 = (R + 3) & 3;
    const int y = y0 - 2 + s;
    if constexpr (!kRowAhead<TF>) {
      load_row(y, buf);
      if constexpr (G > 1) __builtin_amdgcn_sched_barrier(0);
    }
    const int fl = (y >= 0 && y < NY) ? (buf.fl & cb.xin) : 0;  // raw masks of the cell
    const int fo = (fl | MB_XOUT) & cb.xm;                      // ... with the column bounds

    const Fields in = fields(y, buf);
    // ---- u/2 on row y: shared part
    const int flm = from_lower_lane(fl), flp = from_upper_lane(fl);
    FaceC<EXACT> fu;
    face_setup<SCH>(fu, fo & MB_UFLUX, flm & MB_UFLUX, flp & MB_UFLUX, in.uu, in.hu, ku,
                    dv);
    const double uum = from_lower_lane(in.uu);
    const bool updu = fo & MB_UUPD;
    const double D0 = in.ho;
    double D1 = D0;
    D1 = sel(updu, D0 - dtu * (in.uu * dy - uum * dy) * ard1, D0);
    CellK k1{};
    Den e1{}, e2{};  // D1, D2 as denominators (EXACT)
    if constexpr (EXACT) e1 = dv.den(D1);
    else k1 = cell_factors(D0, D1, dtcu);
    flw[w3] = fo;
    d1w[w3] = D1;

    // ---- v/2 on row yv = y-2: shared part (faces from row y0-1 on)
    const int yv = y - 2;
    FaceC<EXACT> fv;
    bool updv = false;
    double D2 = d1w[w1];
    CellK k2{};
    if constexpr (VF) {
      const bool yface = yv >= isub && yv <= NY - 2 - isub;
      face_setup<SCH>(fv, yface & ((flw[w1] & MB_VFLUX) != 0), flw[w0] & MB_VFLUX,
                      flw[w2] & MB_VFLUX, in.vv, in.hv, kv, dv);
      updv = (yface && yv >= 1 + isub) & ((flw[w1] & MB_VUPD) != 0);
      D2 = sel(updv, d1w[w1] - dtv * (in.vv * dx - vvp * dx) * ard1, D2);
      if constexpr (EXACT) e2 = dv.den(D2);
      else k2 = cell_factors(d1w[w1], D2, dtcv);
    }
    const bool st_ok = (VR && yv >= y0 && yv < NY) & ((flw[w1] & MB_XOUT) != 0);
    const uint32_t cv = (uint32_t)(x + NX * yv);
    TF res[G];
    double a2v = 0.0;
    vvp = in.vv;
    if constexpr (kRowAhead<TF>) load_shared(y + 1, buf);

    // u/2 on row y (adv_split_u.F90:219-286)
    auto sub_u = [&](int g) {
      const TF fc = buf.f[g];
      const TF fm1 = from_lower_lane(fc), fp1 = from_upper_lane(fc);
      const TF fp2 = from_upper_lane(fp1);
      const TF Fu = face_flux<TF, SCH, DIFF>(fu, fm1, fc, fp1, fp2, AH, ku, dv);
      const TF Fum = from_lower_lane(Fu);
      double advu = 0.0;
      TF F1 = fc;
      if constexpr (EXACT) {
        F1 = cell_update_exact(updu, D0, e1, fc, Fu, Fum, fracu, dy, ard1, dt, &advu, dv);
      } else {
        F1 = cell_update_fast(updu, k1, fc, Fu, Fum);
      }
      f1w[g][w3] = F1;
      if constexpr (ADV) a1w[w3][g] = 0.0 + advu;
      if constexpr (kRowAhead<TF>) load_f(y + 1, buf, g);
    };
    // v/2 on row yv (adv_split_v.F90:77-131)
    auto sub_v = [&](int g) {
      if constexpr (VF) {
        const TF Fv = face_flux<TF, SCH, DIFF>(fv, f1w[g][w0], f1w[g][w1], f1w[g][w2], f1w[g][w3],
                                               AH, kv, dv);
        if constexpr (VR) {
          double advv = 0.0;
          TF F2 = f1w[g][w1];
          if constexpr (EXACT) {
            F2 = cell_update_exact(updv, d1w[w1], e2, F2, Fv, fvp[g], fracv, dx, ard1, dt, &advv,
                                   dv);
          } else {
            F2 = cell_update_fast(updv, k2, F2, Fv, fvp[g]);
          }
          res[g] = F2;
          if constexpr (ADV) {
            if (g == 0) a2v = a1w[w1][0] + advv;
          }
        }
        fvp[g] = Fv;
      }
    };
    // FP64 a sub-step at a time, so that its tracers' division chains
    // interleave; FP32 a tracer at a time, for fewer live registers
    if constexpr (EXACT) {
#pragma unroll
      for (int g = 0; g < G; g++) sub_u(g);
      dv.pin();
#pragma unroll
      for (int g = 0; g < G; g++) sub_v(g);
      dv.pin();
    } else {
#pragma unroll
      for (int g = 0; g < G; g++) {
        sub_u(g);
        sub_v(g);
      }
    }
    // (past the group's last tracer the pointers and values repeat it)
    if (VR && st_ok) {
#pragma unroll
      for (int g = 0; g < G; g++) sto(f2_g[g], cv * (uint32_t)sizeof(TF), res[g]);
      if constexpr (ST) {
#pragma unroll
        for (int g = 0; g < G; g++)
          sto(f2_g[g] + a.f1_off, cv * (uint32_t)sizeof(TF), f1w[g][w1]);
      }
      if constexpr (ADV) sto(a2, cv * 8u, a2v);
      if (it.grp == 0) sto(d2, cv * 8u, D2);
    }
  };

  constexpr std::true_type on{};
  constexpr std::false_type off{};
  Row r;
  if constexpr (kRowAhead<TF>) load_row(y0 - 2, r);
  if constexpr (Div::kTests && !MOM) {
    if (nsteps > 8) {
      look_ahead<G>(dv, nsteps, [&](int s, int g, int& fl) {
        const uint32_t c = cell(y0 - 2 + s);
        fl = flags[c] & cb.xin;
        return ldo((const uint32_t*)fin_g[g], c * 8u + 4u);
      });
      if (dv.stop()) return;
    }
  }
  if constexpr (EXACT || G == 1) {
    step(Slot<0>{}, off, off, r, 0);
    if (dv.stop()) return;
    step(Slot<1>{}, off, off, r, 1);
    step(Slot<2>{}, off, off, r, 2);
  } else {
    // one body for the three rows, the windows moved instead of renamed: less
    // code (9 tracers: 55 -> 50 KB; 700 x 600 x 30: 1250 -> 1167 us)
#pragma unroll 1
    for (int s = 0; s < 3; s++) {
      flw[3] = flw[0]; flw[0] = flw[1];
      d1w[3] = d1w[0]; d1w[0] = d1w[1];
#pragma unroll
      for (int g = 0; g < G; g++) {
        f1w[g][3] = f1w[g][0];
        f1w[g][0] = f1w[g][1];
      }
      step(Slot<2>{}, off, off, r, s);
    }
  }
  step(Slot<3>{}, on, off, r, 3);
  if (dv.stop()) return;
  for (int s = 4; s < nsteps; s += 4) {
    step(Slot<0>{}, on, on, r, s);
    step(Slot<1>{}, on, on, r, s + 1);
    step(Slot<2>{}, on, on, r, s + 2);
    step(Slot<3>{}, on, on, r, s + 3);
    if (dv.stop()) return;
  }

  // level 0 of the work fields (the second kernel reads levels K-2..K+2 of
  // f2 and K-1..K+1 of d2 from one base): the input tracers and ho
  if (A.lev0 && it.lev == 1 && xout) {
    for (int yv = y0; yv < y0 + A.rows[0] && yv < NY; yv++) {
      const uint32_t c = (uint32_t)(x + NX * yv);
      for (int g = 0; g < ntr; g++) {
        const long tg = (long)(t0 + g) * ts;
        a.f2[tg + c] = a.fin[tg + c];
      }
      if (it.grp == 0) a.d2[c] = a.ho[c];
    }
  }
}

// ---- kernel 2: w, then v/2 and u/2 at level K -------------------------------------------
// BUD: some domain of the launch forms its budgets in the step (the
// variant without them carries none of their code or registers)
template <typename TF, int SCH, int G, bool EXACT, bool ADV, bool DIFF, bool BUD, int MOM, bool ST,
          typename Div>
__device__ __forceinline__ void strip_wvu(const FusedArgs<TF>& A, Div& dv) {
  StripItem it;
  if (!strip_item<1>(A, it)) return;
  const FusedDomain<TF>& a = A.doms[it.dom];
  const int lane = threadIdx.x & 63;
  const int NX = a.d.NX, NY = a.d.NY, kmax = a.d.kmax;
  const long NXY = a.d.NXY;
  const int K = it.lev;
  const int kshift = A.kshift;
  const int x = it.sx * kStripOut - 2 + lane;
  const int y0 = it.sy * A.rows[1];
  const int t0 = it.grp * G;
  const int ntr = min(G, A.ntracers - t0);
  constexpr int isub = SCH == UPSTREAM ? 0 : 1;
  const ColumnBits cb = column_bits(x, lane, NX, isub);
  const bool xout = (cb.xm & MB_XOUT) != 0;
  const double dt = A.dt, dth = 0.5 * A.dt, dx = a.dx, dy = a.dy, ard1 = a.ard1, AH = A.AH;
  const double dtcu = dt * (0.5 * dy * ard1), dtcv = dt * (0.5 * dx * ard1);
  const FaceK ku = face_k(dth, dx, AH), kv = face_k(dth, dy, AH);
  const long ts = a.tstride;
  const long oK = NXY * (long)K;
  // the w sub-step's levels: the flux at K+1/2 exists below kmax, the one at
  // K-1/2 above level 1 (or at level 1 with kshift); level K is updated up
  // to kmax-kshift (adv_split_w.F90:249-300)
  const bool wk_on = K <= kmax - 1, wp_on = K > 1 || kshift, kdo = K <= kmax - kshift;
  // where the limiter applies at the faces K-1/2 and K+1/2, going up / down
  const bool limp_up = SCH != UPSTREAM && K - 1 > 1 - kshift, limp_dn = SCH != UPSTREAM && K - 1 < kmax - 1;
  const bool limk_up = SCH != UPSTREAM && K > 1 - kshift, limk_dn = SCH != UPSTREAM && K < kmax - 1;
  // tracers after u/2 + v/2: one base per tracer (level 0), levels K-2..K+2
  // as byte offsets; layer heights K-1..K+1 (level 0 of both holds the input)
  const TF* f2_g[G];
  TF* fo_g[G];
#pragma unroll
  for (int g = 0; g < G; g++) {
    const long tg = (long)(t0 + min(g, ntr - 1)) * ts;
    f2_g[g] = a.f2 + tg;
    fo_g[g] = a.fout + tg + oK;
  }
  uint32_t lvo[5];
#pragma unroll
  for (int m = 0; m < 5; m++) {
    // (level 0 takes part with kshift only; a caller may leave it unset)
    const int l = K - 2 + m;
    lvo[m] = (uint32_t)(((l >= 1 - kshift && l <= kmax) ? l : K) * NXY * (long)sizeof(TF));
  }
  const bool has_kp1 = K < kmax;
  // d2 at K-1, K, K+1 and ww at K-1, K from one base each (level K-1) and
  // byte offsets
  const double *dKm1 = a.d2 + oK - NXY, *wwKm1 = a.ww + oK - NXY;
  const uint32_t lstep = (uint32_t)(NXY * 8), lup = has_kp1 ? 2u * lstep : lstep;
  const double *vv = a.vv + oK, *hv = a.hv + oK, *uu = a.uu + oK, *hu = a.hu + oK;
  const double* a2 = ADV ? a.a2 + oK : nullptr;
  double* hires = a.hires ? a.hires + oK : nullptr;
  const uint8_t* flags = a.flags;
  const int nsteps = A.rows[1] + 4;
  auto cell = [&](int y) -> uint32_t {
    return (y >= 0 && y < NY) ? (uint32_t)(cb.xc + NX * y) : (uint32_t)cb.xc;
  };

  // inputs of the step of row y: the w row y, and the v and u faces of row
  // y-2 (v also y-3)
  struct Row {
    int fl;
    double wwK, wwKm1, dKm1, dK, dKp1, vv, hv, uu, hu, a2;
    double wwKn, wwKm1n, ho, hn, uun, hun, vvn, hvn;  // MOM
    TF f[G][5];
  };
  [[maybe_unused]] const double *ho = MOM ? a.ho + oK : nullptr, *hn = MOM ? a.hn + oK : nullptr;
  [[maybe_unused]] const uint32_t east = x >= 0 && x + 1 < NX ? 8 : 0;
  auto load_shared = [&](int y, Row& r) {
    const uint32_t c = cell(y), c2 = cell(y - 2);
    const uint32_t b8 = c * 8u, b82 = c2 * 8u;
    r.fl = flags[c];
    r.wwK = ldo(wwKm1, b8 + lstep);
    r.wwKm1 = ldo(wwKm1, b8);
    r.dKm1 = ldo(dKm1, b8);
    r.dK = ldo(dKm1, b8 + lstep);
    r.dKp1 = ldo(dKm1, b8 + lup);
    r.vv = ldo(vv, b82);
    r.uu = ldo(uu, b82);
    r.hu = ldo(hu, b82);
    if constexpr (MOM == MOM_V) {
      const uint32_t n = cell(y + 1) * 8u, n2 = cell(y - 1) * 8u;
      r.wwKn = ldo(wwKm1, n + lstep);
      r.wwKm1n = ldo(wwKm1, n);
      r.vvn = ldo(vv, n2);
      r.uun = ldo(uu, n2);
      r.hun = ldo(hu, n2);
      r.ho = ldo(ho, n2);
      r.hn = ldo(hn, n2);
    } else {
      r.hv = ldo(hv, b82);
      if constexpr (MOM == MOM_U) {
        r.ho = ldo(ho, b82);
        r.hn = ldo(hn, b82);
        // w and v of lane 63 too: the u face of lane 61 reads its tracer
        r.wwKn = ldo(wwKm1, b8 + lstep + east);
        r.wwKm1n = ldo(wwKm1, b8 + east);
        r.vvn = ldo(vv, b82 + east);
        r.hvn = ldo(hv, b82 + east);
      }
    }
    if constexpr (ADV) r.a2 = ldo(a2, b8);
  };
  // the row's w, transports and heights (momentum: averaged as in the first
  // kernel; w at level 0 is zero)
  struct Fields {
    double wwK, wwKm1, vv, hv, uu, hu;
  };
  auto fields = [&](const Row& r) -> Fields {
    if constexpr (MOM == MOM_U) {
      return {0.5 * (r.wwK + r.wwKn), K == 1 ? 0.0 : 0.5 * (r.wwKm1 + r.wwKm1n),
              0.5 * (r.vv + r.vvn),   0.5 * (r.hv + r.hvn),
              0.5 * (r.uu + from_upper_lane(r.uu)), from_upper_lane(0.5 * (r.ho + r.hn))};
    } else if constexpr (MOM == MOM_V) {
      return {0.5 * (r.wwK + r.wwKn), K == 1 ? 0.0 : 0.5 * (r.wwKm1 + r.wwKm1n),
              0.5 * (r.vv + r.vvn),   0.5 * (r.ho + r.hn),
              0.5 * (r.uu + r.uun),   0.5 * (r.hu + r.hun)};
    } else {
      return {r.wwK, r.wwKm1, r.vv, r.hv, r.uu, r.hu};
    }
  };
  auto load_f = [&](int y, Row& r, int g) {
    const uint32_t b = cell(y) * (uint32_t)sizeof(TF);
#pragma unroll
    for (int m = 0; m < 5; m++) r.f[g][m] = ldo(f2_g[g], b + lvo[m]);
  };
  auto load_row = [&](int y, Row& r) {
    load_shared(y, r);
#pragma unroll
    for (int g = 0; g < G; g++) load_f(y, r, g);
  };

  int flw[4] = {0, 0, 0, 0}, fow[4] = {0, 0, 0, 0};
  double d3w[4] = {1, 1, 1, 1};
  double a3w[ADV ? 4 : 1][G];
  TF f3w[G][4];
  // budget (when a.bpart is set): the lane's sums over the rows it writes of
  // hires*f per tracer and of hires, interior water cells only, kept in LDS
  // (one slot per lane, output and wavefront) so they cost no registers
  const bool bud = BUD && a.bpart != nullptr;
  __shared__ double bsh[4][G + 1][64];
  const int wv = threadIdx.x >> 6;
  if (bud) {
#pragma unroll
    for (int q = 0; q <= G; q++) bsh[wv][q][lane] = 0.0;
  }
  TF fvp[G];  // as in the first kernel
  double vvp = 0.0;
#pragma unroll
  for (int g = 0; g < G; g++) {
    fvp[g] = TF(0);
#pragma unroll
    for (int q = 0; q < 4; q++) f3w[g][q] = TF(0);
  }
  if constexpr (ADV) {
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int g = 0; g < G; g++) a3w[q][g] = 0.0;
  }

  // one row of the march (VF, VR and the stores as in the first kernel)
  auto step = [&](auto slot, auto vfc, auto vrc, Row& buf, int s) {
    constexpr int R = decltype(slot)::value;
    constexpr bool VF = decltype(vfc)::value, VR = decltype(vrc)::value;
    constexpr int w0 = R & 3, w1 = (R + 1) & 3, w2 = (R + 2) & 3, w3 = (R + 3) & 3;
    const int y = y0 - 2 + s;
    if constexpr (!kRowAhead<TF>) {
      load_row(y, buf);
      if constexpr (G > 1) __builtin_amdgcn_sched_barrier(0);
    }
    const int fl = (y >= 0 && y < NY) ? (buf.fl & cb.xin) : 0;  // raw masks of the cell
    const int fo = (fl | MB_XOUT) & cb.xm;                      // ... with the column bounds

    const Fields in = fields(buf);
    // ---- w on row y: shared part
    const bool wcol = (y <= NY - 2) & ((fo & MB_WCOL) != 0);
    const bool wupd = wcol & kdo;
    const double D2K = buf.dK;
    double D3 = D2K;
    D3 = sel(wupd, D2K - dt * (in.wwK - in.wwKm1), D2K);
    CellK k3{};
    Den e3{}, e4{}, e5{};  // D3, D4, D5 as denominators (EXACT)
    if constexpr (EXACT) e3 = dv.den(D3);
    else k3 = cell_factors(D2K, D3, dt);
    WFace<EXACT> wfk, wfp;
    const bool onk = wcol & wk_on, onp = wcol & wp_on;
    wface_setup<SCH>(wfk, onk ? in.wwK : 0.0, dt, D2K, buf.dKp1, onk, dv);
    wface_setup<SCH>(wfp, onp ? in.wwKm1 : 0.0, dt, buf.dKm1, D2K, onp, dv);
    flw[w3] = fl;
    fow[w3] = fo;
    d3w[w3] = D3;

    // ---- v/2 and u/2 on row yv = y-2: shared part
    const int yv = y - 2;
    FaceC<EXACT> fv, fu;
    bool updv = false, updu = false;
    double D4 = d3w[w1], D5 = d3w[w1];
    CellK k4{}, k5{};
    if constexpr (VF) {
      const bool yface = yv >= isub && yv <= NY - 2 - isub;
      face_setup<SCH>(fv, yface & ((flw[w1] & MB_VFLUX) != 0), flw[w0] & MB_VFLUX,
                      flw[w2] & MB_VFLUX, in.vv, in.hv, kv, dv);
      updv = (yface && yv >= 1 + isub) & ((flw[w1] & MB_VUPD) != 0);
      D4 = sel(updv, d3w[w1] - dth * (in.vv * dx - vvp * dx) * ard1, D4);
      if constexpr (EXACT) e4 = dv.den(D4);
      else k4 = cell_factors(d3w[w1], D4, dtcv);
    }
    if constexpr (VR) {
      const int flv = flw[w1], fov = fow[w1];
      const int flm = from_lower_lane(flv), flp = from_upper_lane(flv);
      face_setup<SCH>(fu, fov & MB_UFLUX, flm & MB_UFLUX, flp & MB_UFLUX, in.uu, in.hu, ku,
                    dv);
      const double uum = from_lower_lane(in.uu);
      updu = fov & MB_UUPD;
      D5 = sel(updu, D4 - dth * (in.uu * dy - uum * dy) * ard1, D4);
      if constexpr (EXACT) e5 = dv.den(D5);
      else k5 = cell_factors(D4, D5, dtcu);
    }
    const bool st_ok = (VR && yv >= y0 && yv < NY) & ((fow[w1] & MB_XOUT) != 0);
    const uint32_t cv = (uint32_t)(x + NX * yv);
    TF res[G], f4[G];
    double a5v = 0.0, a4[ADV ? G : 1];
    [[maybe_unused]] double fum, fuf;  // MOM: the u fluxes of the row
    [[maybe_unused]] const double A2 = ADV ? buf.a2 : 0.0;
    vvp = in.vv;
    if constexpr (kRowAhead<TF>) load_shared(y + 1, buf);

    // w on row y (adv_split_w.F90:249-300); what the operands of a face that
    // does not exist read in place of a missing level reaches no limiter, and
    // its flux is selected to zero: w = 0 times an infinite tracer is NaN (the
    // short march gives the strip up over that instead)
    auto sub_w = [&](int g) {
      const TF fKm2 = buf.f[g][0], fKm1 = buf.f[g][1], fK = buf.f[g][2];
      const TF fKp1 = buf.f[g][3], fKp2 = buf.f[g][4];
      TF F3 = fK;
      double advw = 0.0;
      if constexpr (EXACT) {
        TF wprev =
            wflux_exact<SCH>(wfp, limp_up & onp, limp_dn & onp, fKm2, fKm1, fK, fKp1, dv);
        TF wk = wflux_exact<SCH>(wfk, limk_up & onk, limk_dn & onk, fKm1, fK, fKp1, fKp2, dv);
        if constexpr (!Div::kTests) {
          wprev = onp ? wprev : TF(0);
          wk = onk ? wk : TF(0);
        }
        const double aw = 1.0 * (wk - wprev);
        const double f3 = dv.over(D2K * fK - dt * aw, e3, wupd);
        advw = wupd ? aw : 0.0;
        F3 = wupd ? f3 : fK;
      } else {
        const TF p = wflux_fast<SCH>(wfp, limp_up, limp_dn, fKm2, fKm1, fK, fKp1);
        const TF q = wflux_fast<SCH>(wfk, limk_up, limk_dn, fKm1, fK, fKp1, fKp2);
        const TF wprev = wp_on ? p : TF(0), wk = wk_on ? q : TF(0);
        F3 = cell_update_fast(wupd, k3, fK, wk, wprev);
      }
      f3w[g][w3] = F3;
      if constexpr (ADV) a3w[w3][g] = A2 + advw;
      if constexpr (kRowAhead<TF>) load_f(y + 1, buf, g);
    };
    // v/2 on row yv (adv_split_v.F90:77-131)
    auto sub_v = [&](int g) {
      if constexpr (VF) {
        const TF Fv = face_flux<TF, SCH, DIFF>(fv, f3w[g][w0], f3w[g][w1], f3w[g][w2], f3w[g][w3],
                                               AH, kv, dv);
        if constexpr (VR) {
          double advv = 0.0;
          TF F4 = f3w[g][w1];
          if constexpr (EXACT) {
            F4 = cell_update_exact(updv, d3w[w1], e4, F4, Fv, fvp[g], 0.5, dx, ard1, dt, &advv, dv);
          } else {
            F4 = cell_update_fast(updv, k4, F4, Fv, fvp[g]);
          }
          f4[g] = F4;
          if constexpr (ADV) a4[g] = a3w[w1][g] + advv;
        }
        fvp[g] = Fv;
      }
    };
    // u/2 on row yv (adv_split_u.F90:219-286)
    auto sub_u = [&](int g) {
      if constexpr (VR) {
        const TF F4 = f4[g];
        double advu = 0.0;
        const TF fm1 = from_lower_lane(F4), fp1 = from_upper_lane(F4);
        const TF fp2 = from_upper_lane(fp1);
        const TF Fu = face_flux<TF, SCH, DIFF>(fu, fm1, F4, fp1, fp2, AH, ku, dv);
        const TF Fum = from_lower_lane(Fu);
        TF F5 = F4;
        if constexpr (MOM) {
          fum = Fum; fuf = Fu;
          advu = updu ? 0.5 * (Fu * dy - Fum * dy) * ard1 : 0.0;
        } else if constexpr (EXACT) {
          F5 = cell_update_exact(updu, D4, e5, F4, Fu, Fum, 0.5, dy, ard1, dt, &advu, dv);
        } else {
          F5 = cell_update_fast(updu, k5, F4, Fu, Fum);
        }
        res[g] = F5;
        if constexpr (ADV) {
          if (g == 0) a5v = a4[0] + advu;
        }
      }
    };
    // (the order as in the first kernel)
    if constexpr (EXACT) {
#pragma unroll
      for (int g = 0; g < G; g++) sub_w(g);
      dv.pin();
#pragma unroll
      for (int g = 0; g < G; g++) sub_v(g);
      dv.pin();
#pragma unroll
      for (int g = 0; g < G; g++) sub_u(g);
      dv.pin();
    } else {
#pragma unroll
      for (int g = 0; g < G; g++) {
        sub_w(g);
        sub_v(g);
        sub_u(g);
      }
    }
    // (past the group's last tracer the pointers and values repeat it)
    if (VR && st_ok) {
      if constexpr (ST) {
#pragma unroll
        for (int g = 0; g < G; g++) {
          sto(const_cast<TF*>(f2_g[g]) + (a.f3_off + oK), cv * (uint32_t)sizeof(TF), f3w[g][w1]);
          sto(const_cast<TF*>(f2_g[g]) + (a.f4_off + oK), cv * (uint32_t)sizeof(TF), f4[g]);
        }
        if (a.fout) {
#pragma unroll
          for (int g = 0; g < G; g++) sto(fo_g[g], cv * (uint32_t)sizeof(TF), res[g]);
        }
      } else if constexpr (!MOM) {
#pragma unroll
        for (int g = 0; g < G; g++) sto(fo_g[g], cv * (uint32_t)sizeof(TF), res[g]);
      }
      if constexpr (MOM == MOM_U) {
        if (yv == NY - 1) {  // the advected velocity the V part starts from there
          double advn;
          DivFull df;
          a.mrow[x + (long)NX * K] = cell_update_exact(updu, D4, df.den(D5), f4[0], fuf, fum, 0.5,
                                                       dy, ard1, dt, &advn, df);
        }
      }
      if constexpr (ADV) {
        if (a.advres) a.advres[oK + cv] = a5v;
      }
      if (it.grp == 0 && hires) sto(hires, cv * 8u, D5);
      // interior water cell of the mass and volume budgets
      if (BUD && bud && (flw[w1] & MB_WCOL) && x >= 2 && x <= NX - 3 && yv >= 2 &&
          yv <= NY - 3) {
#pragma unroll
        for (int g = 0; g < G; g++)
          bsh[wv][g][lane] = __builtin_fma(D5, (double)res[g], bsh[wv][g][lane]);
        if (it.grp == 0) bsh[wv][G][lane] += D5;
      }
    }
  };

  constexpr std::true_type on{};
  constexpr std::false_type off{};
  Row r;
  if constexpr (kRowAhead<TF>) load_row(y0 - 2, r);
  if constexpr (Div::kTests && !MOM) {
    if (nsteps > 8) {
      look_ahead<G>(dv, nsteps, [&](int s, int g, int& fl) {
        const uint32_t c = cell(y0 - 2 + s);
        fl = flags[c] & cb.xin;
        return ldo((const uint32_t*)f2_g[g], c * 8u + (lvo[2] + 4u));
      });
      if (dv.stop()) return;
    }
  }
  if constexpr (EXACT || G == 1) {
    step(Slot<0>{}, off, off, r, 0);
    if (dv.stop()) return;
    step(Slot<1>{}, off, off, r, 1);
    step(Slot<2>{}, off, off, r, 2);
  } else {
    // (as in the first kernel)
#pragma unroll 1
    for (int s = 0; s < 3; s++) {
      flw[3] = flw[0]; flw[0] = flw[1];
      fow[3] = fow[0]; fow[0] = fow[1];
      d3w[3] = d3w[0]; d3w[0] = d3w[1];
#pragma unroll
      for (int g = 0; g < G; g++) {
        f3w[g][3] = f3w[g][0];
        f3w[g][0] = f3w[g][1];
      }
      step(Slot<2>{}, off, off, r, s);
    }
  }
  step(Slot<3>{}, on, off, r, 3);
  if (dv.stop()) return;
  for (int s = 4; s < nsteps; s += 4) {
    step(Slot<0>{}, on, on, r, s);
    step(Slot<1>{}, on, on, r, s + 1);
    step(Slot<2>{}, on, on, r, s + 2);
    step(Slot<3>{}, on, on, r, s + 3);
    if (dv.stop()) return;
  }

  // the budget partials of this strip-level: the lanes' sums added over the
  // wavefront in a six-level FP64 tree (a partial is then within R + 6
  // roundings of exact for terms of one sign, R the strip's rows), written
  // by lane 0 as a (value, 0) pair; the final pass adds the pairs as
  // double-doubles
  if (bud) {
    const long nsl = (long)a.nsx * a.nsy[1] * kmax;
    const long sl = ((long)(K - 1) * a.nsy[1] + it.sy) * a.nsx + it.sx;
    auto wave_sum = [&](double v, int q) {
      double h = v;
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1) h += __shfl_xor(h, m);
      if (lane == 0) {
        a.bpart[2 * ((long)q * nsl + sl)] = h;
        a.bpart[2 * ((long)q * nsl + sl) + 1] = 0.0;
      }
    };
#pragma unroll
    for (int g = 0; g < G; g++)
      if (g < ntr) wave_sum(bsh[wv][g][lane], t0 + g);
    if (it.grp == 0) wave_sum(bsh[wv][G][lane], A.ntracers);
  }

  // level 0 passes through (the step updates levels 1..kmax)
  if (K == 1 && xout) {
    for (int yv = y0; yv < y0 + A.rows[1] && yv < NY; yv++) {
      const uint32_t c = (uint32_t)(x + NX * yv);
      for (int g = 0; !MOM && a.fout && g < ntr; g++) {
        const long tg = (long)(t0 + g) * ts;
        a.fout[tg + c] = a.fin[tg + c];
      }
      if (it.grp == 0 && a.hires) a.hires[c] = a.ho[c];
      if constexpr (ADV) {
        if (a.advres) a.advres[c] = 0.0;
      }
    }
  }
}

// ---- the kernels --------------------------------------------------------------------
// The exact flavour marches a strip with the short divisions and, where one of
// them left its range, again with the full ones: a call, so that the rarely
// taken march shares no registers with the other (inlined it took the FP64
// kernels from 126 and 189 to 250 VGPRs).  The call takes the kernel
// argument's address and makes it uniform again.
// Wavefronts per SIMD the kernels must leave room for: u/v FP64 4, the others
// 3.  Left to itself the compiler trades them for instruction-level
// parallelism, and 400 x 400 x 40 x 2 FP64 tracers take 419 us (3 and 2)
// against 400; more than these spill in the row loop (FP32 at 4: 2.6 -> 3.2
// ms on the 18-tracer batch).
template <typename TF>
constexpr int kWavesUv = sizeof(TF) == 8 ? 4 : 3;
constexpr int kWavesWvu = 3;
template <typename TF>
__device__ __forceinline__ const FusedArgs<TF>& uniform_args(uint64_t p) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)p);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
  using Arg = const __attribute__((address_space(4))) FusedArgs<TF>;
  return *(const FusedArgs<TF>*)(Arg*)(((uint64_t)hi << 32) | lo);
}
template <typename TF, int SCH, int G, bool ADV, bool DIFF, int MOM, bool ST>
__device__ __attribute__((noinline)) void strip_uv_full(uint64_t args) {
  DivFull dv;
  strip_uv<TF, SCH, G, true, ADV, DIFF, MOM, ST>(uniform_args<TF>(args), dv);
}
template <typename TF, int SCH, int G, bool ADV, bool DIFF, bool BUD, int MOM, bool ST>
__device__ __attribute__((noinline)) void strip_wvu_full(uint64_t args) {
  DivFull dv;
  strip_wvu<TF, SCH, G, true, ADV, DIFF, BUD, MOM, ST>(uniform_args<TF>(args), dv);
}

// upstream divides once per cell and sub-step and waits for memory: full
// divisions cost it nothing, while the tests of the short ones keep Courant
// numbers and heights that it does not read (400 x 400 x 40: one tracer 183 us,
// 202 with them; two 262, 282)
template <bool EXACT, int SCH>
constexpr bool kShort = EXACT && SCH != UPSTREAM;

template <typename TF, int SCH, int G, bool EXACT, bool ADV, bool DIFF, int MOM = MOM_NONE,
          bool ST = false>
__global__ __launch_bounds__(256, kWavesUv<TF>) void k_strip_uv(FusedArgs<TF> A) {
  std::conditional_t<kShort<EXACT, SCH>, DivNewton, DivFull> dv;
  strip_uv<TF, SCH, G, EXACT, ADV, DIFF, MOM, ST>(A, dv);
  if constexpr (kShort<EXACT, SCH>) {
    if (dv.bad)
      strip_uv_full<TF, SCH, G, ADV, DIFF, MOM, ST>(
          (uint64_t)__builtin_amdgcn_kernarg_segment_ptr());
  }
}

template <typename TF, int SCH, int G, bool EXACT, bool ADV, bool DIFF, bool BUD,
          int MOM = MOM_NONE, bool ST = false>
__global__ __launch_bounds__(256, kWavesWvu) void k_strip_wvu(FusedArgs<TF> A) {
  std::conditional_t<kShort<EXACT, SCH>, DivNewton, DivFull> dv;
  strip_wvu<TF, SCH, G, EXACT, ADV, DIFF, BUD, MOM, ST>(A, dv);
  if constexpr (kShort<EXACT, SCH>) {
    if (dv.bad)
      strip_wvu_full<TF, SCH, G, ADV, DIFF, BUD, MOM, ST>(
          (uint64_t)__builtin_amdgcn_kernarg_segment_ptr());
  }
}

template <typename TF>
void strip_plan(FusedArgs<TF>& a, int group) {
  a.ngroups = (a.ntracers + group - 1) / group;
  for (int p = 0; p < 2; p++) {
    long items = 0;
    for (int i = 0; i < a.ndom; i++) {
      FusedDomain<TF>& d = a.doms[i];
      d.nsx = (d.d.NX + kStripOut - 1) / kStripOut;
      d.nsy[p] = (d.d.NY + a.rows[p] - 1) / a.rows[p];
      d.item_begin[p] = items;
      items += (long)d.nsx * d.nsy[p] * d.d.kmax * a.ngroups;
    }
    a.nitems[p] = items;
  }
}

// the first kernel alone (its fractions in A; FP64): hscheme only
template <typename TF, int G, bool ADV>
hipError_t launch_uv(hipStream_t st, const FusedArgs<TF>& A) {
  const unsigned grid = (unsigned)((((A.nitems[0] + 3) / 4 + 7) / 8) * 8);
#define GT_UV(S)                                                                              \
  if (A.AH > 0.0)                                                                             \
    hipLaunchKernelGGL((k_strip_uv<TF, S, G, true, ADV, true>), dim3(grid), dim3(256), 0, st, A); \
  else                                                                                        \
    hipLaunchKernelGGL((k_strip_uv<TF, S, G, true, ADV, false>), dim3(grid), dim3(256), 0, st, A)
  switch (A.hscheme) {
    case P2_PDM: GT_UV(P2_PDM); break;
    case SUPERBEE: GT_UV(SUPERBEE); break;
    case MUSCL: GT_UV(MUSCL); break;
    case P2: GT_UV(P2); break;
    case UPSTREAM: GT_UV(UPSTREAM); break;
    default: return hipErrorInvalidValue;
  }
#undef GT_UV
  return hipGetLastError();
}

// both kernels of a state variant
template <typename TF, int SCH, int G, bool EXACT>
hipError_t launch_states_one(hipStream_t st, const FusedArgs<TF>& A) {
  auto grid = [&](int p) { return dim3((unsigned)((((A.nitems[p] + 3) / 4 + 7) / 8) * 8)); };
  auto go = [&](auto diff) -> hipError_t {
    constexpr bool D = decltype(diff)::value;
    hipLaunchKernelGGL((k_strip_uv<TF, SCH, G, EXACT, false, D, MOM_NONE, true>), grid(0),
                       dim3(256), 0, st, A);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((k_strip_wvu<TF, SCH, G, EXACT, false, D, false, MOM_NONE, true>), grid(1),
                       dim3(256), 0, st, A);
    return hipGetLastError();
  };
  return A.AH > 0.0 ? go(std::true_type{}) : go(std::false_type{});
}
template <typename TF, int G, bool EXACT>
hipError_t dispatch_states(hipStream_t st, const FusedArgs<TF>& a) {
  switch (a.hscheme) {
    case P2_PDM: return launch_states_one<TF, P2_PDM, G, EXACT>(st, a);
    case SUPERBEE: return launch_states_one<TF, SUPERBEE, G, EXACT>(st, a);
    case MUSCL: return launch_states_one<TF, MUSCL, G, EXACT>(st, a);
    case P2: return launch_states_one<TF, P2, G, EXACT>(st, a);
    case UPSTREAM: return launch_states_one<TF, UPSTREAM, G, EXACT>(st, a);
    default: return hipErrorInvalidValue;
  }
}

// both kernels of a momentum variant
template <int SCH, int MOM>
hipError_t launch_momentum_one(hipStream_t st, const FusedArgs<double>& A) {
  auto grid = [&](int p) { return dim3((unsigned)((((A.nitems[p] + 3) / 4 + 7) / 8) * 8)); };
  hipLaunchKernelGGL((k_strip_uv<double, SCH, 1, true, true, false, MOM>), grid(0), dim3(256), 0,
                     st, A);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_strip_wvu<double, SCH, 1, true, true, false, false, MOM>), grid(1),
                     dim3(256), 0, st, A);
  return hipGetLastError();
}

template <typename TF, int SCH, int G, bool EXACT, bool ADV, bool DIFF>
hipError_t launch_two(hipStream_t st, const FusedArgs<TF>& A) {
  auto grid = [&](int p) { return (unsigned)((((A.nitems[p] + 3) / 4 + 7) / 8) * 8); };
  hipLaunchKernelGGL((k_strip_uv<TF, SCH, G, EXACT, ADV, DIFF>), dim3(grid(0)), dim3(256), 0, st,
                     A);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  bool bud = false;
  for (int i = 0; i < A.ndom; i++) bud = bud || A.doms[i].bpart != nullptr;
  if (bud)
    hipLaunchKernelGGL((k_strip_wvu<TF, SCH, G, EXACT, ADV, DIFF, true>), dim3(grid(1)),
                       dim3(256), 0, st, A);
  else
    hipLaunchKernelGGL((k_strip_wvu<TF, SCH, G, EXACT, ADV, DIFF, false>), dim3(grid(1)),
                       dim3(256), 0, st, A);
  return hipGetLastError();
}

template <typename TF, int SCH, int G, bool EXACT, bool ADV>
hipError_t launch_one(hipStream_t st, const FusedArgs<TF>& A) {
  return A.AH > 0.0 ? launch_two<TF, SCH, G, EXACT, ADV, true>(st, A)
                    : launch_two<TF, SCH, G, EXACT, ADV, false>(st, A);
}

// one scheme at compile time (hscheme == vscheme)
template <typename TF, int G, bool EXACT, bool ADV>
hipError_t dispatch_scheme(hipStream_t st, const FusedArgs<TF>& a) {
  if (a.hscheme != a.vscheme) return hipErrorInvalidValue;
  switch (a.hscheme) {
    case P2_PDM: return launch_one<TF, P2_PDM, G, EXACT, ADV>(st, a);
    case SUPERBEE: return launch_one<TF, SUPERBEE, G, EXACT, ADV>(st, a);
    case MUSCL: return launch_one<TF, MUSCL, G, EXACT, ADV>(st, a);
    case P2: return launch_one<TF, P2, G, EXACT, ADV>(st, a);
    case UPSTREAM: return launch_one<TF, UPSTREAM, G, EXACT, ADV>(st, a);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace gt
