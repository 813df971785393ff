// gt_batched_f64.hip -- the launch plan of the HALFSPLIT strip kernels
// (gt_strip_impl.h) and the choice of their instantiation.
#include "gt_strip_impl.h"

namespace gt {

void strip_rows(int tile, int rows[2]) {
  static const int r[3] = {16, 32, 8};
  if (tile == 12) {
    rows[0] = rows[1] = 4;
  } else if (tile >= 3 && tile < 12) {
    rows[0] = r[(tile - 3) % 3];
    rows[1] = r[(tile - 3) / 3];
  } else {
    rows[0] = rows[1] = r[(tile >= 0 && tile < 3) ? tile : 0];
  }
}

bool fused_supported(int hscheme, int vscheme) {
  return hscheme == vscheme &&
         (hscheme == UPSTREAM || hscheme == P2 || hscheme == SUPERBEE || hscheme == MUSCL ||
          hscheme == P2_PDM);
}

template void strip_plan<double>(FusedArgs<double>&, int);
template void strip_plan<float>(FusedArgs<float>&, int);

// strip-levels of a launch at R rows per strip, times n
template <typename TF>
static long strip_levels(const FusedArgs<TF>& a, int R, int n) {
  long items = 0;
  for (int i = 0; i < a.ndom; i++) {
    const Dims& d = a.doms[i].d;
    items += (long)((d.NX + kStripOut - 1) / kStripOut) * ((d.NY + R - 1) / R) * d.kmax * n;
  }
  return items;
}

// The time of a launch of groups of g tracers and strips of R rows, in us: the
// march is R + 4 steps, and a step takes what one wavefront needs for it alone
// plus its share of all W wavefronts' work (times work, for the momentum
// variants: 130 x 120 x 40 81 us with 8 rows, 92 with 4).  Fitted to P2-PDM from 20 x 16 x 5
// to 700 x 600 x 30, 1 to 18 tracers, every g and R of 4, 8 and 16, to 10-15%;
// the choices made from it are 2% slower than the best pair measured in the
// mean, 15% at worst.
template <typename TF>
static double plan_cost(const FusedArgs<TF>& a, int g, int R, double work) {
  struct Fit {
    int g;
    double alone, share;  // us, us per 1000 wavefronts
  };
  static const Fit f32[] = {{1, 2.0, 0.50}, {3, 2.85, 0.77}, {6, 3.9, 1.13}, {9, 4.6, 1.62}};
  static const Fit f64[] = {{1, 2.1, 0.66}, {2, 2.7, 0.92}};
  const Fit* f = sizeof(TF) == 4 ? f32 : f64;
  while (f->g < g) f++;
  const long W = strip_levels(a, R, (a.ntracers + g - 1) / g);
  return (R + 4) * (f->alone + work * f->share * 1e-3 * (double)W);
}
template <typename TF>
static int plan_rows(const FusedArgs<TF>& a, int g, double work, double* cost) {
  int best = 16;
  *cost = plan_cost(a, g, 16, work);
  for (int R = 8; R >= 4; R /= 2) {
    const double c = plan_cost(a, g, R, work);
    if (c < *cost) {
      *cost = c;
      best = R;
    }
  }
  return best;
}

// Tracers per wavefront: the group whose best strips cost least (FP32: 18 on
// 100 x 100 x 20 62 us in groups of 3, 80 in groups of 9; 9 on 130 x 120 x 40
// 82 with 9 and 4 rows, 106 with 9 and 8; 18 on 700 x 600 x 30 2.03 ms with 9,
// 2.08 with 6).  FP64 takes two unless one is a tenth better (two tracers on
// 20 x 16 x 5: 20 us one at a time, 26 together; on 400 x 400 x 40 two
// together, 376).
template <typename TF>
int strip_auto_group(const FusedArgs<TF>& a) {
  if (a.ntracers == 1) return 1;
  double cost, best = 0.0;
  int g = 0;
  auto take = [&](int group, double bias) {
    (void)plan_rows(a, group, 1.0, &cost);
    if (g == 0 || cost * bias < best) {
      best = cost * bias;
      g = group;
    }
  };
  if constexpr (sizeof(TF) == 8) {
    take(2, 1.0);
    take(1, 1.1);
  } else {
    for (int group : {9, 6, 3, 1}) take(group, 1.0);
  }
  return g;
}

// Strip heights.  A strip's march is a chain of rows + 4 steps, so where
// 4-row strips fit the chip at once they are the fastest (100 x 100 x 20, one
// FP64 tracer: 31 us, 38 with 8 rows, 61 with 16); beyond a few wavefronts per
// SIMD the four ghost rows cost more than the shorter chain gives, and taller
// strips follow (256 x 256 x 30: 16/8 92 us, 8/8 97, 16/16 99, 32/32 141; 400
// x 400 x 40 x 2: 16/16 371, 8/8 373, 32/32 389).  FP32 strips stay at 8 rows
// longer (300 x 300 x 40 x 9: 8/8 366 us, 16/8 394; 700 x 600 x 30 x 6: 8/8
// 854, 16/16 865), and the largest grids take 32 (2000 x 1500 x 50 x 6: 9.9 ms
// against 10.0 with 16).
template <typename TF>
void strip_auto_rows(FusedArgs<TF>& a, int group, double work) {
  const int ng = (a.ntracers + group - 1) / group;
  const long i8 = strip_levels(a, 8, ng), s8 = strip_levels(a, 8, 1);
  double cost;
  const bool shortest = plan_rows(a, group, work, &cost) == 4;
  const long upto8[2] = {sizeof(TF) == 8 ? 4096 : 16384, sizeof(TF) == 8 ? 8192 : 16384};
  const bool tall[2] = {sizeof(TF) == 4 && i8 >= 65536, sizeof(TF) == 4 && s8 >= 200000};
  for (int p = 0; p < 2; p++)
    a.rows[p] = shortest ? 4 : (i8 <= upto8[p] ? 8 : (tall[p] ? 32 : 16));
}
template int strip_auto_group<double>(const FusedArgs<double>&);
template int strip_auto_group<float>(const FusedArgs<float>&);
template void strip_auto_rows<double>(FusedArgs<double>&, int, double);
template void strip_auto_rows<float>(FusedArgs<float>&, int, double);

hipError_t launch_fused_f64_g1(hipStream_t st, const FusedArgs<double>& a);
hipError_t launch_fused_f64_g2(hipStream_t st, const FusedArgs<double>& a);
hipError_t launch_fused_f64_adv(hipStream_t st, const FusedArgs<double>& a);
hipError_t launch_strip_uv_g1(hipStream_t st, const FusedArgs<double>& a);
hipError_t launch_strip_uv_adv(hipStream_t st, const FusedArgs<double>& a);

hipError_t launch_strip_uv_f64(hipStream_t st, const FusedArgs<double>& a, bool adv) {
  return adv ? launch_strip_uv_adv(st, a) : launch_strip_uv_g1(st, a);
}

hipError_t launch_fused_f64(hipStream_t st, const FusedArgs<double>& a, int group, bool adv) {
  if (adv) return launch_fused_f64_adv(st, a);
  return group == 2 ? launch_fused_f64_g2(st, a) : launch_fused_f64_g1(st, a);
}

}  // namespace gt

namespace gt {
hipError_t launch_fused_f32_g1(hipStream_t st, const FusedArgs<float>& a);
hipError_t launch_fused_f32_g3(hipStream_t st, const FusedArgs<float>& a);
hipError_t launch_fused_f32_g6(hipStream_t st, const FusedArgs<float>& a);
hipError_t launch_fused_f32_g9(hipStream_t st, const FusedArgs<float>& a);

hipError_t launch_fused_f32(hipStream_t st, const FusedArgs<float>& a, int group) {
  switch (group) {
    case 1: return launch_fused_f32_g1(st, a);
    case 6: return launch_fused_f32_g6(st, a);
    case 9: return launch_fused_f32_g9(st, a);
    default: return launch_fused_f32_g3(st, a);
  }
}
}  // namespace gt
