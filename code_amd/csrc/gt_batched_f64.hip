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

// The tracers per wavefront that cost least: a group's time is that of its
// shared work and its slots, filled or not (1, 3, 6, 9 FP32 tracers: 27, 50,
// 87, 128 in units of 10 us on the eight subdomains; 9 needs a grid that
// fills the chip many times over, at 256 x 192 x 30 it takes 328 us for 18
// tracers against 300 with 6).  Where even 4-row strips leave the chip short
// of wavefronts a smaller group makes more of them (64 x 64 x 30 x 18: 60 us
// with 6, 78 with 9; 6 tracers: 32 us with 3, 40 with 6).
template <typename TF>
int strip_auto_group(const FusedArgs<TF>& a) {
  if constexpr (sizeof(TF) == 8) return a.ntracers >= 2 ? 2 : 1;
  if (a.ntracers == 1) return 1;
  auto groups = [&](int g) { return (a.ntracers + g - 1) / g; };
  const int c3 = groups(3) * 50, c6 = groups(6) * 87;
  const int c9 = groups(9) * (strip_levels(a, 8, groups(9)) >= 32768 ? 128 : 138);
  int g = c9 <= c6 && c9 <= c3 ? 9 : (c6 <= c3 ? 6 : 3);
  while (g > 3 && strip_levels(a, 4, groups(g)) < 2560) g -= 3;
  return g;
}

// Strip heights.  A strip's march is a chain of rows + 4 steps, so where
// 4-row strips fit the chip at once they are the fastest (100 x 100 x 20, one
// FP64 tracer: 31 us, 38 with 8 rows, 61 with 16); beyond one round of
// wavefronts the four ghost rows cost more than the shorter chain gives, and
// taller strips follow (256 x 256 x 30: 16/8 92 us, 8/8 97, 16/16 99, 32/32
// 141; 400 x 400 x 40 x 2: 16/16 371, 8/8 373, 32/32 389).  FP32 strips stay
// at 8 rows longer (256 x 192 x 30 x 6: 8/8 105 us, 16/16 137; 512 x 384 x 30
// x 6: 16/8 434, 16/16 455), and the largest grids take 32 (2000 x 1500 x 50
// x 6: 9.9 ms against 10.3 with 16).
template <typename TF>
void strip_auto_rows(FusedArgs<TF>& a, int group) {
  const int ng = (a.ntracers + group - 1) / group;
  const long i4 = strip_levels(a, 4, ng), i8 = strip_levels(a, 8, ng);
  const long s8 = strip_levels(a, 8, 1);
  const long upto8[2] = {sizeof(TF) == 8 ? 4096 : 8192, sizeof(TF) == 8 ? 8192 : 16384};
  const bool tall[2] = {sizeof(TF) == 4 && i8 >= 65536, sizeof(TF) == 4 && s8 >= 200000};
  for (int p = 0; p < 2; p++)
    a.rows[p] = i4 <= 3072 ? 4 : (i8 <= upto8[p] ? 8 : (tall[p] ? 32 : 16));
}
template int strip_auto_group<double>(const FusedArgs<double>&);
template int strip_auto_group<float>(const FusedArgs<float>&);
template void strip_auto_rows<double>(FusedArgs<double>&, int);
template void strip_auto_rows<float>(FusedArgs<float>&, int);

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
