// interaction_kernel_inplace's instantiations, for the translation unit of each storage type.
#pragma once

#include <algorithm>

#include "variants.hpp"

namespace spo_dev {

// Radices (R1, R2) of the phi lengths that an angular grid takes up to MJMax 31: coprime wherever the length allows
// it (no twiddles), the smaller one second (a thread holds R2 values of the row, of exp(i A) and of the next exp(i A):
// 22 points as 2 x 11 in FP64 took 347 us at the HardWall workload, as 11 x 2 150), one pass up to 8 points. Four
// wavefronts a SIMD leave a lane 128 registers, and in FP64 the offsets and exp(i A) values that live across the R1 pass
// do not all fit: the default variants spill 2 registers at 22 points (12 bytes of scratch a lane), 1 at 42 (8), 10 at 44
// (44), 6 at 48 (28), 1 at 50 (8), 10 at 54 (44) and 74 at 64 (236); none at the other lengths and none in complex64.
// At 48 points (13 theta, 96 x 48 x 16 x 16) a launch writes 1.04 GB of scratch beside the wave's 4.19 GB.
#define SPO_PHI_RADICES(X)                                                                                    \
  X(2, 1) X(4, 1) X(6, 1) X(8, 1) X(5, 2) X(4, 3) X(7, 2) X(4, 4) X(9, 2) X(5, 4) X(11, 2) X(8, 3) X(7, 4)      \
  X(10, 3) X(8, 4) X(9, 4) X(8, 5) X(14, 3) X(11, 4) X(16, 3) X(10, 5) X(9, 6) X(8, 7) X(12, 5) X(8, 8)

// The wavefronts of a workgroup, in order of preference. A workgroup's phases wait for each other, so a CU needs
// several workgroups or many wavefronts in one; their number is set by the tile's LDS. The fewest wavefronts that give
// a CU 12 (FP64; complex64, half the latency per value, 16) are the fastest: fewer barriers' worth of idle lanes in
// the phi passes. Measured on MI355X, us per launch, FP64 tiles of 8 columns with 1 / 2 / 4 / 8 / 16 wavefronts:
//   4 KB (JMax 4, 3 theta x 10 phi): 75 / 90 / 122;  18 KB (JMax 10): - / 150 / 163 / 190;
//   26 KB (JMax 12): 253 with 4, 288 with 8;  52 KB (JMax 18): 490 with 4, 518 with 8;
//   82 KB (JMax 24, 13 theta x 48 phi): 5030 with 4, 4050 with 8, 5370 with 16;  117 KB (JMax 28): 6110, 5450, 4760.
// Complex64 takes tiles of 16 columns (whole 128-byte lines of a row; at 13 theta x 48 phi 2500 us against 3110 of 8
// columns), except the shortest rows, where one wavefront's worth of them is enough. A launch of few workgroups
// (the device holds 4096 of these) takes two wavefronts for the latency (64 x 16 x 4 x 4: 13.5 us against 15.2).
// 56 points in FP64 stay with interaction_mfma_kernel: at 13 to 15 theta one tile fills a CU, and with the 16 wavefronts
// that it then takes this kernel spilled 25 registers: 594 us (48 x 24 x 8 x 8, 14 theta) against 546 there, and 2149
// against 1960 (96 x 48 x 8 x 8).
template <typename T>
std::vector<Variant> interaction_inplace_variants(int nphi, int n_theta, long columns) {
  std::vector<Variant> out;
  if (n_theta > 16) return out;
#define Y(R1, R2, NT, W)                                                                                      \
  out.push_back({reinterpret_cast<const void*>(interaction_kernel_inplace<T, R1, R2, NT, W>), 64 * W, W,       \
                 angular_lds<T>(8 * NT * n_theta, nphi), {}, InteractionKind::in_place, 8 * NT, R1, R2});
#define X(R1, R2)                                                                                             \
  if (nphi == R1 * R2) {                                                                                      \
    if constexpr (R1 * R2 <= 12) {                                                                            \
      Y(R1, R2, 1, 1) Y(R1, R2, 1, 2)                                                                         \
    } else if constexpr (sizeof(T) == 4) {                                                                    \
      Y(R1, R2, 2, 4) Y(R1, R2, 2, 8) Y(R1, R2, 2, 16)                                                        \
    } else if constexpr (R1 * R2 == 56) {  /* see above */                                                    \
    } else if constexpr (R1 * R2 <= 22) {                                                                     \
      Y(R1, R2, 1, 1) Y(R1, R2, 1, 2) Y(R1, R2, 1, 4)                                                         \
    } else {                                                                                                  \
      Y(R1, R2, 1, 2) Y(R1, R2, 1, 4) Y(R1, R2, 1, 8) Y(R1, R2, 1, 16)                                        \
    }                                                                                                         \
  }
  SPO_PHI_RADICES(X)
#undef X
#undef Y
  if (out.empty()) return out;
  const int resident = std::max<int>(1, 163840 / out[0].lds), need = sizeof(T) == 8 ? 12 : 16;
  int best = out.back().param;
  for (auto v = out.rbegin(); v != out.rend(); ++v)
    if (resident * v->param >= need) best = v->param;
  if (best == 1 && columns / out[0].columns < 4096) best = 2;
  std::stable_sort(out.begin(), out.end(), [&](const Variant& a, const Variant& b) { return (a.param == best) > (b.param == best); });
  return out;
}

}  // namespace spo_dev
