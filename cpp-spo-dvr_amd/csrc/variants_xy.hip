// Instantiations of the T_xy kernel.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "variants.hpp"

namespace spo_dev {

// T_xy tiles with whole-line DFTs in registers (NX = NY a register radix; C izr per tile, C * NX threads): every even
// line length up to 16. Other lengths, and NX != NY, run the run-time engine: 12 x 12 in FP64 12.2 ms per launch (62640
// planes of 160 x 40) against 2.56 here, 10 x 10 in complex64 997 us against 143, 6 x 6 in FP64 113 us against 22.
#define SPO_XY_REG_SHAPES(X)                                                                                  \
  X(16, 16, 32) X(16, 16, 16) X(16, 16, 8) X(14, 14, 32) X(14, 14, 16) X(12, 12, 32) X(12, 12, 16) X(10, 10, 32) \
  X(10, 10, 16) X(8, 8, 32) X(8, 8, 16) X(6, 6, 32) X(4, 4, 64) X(4, 4, 32) X(2, 2, 64)

template <typename T>
std::vector<Variant> xy_reg_variants(int nx, int ny) {
  std::vector<Variant> out;
  // FP64 tiles of 16 izr at 16 x 16 go through LDS in halves (xy_reg_kernel SPLIT): 35 KB instead of 70 KB.
#define X(A, B, CC)                                                                                          \
  if (nx == A && ny == B) {                                                                                  \
    constexpr bool split = sizeof(T) == 8 && A == 16 && CC == 16;                                            \
    out.push_back({reinterpret_cast<const void*>(spo_dev::xy_reg_kernel<T, A, B, CC, split>), CC * A, CC,    \
                   spo_dev::xy_reg_lds<T>(A, B, CC, split)});                                               \
  }
  SPO_XY_REG_SHAPES(X)
#undef X
  // Default (first) variant, as measured on MI355X: the widest tile in both precisions. FP64 at 16 x 16: tiles of
  // 32 izr 3.04 ms per time step, of 16 (through LDS in halves) 3.12, of 8 3.43; at 8 x 8: 32 izr 0.112, 16 izr
  // 0.115. Complex64 at 16 x 16: 32 izr 1.76, 16 izr 1.90, 8 izr 2.58. Per launch at 12 x 12 in FP64 32 izr 2.56 ms, 64
  // izr 2.58, 16 izr 2.70; at 10 x 10 in complex64 143 us, 147, 150; at 6 x 6 in FP64 32 izr 21.7 us, 64 izr 23.1.
  std::stable_sort(out.begin(), out.end(), [](const Variant& a, const Variant& b) { return a.param > b.param; });
  return out;
}

template std::vector<Variant> xy_reg_variants<double>(int, int);
template std::vector<Variant> xy_reg_variants<float>(int, int);

}  // namespace spo_dev
