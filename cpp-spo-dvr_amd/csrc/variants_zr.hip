// Instantiations of the T_Zr kernel.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "variants.hpp"

namespace spo_dev {

namespace {

// Shapes with compile-time radices (NZ, NR, A1, A2, B1, B2, threads): NR = A1 A2, NZ = B1 B2. The variants of one
// shape (its radices, its block size) compute the same transforms with their roundings in another order; the launch
// tuner picks among them. FP64 order of preference. Measured on MI355X at 96 x 48, FP64 / complex64, us per launch of
// 82688 planes: 4 x 12, 12 x 8, 384 threads 2695 / 1593; 6 x 8 with 384 2715 / 1590; 6 x 8 with 512 2750 / 1488;
// 4 x 12 with 512 2730 / 1531; 3 x 16 with 384 2833 / 1598, with 512 2843 / 1501, with 192 3004 / 1719. The kernel
// that wrote its passes in Stockham order (two barriers a pass, every butterfly of a thread in registers) took
// 2884 / 1604 at its best. 128 x 32 (FP64): 135 with 512 threads, 145 with 256.
// What the compile-time radices gain over the run-time-shaped kernel at the same shape, us per launch of 5824 planes, FP64
// and complex64, each at its best block: 96 x 48 202 against 220 and 115 against 157; 128 x 32 181 / 191 and 99 / 125;
// 96 x 32 132 / 149 and 75 / 101; 80 x 16 54 / 65 and 40 / 52; 64 x 16 41 / 52 and 30 / 42. A shape is listed while it
// gains: 176 x 56 (7 x 8, 11 x 16, 512 threads) took 830 and 618 us where the run-time-shaped kernel, with 16 x 11 along Z
// and 1024 threads, takes 591 and 473 (the kernel in Stockham order 693 and 720).
#define SPO_ZR_SHAPES(X)                                                                                     \
  X(96, 48, 4, 12, 12, 8, 384) X(96, 48, 6, 8, 12, 8, 384) X(96, 48, 6, 8, 12, 8, 512)                        \
  X(96, 48, 4, 12, 12, 8, 512) X(96, 48, 3, 16, 12, 8, 384) X(96, 48, 3, 16, 12, 8, 512)                       \
  X(96, 48, 3, 16, 12, 8, 192)                                                                                 \
  X(128, 32, 4, 8, 16, 8, 512) X(128, 32, 4, 8, 16, 8, 256) X(64, 16, 4, 4, 8, 8, 256)                         \
  X(64, 16, 4, 4, 8, 8, 128) X(80, 16, 4, 4, 8, 10, 256) X(80, 16, 4, 4, 8, 10, 128)                           \
  X(96, 32, 4, 8, 12, 8, 512) X(96, 32, 4, 8, 12, 8, 256)

// The two radices of an axis (first <= second <= most, as equal as they come), or {0, 0}.
struct RadixPair {
  int low, high;
};
RadixPair radix_pair(int n, int most = 16) {
  for (int low = most; low >= 1; --low)
    if (low * low <= n && n % low == 0 && register_radix(low, most) && register_radix(n / low, most)) return {low, n / low};
  return {0, 0};
}

ZrShape zr_shape(int nz, int nr, int a1, int a2, int b1, int b2) {
  return {nz, nr, a1, a2, b1, b2, inverse_of(a2), inverse_of(nz), inverse_of(nr)};
}

}  // namespace

template <typename T>
std::vector<Variant> zr_variants(int nz, int nr) {
  std::vector<Variant> out;
  const std::size_t lds = zr_plane_lds<T>(nz, nr);
#define X(A, B, A1, A2, B1, B2, TH)                                                                              \
  if (nz == A && nr == B)                                                                                        \
    out.push_back({reinterpret_cast<const void*>(zr_inplace_kernel<T, ZrStatic<A, B, A1, A2, B1, B2>, TH>), TH, \
                   TH, lds, zr_shape(A, B, A1, A2, B1, B2)});
  SPO_ZR_SHAPES(X)
#undef X
  if (!out.empty()) {
    // complex64 planes take half the LDS, and the largest block is the fastest
    if (sizeof(T) == 4)
      std::stable_sort(out.begin(), out.end(), [](const Variant& a, const Variant& b) { return a.threads > b.threads; });
    return out;
  }
  // Any other shape whose axes are products of two radices: the run-time-shaped kernel. The longer radix of r goes to
  // the second pass (its HBM runs are a2 values long), the shorter of Z to the pass that transforms twice. Other
  // orders of the same radices were 4 to 100 % slower (160 x 40 in FP64: 4.14 ms against 4.56 to 6.25; 110 x 48: 49 us
  // against 51 to 56; 90 x 40 in complex64: 222 us against 226 to 230).
  const RadixPair r = radix_pair(nr), z = radix_pair(nz);
  if (r.low == 0 || z.low == 0) return out;
  const ZrShape s = zr_shape(nz, nr, r.low, r.high, z.high, z.low);
#define X(TH) out.push_back({reinterpret_cast<const void*>(zr_inplace_kernel<T, ZrRunTime<16>, TH>), TH, TH, lds, s});
  X(256) X(512) X(1024)
#undef X
  // Block size: the largest with which the workgroups that the planes' LDS lets onto a CU (160 KB) stay within the
  // wavefronts that the kernel's registers allow there (FP64 16, complex64 28). Measured, us with 256 / 512 / 1024
  // threads: 160 x 40 in FP64, one workgroup per CU, 5141 / 4238 / 4138; 110 x 48 in FP64, one, 62.7 / 52.3 / 48.6;
  // 90 x 40 in complex64, five, 222 / 229 / 371.
  const int resident = std::max<int>(1, 163840 / lds), most = 64 * (sizeof(T) == 8 ? 16 : 28);
  int best = 256;
  for (int th : {512, 1024})
    if (resident * th <= most) best = th;
  std::stable_sort(out.begin(), out.end(),
                   [&](const Variant& a, const Variant& b) { return (a.threads == best) > (b.threads == best); });
  return out;
}

const void* specular_plane(int nz, int nr, ZrShape& shape) {
  const RadixPair r = radix_pair(nr, 22), z = radix_pair(nz, 22);
  if (r.low == 0 || z.low == 0) return nullptr;
  shape = zr_shape(nz, nr, r.low, r.high, z.high, z.low);
  return reinterpret_cast<const void*>(specular_plane_kernel<kSpecularThreads>);
}

template std::vector<Variant> zr_variants<double>(int, int);
template std::vector<Variant> zr_variants<float>(int, int);

}  // namespace spo_dev
