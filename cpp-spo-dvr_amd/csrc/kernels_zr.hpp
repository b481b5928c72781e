// T_Zr for any grid whose axes are products of two register radices: one (irot, ixy) plane per workgroup, the whole
// (Z, r) plane in LDS, every pass in place.
//
// An axis N = R1 R2 takes two passes. The first transforms x[j + r R2] over r (radix R1, fixed j < R2) and leaves
// output k1 where element r = k1 was; the second takes the R2 elements j of one k1, at k1 R2 + j, times W_N^{j k1},
// and leaves output k2 where element j = k2 was. Place k1 R2 + k2 then holds frequency k1 + R1 k2: the factor table
// is laid out in that order once (zr_factor_order), and the inverse transform runs the same passes backwards, so the
// wave comes out in natural order. A butterfly writes only the places it has read: a thread needs no more registers
// than one butterfly, whatever the number of butterflies it takes, and one barrier separates two passes (writing in
// Stockham order needs a second barrier between the reads and the writes of a pass, and every butterfly of the
// thread held across it). The second Z pass, the factor and the first inverse Z pass are one pass.
//
// The plane costs 2 P complex values of HBM traffic and 12 P of LDS traffic (six round trips). Rows in LDS are
// padded to an odd length, so the passes that run lanes along iz touch distinct bank groups; the HBM passes run
// lanes along j (consecutive addresses) and the Z passes along the place in the row.
//
// Measured on MI355X against the run-time engine's plane kernel (a tile in and out of LDS around every stage, radices
// up to 8 and 11): 160 x 40 in FP64 (62640 planes) 20.6 -> 4.14 ms, 110 x 48 in FP64 246 -> 49 us, 90 x 40 in
// complex64 1254 -> 222 us. Bound by LDS and the vector units where one plane fills a CU's LDS (nothing overlaps its
// loads: 160 x 40, 3.1 TB/s), by HBM with two or more in FP64 (96 x 48, 4.5 TB/s), by the vector units in complex64 (95 %
// busy at 96 x 48, LDS 62 %).
#pragma once

#include <type_traits>

#include "fft_ct.hpp"
#include "kernels.hpp"
#include "kernels_ct.hpp"

namespace spo_dev {

// The shape of a plane at run time: NR = a1 a2, NZ = b1 b2 (a radix 1 is a pass left out), and m / 2^32 = 1 / n
// rounded up for the divisors of the task indices (exact for every index below 2^32 / n).
struct ZrShape {
  int nz, nr, a1, a2, b1, b2;
  unsigned inv_a2, inv_nz, inv_nr;
};

// fast_div's multiplier for the divisor n.
inline unsigned inverse_of(int n) { return n == 1 ? 0u : static_cast<unsigned>(((1ull << 32) + n - 1) / n); }

__device__ __forceinline__ int fast_div(int x, int n, unsigned inv) {
  return n == 1 ? x : static_cast<int>(__umulhi(static_cast<unsigned>(x), inv));
}

// Calls f with the radix (at most MOST) as a compile-time constant.
template <int MOST, class F>
__device__ __forceinline__ void with_radix(int r, F&& f) {
  if constexpr (MOST > 16) {
    if (r == 18) return f(std::integral_constant<int, 18>{});
    if (r == 20) return f(std::integral_constant<int, 20>{});
    if (r == 22) return f(std::integral_constant<int, 22>{});
  }
  switch (r) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    case 9: f(std::integral_constant<int, 9>{}); break;
    case 10: f(std::integral_constant<int, 10>{}); break;
    case 11: f(std::integral_constant<int, 11>{}); break;
    case 12: f(std::integral_constant<int, 12>{}); break;
    case 14: f(std::integral_constant<int, 14>{}); break;
    case 15: f(std::integral_constant<int, 15>{}); break;
    case 16: f(std::integral_constant<int, 16>{}); break;
    default: break;
  }
}
template <int MOST, int R, class F>
__device__ __forceinline__ void with_radix(std::integral_constant<int, R>, F&& f) {
  f(std::integral_constant<int, R>{});
}

// The plane's shape as run-time values or as compile-time constants.
template <int MOST>
struct ZrRunTime {
  static constexpr int kMost = MOST;  // the largest radix
  ZrShape s;
  __device__ __forceinline__ explicit ZrRunTime(const ZrShape& shape) : s(shape) {}
  __device__ __forceinline__ int nz() const { return s.nz; }
  __device__ __forceinline__ int nr() const { return s.nr; }
  __device__ __forceinline__ int a1() const { return s.a1; }
  __device__ __forceinline__ int a2() const { return s.a2; }
  __device__ __forceinline__ int b1() const { return s.b1; }
  __device__ __forceinline__ int b2() const { return s.b2; }
  __device__ __forceinline__ int div_a2(int x) const { return fast_div(x, s.a2, s.inv_a2); }
  __device__ __forceinline__ int div_nz(int x) const { return fast_div(x, s.nz, s.inv_nz); }
  __device__ __forceinline__ int div_nr(int x) const { return fast_div(x, s.nr, s.inv_nr); }
};
template <int NZ, int NR, int A1, int A2, int B1, int B2>
struct ZrStatic {
  static constexpr int kMost = 16;
  static_assert(A1 * A2 == NR && B1 * B2 == NZ, "ZrStatic: radices must multiply to the lengths");
  __device__ __forceinline__ explicit ZrStatic(const ZrShape&) {}
  template <int V>
  using c = std::integral_constant<int, V>;
  __device__ __forceinline__ c<NZ> nz() const { return {}; }
  __device__ __forceinline__ c<NR> nr() const { return {}; }
  __device__ __forceinline__ c<A1> a1() const { return {}; }
  __device__ __forceinline__ c<A2> a2() const { return {}; }
  __device__ __forceinline__ c<B1> b1() const { return {}; }
  __device__ __forceinline__ c<B2> b2() const { return {}; }
  __device__ __forceinline__ int div_a2(int x) const { return x / A2; }
  __device__ __forceinline__ int div_nz(int x) const { return x / NZ; }
  __device__ __forceinline__ int div_nr(int x) const { return x / NR; }
};

// Row length of the plane in LDS (odd) and its LDS bytes (complex64: the twiddles and their remainders behind it).
__host__ __device__ constexpr int zr_row(int nr) { return nr | 1; }
template <typename T>
inline std::size_t zr_plane_lds(int nz, int nr) {
  return std::size_t(nz) * zr_row(nr) * sizeof(cx<T>) +
         (zr_twiddles_in_lds<T>() ? std::size_t(nz + nr) * 2 * sizeof(cx<T>) : 0);
}

// One plane through the passes: read from `plane`, every value of the result handed to out(iz, ir, value).
// factor and factor_lo (complex64: its FP32 remainders, mul_hilo) in the order of zr_factor_order; eps_z, eps_r: the
// complex64 twiddle tables' modulus corrections (twiddle()). FP64 keeps the twiddles in the cache, where they do not
// compete with the plane for LDS bandwidth; complex64 holds them and their remainders in LDS.
// row >= 0: only Z row `row` of the result is formed (the inverse r passes run for that row alone).
template <typename T, class Dims, int THREADS, class Out>
__device__ __forceinline__ void zr_transform(const cx<T>* plane, const ZrShape& shape, const cx<T>* table_z,
                                             const cx<T>* table_r, const cx<T>* factor, const T* eps_z, const T* eps_r,
                                             const cx<T>* factor_lo, int row, Out&& out) {
  extern __shared__ unsigned char smem_raw[];
  cx<T>* t = reinterpret_cast<cx<T>*>(smem_raw);
  const Dims d(shape);
  const auto nz = d.nz();
  const auto nr = d.nr();
  const auto a1 = d.a1();
  const auto a2 = d.a2();
  const auto b1 = d.b1();
  const auto b2 = d.b2();
  const int ld = zr_row(nr);
  const int tid = threadIdx.x;
  const cx<T>* lo_r = nullptr;
  const cx<T>* lo_z = nullptr;
  if constexpr (zr_twiddles_in_lds<T>()) {
    cx<T>* tw_r = t + nz * ld;
    cx<T>* tw_z = tw_r + nr;
    cx<T>* l_r = tw_z + nz;
    cx<T>* l_z = l_r + nr;
    for (int e = tid; e < nr; e += THREADS) {
      const cx<T> w = table_r[e];
      const T k = eps_r[e];
      tw_r[e] = w;
      l_r[e] = {k * w.x, k * w.y};
    }
    for (int e = tid; e < nz; e += THREADS) {
      const cx<T> w = table_z[e];
      const T k = eps_z[e];
      tw_z[e] = w;
      l_z[e] = {k * w.x, k * w.y};
    }
    table_r = tw_r;
    table_z = tw_z;
    lo_r = l_r;
    lo_z = l_z;
  }

  // r forward, radix a1: butterfly (iz, j < a2) from HBM.
  with_radix<Dims::kMost>(a1, [&](auto radix) {
    constexpr int R = decltype(radix)::value;
    const int n = nz * a2;
#pragma unroll 2
    for (int b = tid; b < n; b += THREADS) {
      const int iz = d.div_a2(b), j = b - iz * a2;
      const cx<T>* src = plane + (iz * nr + j);
      cx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = src[r * a2];
      rdft<R, T>(v, -1);
      cx<T>* dst = t + (iz * ld + j);
#pragma unroll
      for (int r = 0; r < R; ++r) dst[r * a2] = v[r];
    }
  });
  __syncthreads();
  // r forward, radix a2: butterfly (iz, k1 < a1), lanes along iz.
  with_radix<Dims::kMost>(a2, [&](auto radix) {
    constexpr int R = decltype(radix)::value;
    if constexpr (R > 1) {
      const int n = nz * a1;
      for (int b = tid; b < n; b += THREADS) {
        const int k1 = d.div_nz(b), iz = b - k1 * nz;
        cx<T>* p = t + (iz * ld + k1 * R);
        cx<T> v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = p[r];
        twiddle_lo<T, R>(v, table_r, lo_r, k1, -1);
        rdft<R, T>(v, -1);
#pragma unroll
        for (int r = 0; r < R; ++r) p[r] = v[r];
      }
    }
  });
  __syncthreads();
  // Z forward, radix b1: butterfly (place in the row, j < b2), lanes along the row.
  with_radix<Dims::kMost>(b1, [&](auto radix) {
    constexpr int R = decltype(radix)::value;
    const int n = nr * b2, step = b2 * ld;
    for (int b = tid; b < n; b += THREADS) {
      const int j = d.div_nr(b), pr = b - j * nr;
      cx<T>* p = t + (j * ld + pr);
      cx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = p[r * step];
      rdft<R, T>(v, -1);
#pragma unroll
      for (int r = 0; r < R; ++r) p[r * step] = v[r];
    }
  });
  __syncthreads();
  // Z forward radix b2, x factor, Z inverse radix b2: butterfly (place in the row, k1 < b1).
  with_radix<Dims::kMost>(b2, [&](auto radix) {
    constexpr int R = decltype(radix)::value;
    const int n = nr * b1;
    for (int b = tid; b < n; b += THREADS) {
      const int k1 = d.div_nr(b), pr = b - k1 * nr;
      cx<T>* p = t + (k1 * R * ld + pr);
      const int f = k1 * R * nr + pr;
      cx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = p[r * ld];
      twiddle_lo<T, R>(v, table_z, lo_z, k1, -1);
      rdft<R, T>(v, -1);
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = mul_factor(factor[f + r * nr], v[r], factor_lo, f + r * nr);
      rdft<R, T>(v, +1);
      twiddle_lo<T, R>(v, table_z, lo_z, k1, +1);
#pragma unroll
      for (int r = 0; r < R; ++r) p[r * ld] = v[r];
    }
  });
  __syncthreads();
  // Z inverse, radix b1.
  with_radix<Dims::kMost>(b1, [&](auto radix) {
    constexpr int R = decltype(radix)::value;
    const int n = nr * b2, step = b2 * ld;
    for (int b = tid; b < n; b += THREADS) {
      const int j = d.div_nr(b), pr = b - j * nr;
      cx<T>* p = t + (j * ld + pr);
      cx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = p[r * step];
      rdft<R, T>(v, +1);
#pragma unroll
      for (int r = 0; r < R; ++r) p[r * step] = v[r];
    }
  });
  __syncthreads();
  // r inverse, radix a2 (row mode: of that row alone).
  with_radix<Dims::kMost>(a2, [&](auto radix) {
    constexpr int R = decltype(radix)::value;
    if constexpr (R > 1) {
      const int n = nz * a1;
      for (int b = tid; b < n; b += THREADS) {
        const int k1 = d.div_nz(b), iz = b - k1 * nz;
        if (row >= 0 && iz != row) continue;
        cx<T>* p = t + (iz * ld + k1 * R);
        cx<T> v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = p[r];
        rdft<R, T>(v, +1);
        twiddle_lo<T, R>(v, table_r, lo_r, k1, +1);
#pragma unroll
        for (int r = 0; r < R; ++r) p[r] = v[r];
      }
    }
  });
  __syncthreads();
  // r inverse, radix a1, to HBM.
  with_radix<Dims::kMost>(a1, [&](auto radix) {
    constexpr int R = decltype(radix)::value;
    const int n = nz * a2;
    for (int b = tid; b < n; b += THREADS) {
      const int iz = d.div_a2(b), j = b - iz * a2;
      if (row >= 0 && iz != row) continue;
      const cx<T>* src = t + (iz * ld + j);
      cx<T> v[R];
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = src[r * a2];
      rdft<R, T>(v, +1);
#pragma unroll
      for (int r = 0; r < R; ++r) out(iz, j + r * a2, v[r]);
    }
  });
}

// T_Zr of one (irot, ixy) plane per workgroup. row >= 0: psi is only read, and Z row `row` of each transformed plane
// (NR values) goes to row_out[plane * NR + ir]; row < 0: psi is transformed in place and row_out is unused.
template <typename T, class Dims, int THREADS>
__global__ __launch_bounds__(THREADS) void zr_inplace_kernel(cx<T>* psi, ZrShape shape, const cx<T>* table_z,
                                                             const cx<T>* table_r, const cx<T>* factor, const T* eps_z,
                                                             const T* eps_r, const cx<T>* factor_lo, cx<T>* row_out,
                                                             int row) {
  const Dims d(shape);
  const auto nr = d.nr();
  cx<T>* plane = psi + static_cast<long>(blockIdx.x) * (d.nz() * nr);
  cx<T>* line = row_out + static_cast<long>(blockIdx.x) * nr;
  zr_transform<T, Dims, THREADS>(plane, shape, table_z, table_r, factor, eps_z, eps_r, factor_lo, row,
                                 [&](int iz, int ir, cx<T> v) {
                                   if (row >= 0)
                                     line[ir] = v;
                                   else
                                     plane[iz * nr + ir] = v;
                                 });
}

// The specular grid's whole step by one workgroup, for a grid that fits in LDS: its kinetic step, then (potential != 0)
// exp(-i vasy dt) between rot(dt/2) for iz >= nzpot and the Z and r absorbers
// (src/propagation/specular_operator.cpp:40-71). The grid is a few thousand points and the step is a chain of passes:
// one workgroup does it in 11 us at 128 x 16 and 32 us at 198 x 48 points, where three line-FFT launches and the
// potential's took 38 and 102 us. The axes' radices go up to 22 here: with a whole CU's registers for one workgroup a
// thread has 256, and 512 threads are two lines or more a thread at these sizes.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void specular_plane_kernel(cx<double>* spec, ZrShape shape, const cx<double>* table_z,
                                                                 const cx<double>* table_r, const cx<double>* factor,
                                                                 int potential, int nzpot, const cx<double>* gas,
                                                                 const double* z_opt, const double* r_opt, int r_first,
                                                                 int r_last) {
  zr_transform<double, ZrRunTime<22>, THREADS>(
      spec, shape, table_z, table_r, factor, nullptr, nullptr, nullptr, -1, [&](int iz, int ir, cx<double> v) {
        if (potential) {
          if (iz >= nzpot) v = gas[ir] * v;
          v = scale(v, z_opt[iz]);
          if (ir >= r_first && ir <= r_last) v = scale(v, r_opt[ir]);
        }
        spec[iz * shape.nr + ir] = v;
      });
}

// Place (kz place, kr place) of the plane after the forward passes -> its entry (kz, kr) of the (iz, ir) factor.
inline long zr_factor_order(const ZrShape& s, int place_z, int place_r) {
  const int kz = place_z / s.b2 + s.b1 * (place_z % s.b2), kr = place_r / s.a2 + s.a1 * (place_r % s.a2);
  return static_cast<long>(kz) * s.nr + kr;
}

}  // namespace spo_dev
