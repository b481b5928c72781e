// The interaction-region potential step for any phi length that is a product of two register radices: theta
// contractions on the matrix cores, phi transforms in place, the specular coupling added as the wave is read.
//
// Per workgroup: C = 8 NT consecutive izr (< nz_potential nr) of one (x, y) site, in three phases around a DVR tile in
// LDS (row theta C + column, phi along the row, rows of odd length).
//
// 1. FBR -> DVR, theta: D[theta, col] = sum_J L_m[theta, J] c[J, col] as 16 x 16 x 4 MFMA products of eight complex
//    columns. The blocks mJ = m and -m have one Legendre matrix up to the sign and one set of rotation factors, so they
//    are one task: its fragments and factors are read once, and its products are independent chains. A wavefront's psi
//    operands are loaded before its first product, its next task's fragments before this task's products.
// 2. phi. N = R1 R2 with the elements of a row placed so that each of the three passes (R1 forward; R2 forward, x
//    exp(i A), R2 backward on the same registers; R1 backward) works in place: one barrier a pass, one butterfly's
//    registers. R1 and R2 coprime (Good and Thomas): element n = (R2 n1 + R1 n2) mod N sits at n1 R2 + n2, frequency
//    k = k1 mod R1 = k2 mod R2 comes out at k1 R2 + k2, and there are no twiddles at all; else (Cooley and Tukey)
//    element n = R2 n1 + n2 and frequency k = k1 + R1 k2 with a twiddle W_N^{n2 k1} between the passes. The places of
//    phase 1 and the phi map of exp(i A) are in that order from the host (AngularPlan), so placing costs nothing.
//    Short lengths (R2 = 1) take one pass. In the second pass a thread keeps one k1: its R2 offsets into a row of
//    exp(i A) are set up once.
// 3. DVR -> FBR, x rot(dt/2), stored straight to HBM. The factor depends on J and r alone: the table holds one row
//    per distinct row of the caller's (irot, ir) table (rows of one J come out the same), short enough for the L1.
//
// Bound by latency: the phases of a tile wait for each other. At DZ (13 theta x 48 phi, two 82 KB tiles a CU) wavefronts
// wait in 51 % of their cycles in FP64 and 46 in complex64, with the vector units busy 32 and 52 %, the matrix cores 20
// and 20, LDS 19 and 24: 3.95 and 2.42 ms a launch for 9.33 and 4.67 GB. At 128 registers a lane some FP64 lengths keep
// values in scratch too (variants_angular.hpp).
#pragma once

#include "fft_ct.hpp"
#include "kernels.hpp"
#include "kernels_ct.hpp"
#include "kernels_mfma.hpp"
#include "kernels_zr.hpp"

namespace spo_dev {

// The mJ blocks m and -m (lane m of a wavefront holds task m's): byte offsets of their first rows in a site's column of
// psi and of their phi places in a DVR row, number of J, first fragments of L_m (bytes; forward, backward), whether
// L_{-m} = -L_m, and the first row in the rotation table (bytes).
struct AngularTask {
  int psi[2], place[2];
  int nb, fwd, bwd, negate, rot, pad[3];
};

struct AngularPlan {
  const AngularTask* tasks;
  const int* free_places;  // places of a row that hold no mJ block
  const int* phi_map;      // [op][place]: phi index of exp(i A) for the value at that place after the transforms
  const int* site_order;   // position -> ixy (-1: none), positions of one XCD (position mod 8) holding whole sites
  int n_tasks, n_free, sites_per_xcd, rows;
  unsigned inv_rows, inv_nr;
  int task_initial, side_initial, j_initial;  // the initial channel's task, block (0: m, 1: -m) and row there
  int rot_rows, frag_fwd, frag_bwd;  // table lengths: rows, fragments, fragments
};

constexpr int gcd_of(int a, int b) { return b == 0 ? a : gcd_of(b, a % b); }

// Places of the elements and of the frequencies of a phi row (host; see phase 2).
inline int phi_place(int n, int r1, int r2) {
  if (gcd_of(r1, r2) == 1) {
    for (int n1 = 0; n1 < r1; ++n1)
      for (int n2 = 0; n2 < r2; ++n2)
        if ((r2 * n1 + r1 * n2) % (r1 * r2) == n) return n1 * r2 + n2;
  }
  return n;  // n = r2 n1 + n2
}
inline int phi_frequency(int place, int r1, int r2) {
  const int k1 = place / r2, k2 = place % r2;
  if (gcd_of(r1, r2) != 1) return k1 + r1 * k2;
  for (int k = 0; k < r1 * r2; ++k)
    if (k % r1 == k1 && k % r2 == k2) return k;
  return -1;
}

template <typename T>
inline std::size_t angular_lds(int rows, int nphi) {
  return std::size_t(rows) * (nphi | 1) * sizeof(cx<T>);
}

__device__ __forceinline__ double flip_sign(double v, int bit) {
  return __longlong_as_double(__double_as_longlong(v) ^ (static_cast<long long>(bit) << 32));
}
__device__ __forceinline__ float flip_sign(float v, int bit) { return __int_as_float(__float_as_int(v) ^ bit); }

template <typename T, int R1, int R2, int NT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 4) void interaction_kernel_inplace(
    cx<T>* psi, const cx<double>* spec, Shape s, AngularPlan plan, const int* rep_of, const int* op_of,
    const T* frag_fwd, const T* frag_bwd, const unsigned* low_fwd, const unsigned* low_bwd, const cx<T>* exp_table,
    const cx<T>* rot_pm, const cx<T>* rot_half, const cx<T>* s2sc, const cx<T>* table_phi, const T* eps_phi) {
  using M = Mfma<T>;
  using acc_t = typename M::acc_t;
  constexpr int N = R1 * R2;
  constexpr int LD = N | 1;
  constexpr int C = 8 * NT;
  constexpr int THREADS = 64 * WAVES;
  constexpr unsigned CB = sizeof(cx<T>), TB = sizeof(T);
  constexpr bool kTwiddles = gcd_of(R1, R2) != 1;
  constexpr int TILES = 2 * NT;  // MFMA tiles of a task: side t / NT (m, -m), columns 8 (t % NT) + 0 .. 7
  // Tasks of a wavefront, and how many of them have their operands in flight in phase 1 (64 registers).
  constexpr int TASKS = (N / 2 + WAVES - 1) / WAVES;
  constexpr int DEPTH_MAX = 64 / (TILES * static_cast<int>(TB));
  constexpr int DEPTH = TASKS < DEPTH_MAX ? TASKS : DEPTH_MAX;
  extern __shared__ unsigned char smem_raw[];
  cx<T>* dvr = reinterpret_cast<cx<T>*>(smem_raw);

  // Workgroup -> (tile, site): the sites of an XCD (blockIdx mod 8) in tile pairs, so the halves of a cache line that
  // two neighbouring tiles hold meet in one L2, and the exp(i A) rows of a representative are read by one XCD.
  int tile, ixy;
  {
    const int x = blockIdx.x % 8, q = blockIdx.x / 8, rest = q / 2;
    tile = 2 * (rest / plan.sites_per_xcd) + q % 2;
    ixy = plan.site_order[8 * (rest % plan.sites_per_xcd) + x];
  }
  const int izr0 = tile * C;
  if (ixy < 0 || izr0 >= s.n_zr_pot) return;
  const int cw = min(C, s.n_zr_pot - izr0);
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int n = lane % 16, kk = lane / 16, ri = n & 1, col = n / 2;  // operand column n: complex column and component
  const int n_theta = s.n_theta, n_tasks = plan.n_tasks;
  const unsigned zr_bytes = static_cast<unsigned>(s.n_zr) * CB;

  const rsrc_t site = buffer_rsrc(psi + static_cast<long>(s.n_zr) * s.n_rot * ixy,
                                  static_cast<long>(s.n_zr) * s.n_rot * CB);
  const rsrc_t ffwd = buffer_rsrc(frag_fwd, 64L * plan.frag_fwd * sizeof(T));
  const rsrc_t fbwd = buffer_rsrc(frag_bwd, 64L * plan.frag_bwd * sizeof(T));
  const rsrc_t rots = buffer_rsrc(rot_pm, 2L * plan.rot_rows * s.nr * 16);
  const rsrc_t lo_f = buffer_rsrc(low_fwd, sizeof(T) == 4 ? 512L * s.n_blocks : 0);
  const rsrc_t lo_b = buffer_rsrc(low_bwd, sizeof(T) == 4 ? 512L * s.n_blocks : 0);

  // A task's fields come out of its lane without a memory access.
  const AngularTask mine = plan.tasks[min(lane, n_tasks - 1)];
  auto field = [&](int v, int p) { return __builtin_amdgcn_readlane(v, p); };

  const cx<T>* exp_rows =
      exp_table + static_cast<long>(s.n_tp) * (rep_of[ixy] + static_cast<long>(s.n_rep) * izr0);
  const int exp_stride = s.n_tp * s.n_rep;
  const int* map = plan.phi_map + N * op_of[ixy];
  // The thread's offsets into a row of exp(i A): of its k1 (R2 > 1), or of the whole row.
  constexpr int OFFS = R2 > 1 ? R2 : N;
  const int k1 = R2 > 1 ? tid % R1 : 0;
  int off[OFFS];
#pragma unroll
  for (int r = 0; r < OFFS; ++r) off[r] = map[k1 * OFFS + r];
  auto load_exp = [&](int row, cx<T> (&ev)[OFFS]) {
    const cx<T>* e = exp_rows + (exp_stride * min(row % C, cw - 1) + N * (row / C));
#pragma unroll
    for (int r = 0; r < OFFS; ++r) ev[r] = e[off[r]];
  };

  // Places without a block are zero.
  for (int f = 0; f < plan.n_free; ++f) {
    const int place = plan.free_places[f];
    for (int row = tid; row < plan.rows; row += THREADS) dvr[row * LD + place] = {};
  }

  // 1. FBR -> DVR (theta). J rows past the block meet zero fragment entries; columns past the region are computed and
  // never stored.
  const unsigned b_lane = static_cast<unsigned>(kk) * zr_bytes + static_cast<unsigned>(n) * TB;
  const unsigned izr_bytes = static_cast<unsigned>(izr0) * CB;
  unsigned char* d_lane = smem_raw + (static_cast<unsigned>(M::row(lane, 0) * C + col) * LD) * CB + ri * TB;
  constexpr int d_v = (sizeof(T) == 8 ? 4 : 1) * C * LD * static_cast<int>(CB);  // tile bytes between v and v + 1
  auto load_a = [&](rsrc_t frags, rsrc_t lows, int first, int steps, int p, T (&a)[4], lo_frag_t& lo) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      a[k] = k < steps ? buffer_load<T>(frags, lane * TB, static_cast<unsigned>(first) + k * 64u * TB) : T(0);
    if constexpr (sizeof(T) == 4) lo = legendre_low_fragment(lows, s.mj_max + p);
  };
  T a[4];
  lo_frag_t lo = {};
  if (wave < n_tasks) load_a(ffwd, lo_f, field(mine.fwd, wave), (field(mine.nb, wave) + 3) / 4, wave, a, lo);
#pragma unroll 1
  for (int i0 = 0; i0 < TASKS; i0 += DEPTH) {
    T bv[DEPTH][TILES][4];
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      const int p = wave + WAVES * (i0 + i);
      if (p < n_tasks) {
        const int nb = field(mine.nb, p);
        const unsigned base[2] = {static_cast<unsigned>(field(mine.psi[0], p)) + izr_bytes,
                                  static_cast<unsigned>(field(mine.psi[1], p)) + izr_bytes};
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (4 * k < nb) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
              bv[i][t][k] = buffer_load<T>(site, b_lane + (t % NT) * 8 * CB, base[t / NT] + 4u * k * zr_bytes);
          } else {
#pragma unroll
            for (int t = 0; t < TILES; ++t) bv[i][t][k] = T(0);
          }
      }
    }
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      const int p = wave + WAVES * (i0 + i);
      if (p < n_tasks) {
        const int nb = field(mine.nb, p), next = p + WAVES;
        T na[4] = {};
        lo_frag_t nlo = {};
        if (next < n_tasks) load_a(ffwd, lo_f, field(mine.fwd, next), (field(mine.nb, next) + 3) / 4, next, na, nlo);
        if (p == plan.task_initial) {
          // the initial channel: + rot(dt/2) (s2sc chi)
#pragma unroll
          for (int t = 0; t < TILES; ++t)
            if (t / NT == plan.side_initial) {
              const int izr = min(izr0 + 8 * (t % NT) + col, s.n_zr_pot - 1);
              const int ir = izr - s.nr * fast_div(izr, s.nr, plan.inv_nr);
              const cx<double> in = spec[izr];
              const cx<T> add = rot_half[s.ichn + s.n_rot * ir] * (s2sc[ixy] * cx<T>{T(in.x), T(in.y)});
#pragma unroll
              for (int k = 0; k < 4; ++k)
                if (4 * k + kk == plan.j_initial) bv[i][t][k] += ri ? add.y : add.x;
            }
        }
        acc_t acc[TILES] = {};
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (4 * k < nb) {
#pragma unroll
            for (int t = 0; t < TILES; ++t) acc[t] = M::fma(a[k], bv[i][t][k], acc[t]);
          }
        if constexpr (sizeof(T) == 4) {
#pragma unroll
          for (int t = 0; t < TILES; ++t) acc[t] = legendre_low_product(lo, bv[i][t], acc[t]);
        }
        const int bit = field(mine.negate, p) ? static_cast<int>(0x80000000u) : 0;
        unsigned char* d[2] = {d_lane + field(mine.place[0], p), d_lane + field(mine.place[1], p)};
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (M::row(lane, v) < n_theta) {
#pragma unroll
            for (int t = 0; t < TILES; ++t)
              if (t < NT || p > 0)
                *reinterpret_cast<T*>(d[t / NT] + v * d_v + (t % NT) * 8 * LD * static_cast<int>(CB)) =
                    t < NT ? acc[t][v] : flip_sign(acc[t][v], bit);
          }
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = na[k];
        lo = nlo;
      }
    }
  }
  __syncthreads();

  // 2. phi
  if constexpr (R2 == 1) {
    for (int row = tid; row < plan.rows; row += THREADS) {
      const cx<T>* e = exp_rows + (exp_stride * min(row % C, cw - 1) + N * (row / C));
      cx<T>* p = dvr + row * LD;
      cx<T> v[N];
#pragma unroll
      for (int r = 0; r < N; ++r) v[r] = p[r];
      rdft<N, T>(v, +1);
#pragma unroll
      for (int r = 0; r < N; ++r) v[r] = e[off[r]] * v[r];
      rdft<N, T>(v, -1);
#pragma unroll
      for (int r = 0; r < N; ++r) p[r] = v[r];
    }
    __syncthreads();
  } else {
    constexpr int RB = THREADS / R1;  // rows of a round of the second pass
    const int last = tid < RB * R1 ? plan.rows : 0;
    int row = tid / R1;
    cx<T> ev[OFFS];
    if (row < last) load_exp(row, ev);
    for (int b = tid; b < plan.rows * R2; b += THREADS) {
      const int n2 = fast_div(b, plan.rows, plan.inv_rows), row_a = b - n2 * plan.rows;
      cx<T>* p = dvr + row_a * LD + n2;
      cx<T> v[R1];
#pragma unroll
      for (int r = 0; r < R1; ++r) v[r] = p[r * R2];
      rdft<R1, T>(v, +1);
#pragma unroll
      for (int r = 0; r < R1; ++r) p[r * R2] = v[r];
    }
    __syncthreads();
    {
      cx<T> tw[R2], tw_lo[R2];
      if constexpr (kTwiddles) {
#pragma unroll
        for (int r = 1; r < R2; ++r) {
          tw[r] = conj(table_phi[r * k1]);
          if constexpr (sizeof(T) == 4) {
            const T e = eps_phi[r * k1];
            tw_lo[r] = {e * tw[r].x, e * tw[r].y};
          } else {
            tw_lo[r] = {};
          }
        }
      }
      // The exp(i A) values of the next row are in flight while this one is transformed.
      while (row < last) {
        cx<T> en[R2];
        if (row + RB < last) load_exp(row + RB, en);
        cx<T>* p = dvr + row * LD + k1 * R2;
        cx<T> v[R2];
#pragma unroll
        for (int r = 0; r < R2; ++r) v[r] = p[r];
        if constexpr (kTwiddles) {
#pragma unroll
          for (int r = 1; r < R2; ++r) v[r] = mul_hilo(tw[r], tw_lo[r], v[r]);
        }
        rdft<R2, T>(v, +1);
#pragma unroll
        for (int r = 0; r < R2; ++r) v[r] = ev[r] * v[r];
        rdft<R2, T>(v, -1);
        if constexpr (kTwiddles) {
#pragma unroll
          for (int r = 1; r < R2; ++r) v[r] = mul_hilo(conj(tw[r]), conj(tw_lo[r]), v[r]);
        }
#pragma unroll
        for (int r = 0; r < R2; ++r) p[r] = v[r];
#pragma unroll
        for (int r = 0; r < R2; ++r) ev[r] = en[r];
        row += RB;
      }
    }
    __syncthreads();
    for (int b = tid; b < plan.rows * R2; b += THREADS) {
      const int n2 = fast_div(b, plan.rows, plan.inv_rows), row = b - n2 * plan.rows;
      cx<T>* p = dvr + row * LD + n2;
      cx<T> v[R1];
#pragma unroll
      for (int r = 0; r < R1; ++r) v[r] = p[r * R2];
      rdft<R1, T>(v, -1);
#pragma unroll
      for (int r = 0; r < R1; ++r) p[r * R2] = v[r];
    }
    __syncthreads();
  }

  // 3. DVR -> FBR (theta), x rot(dt/2). theta rows past the grid read the last one (their fragment entries are zero).
  const int k_bwd = (n_theta + 3) / 4;
  const unsigned char* t_lane[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    t_lane[k] = smem_raw + (static_cast<unsigned>(min(4 * k + kk, n_theta - 1) * C + col) * LD) * CB + ri * TB;
  unsigned st_lane[4], rot_lane[NT];
#pragma unroll
  for (int v = 0; v < 4; ++v) st_lane[v] = static_cast<unsigned>(M::row(lane, v)) * zr_bytes + col * CB + ri * TB;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int izr = izr0 + 8 * t + col;
    const int ir = izr - s.nr * fast_div(izr, s.nr, plan.inv_nr);
    rot_lane[t] = (static_cast<unsigned>(M::row(lane, 0) * s.nr + ir) * 2u + ri) * 16u;
  }
  const unsigned rot_v = (sizeof(T) == 8 ? 4u : 1u) * s.nr * 32u;  // bytes between v and v + 1
  if (wave < n_tasks) load_a(fbwd, lo_b, field(mine.bwd, wave), k_bwd, wave, a, lo);
#pragma unroll 1
  for (int p = wave; p < n_tasks; p += WAVES) {
    const int nb = field(mine.nb, p), next = p + WAVES;
    const unsigned rot = static_cast<unsigned>(field(mine.rot, p));
    RotEntry<T> w[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) w[t][v] = buffer_load<RotEntry<T>>(rots, rot_lane[t], rot + v * rot_v);
    T na[4] = {};
    lo_frag_t nlo = {};
    if (next < n_tasks) load_a(fbwd, lo_b, field(mine.bwd, next), k_bwd, next, na, nlo);
    const int place[2] = {field(mine.place[0], p), field(mine.place[1], p)};
    const unsigned out[2] = {static_cast<unsigned>(field(mine.psi[0], p)) + izr_bytes,
                             static_cast<unsigned>(field(mine.psi[1], p)) + izr_bytes};
    T bv[TILES][4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int t = 0; t < TILES; ++t)
        bv[t][k] = k < k_bwd ? *reinterpret_cast<const T*>(t_lane[k] + place[t / NT] + (t % NT) * 8 * LD * static_cast<int>(CB))
                             : T(0);
    acc_t acc[TILES] = {};
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k < k_bwd) {
#pragma unroll
        for (int t = 0; t < TILES; ++t) acc[t] = M::fma(a[k], bv[t][k], acc[t]);
      }
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int t = 0; t < TILES; ++t) acc[t] = legendre_low_product(lo, bv[t], acc[t]);
    }
    const int bit = field(mine.negate, p) ? static_cast<int>(0x80000000u) : 0;
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      if (t >= NT && p == 0) break;  // m = 0 has one block
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const T mine_v = t < NT ? acc[t][v] : flip_sign(acc[t][v], bit);
        const T other = swap_adjacent_lanes(mine_v);
        const RotEntry<T>& f = w[t % NT][v];
        T r;
        if constexpr (sizeof(T) == 4)  // remainder products first, the nearest values fused on top (mul_hilo)
          r = fmaf(f.x, mine_v, fmaf(f.y, other, fmaf(f.lo_x, mine_v, f.lo_y * other)));
        else
          r = f.x * mine_v + f.y * other;
        if (8 * (t % NT) + col < cw && M::row(lane, v) < nb)
          buffer_store<T>(r, site, st_lane[v] + (t % NT) * 8 * CB, out[t / NT]);
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] = na[k];
    lo = nlo;
  }
}

}  // namespace spo_dev
