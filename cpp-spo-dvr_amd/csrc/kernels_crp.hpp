// The CRP surface (SystemID CRPlibrary) on the device: V alone at a molecular geometry, FP64.
// The statements are the value statements of the host restatement (host/crp.cpp) in the same operand order
// (src/crplib/qd_wrapper.cpp:46-66, molecule_surface.cpp:249-315, hexagonal_interaction.cpp, site_interpolation.cpp,
// hexagonal_atom_surface.cpp:109-283, spline.cpp); FMA contraction is off so that the only differences from the
// host are those of the device's sin / cos / acos / atan2 and of the sums over the cluster and over the slab's atoms,
// which are added in a few runs of consecutive terms. A geometry where the host stops with an error (an atom on a
// surface atom, z outside the atom-surface data) gives NaN; the caller turns it into an error.
//
// A workgroup takes 64 points, a lane of every wavefront one of them, and its wavefronts share out what a point needs:
// the cluster's pair terms, the slab's, the molecular cuts, the atom splines, the Fourier terms and the sites, which
// meet in LDS. A point is some 80 000 operations, nine tenths of them pair terms, each a search and a cubic: a thread
// that did it all needed 256 registers and 592 bytes of scratch, one wavefront a SIMD: 318 us for 1000 points and
// 1.92 ms for 300 007 with a slab of 73 atoms (now 43 us and 0.81 ms; the operations bound it, 0.6 ms of them in all),
// 12.9 ms for a potential grid of 4.46 million points and 14.8 for one of 3.94 million with the slab (now 4.3 and 7.0).
// At four wavefronts a SIMD a lane has 128 registers, and 104 to 136 bytes of its values still go to scratch, nearly all of
// them inside the pair sums.
#pragma once

#include <hip/hip_runtime.h>

#include <array>

#include "../host/crp_tables.hpp"

#pragma clang fp contract(off)

namespace spo_dev {

__constant__ std::array<double, 100> kCrpAtomC3v = spo::crp_tables::kAtomC3vTable;
__constant__ std::array<double, 49> kCrpAtomC6v = spo::crp_tables::kAtomC6vTable;
__constant__ std::array<double, 144> kCrpMolecule = spo::crp_tables::kMoleculeTable;

// Device pointers of a packed surface (the layout of spo_hip_crp_surface).
struct CrpDev {
  int c3v, n_basis, n_cuts, n_corrugation, n_cluster, n_h2, n_zdep;
  double a, zso_min, zso_max, r_min, r_max, z_min, h2_asymptote;
  const double* corrugation;
  const double* cluster;
  const int* atom_offsets;
  const double* atom_splines;
  const int* cut_shape;
  const long* cut_offsets;
  const double* cut_data;
  const double* h2;
  const double* zdep;
  int square, cell_nz;
  const double* cell;  // C4v: x[5] y[5] z[nz], f xx yy xxyy zz zzxx zzyy zzxxyy (25 nz each)
};

// SPLINT / UBICAR bisection: the lower knot of the interval holding t.
__device__ inline int crp_bisect(const double* x, int n, double t) {
  int lo = 0, hi = n - 1;
  while (hi - lo > 1) {
    const int k = (hi + lo) / 2;
    if (x[k] > t) {
      hi = k;
    } else {
      lo = k;
    }
  }
  return lo;
}

// SPLINT value; s = x[n] y[n] F''[n]
__device__ inline double crp_splint(const double* s, int n, double t) {
  const double* x = s;
  const double* y = s + n;
  const double* m = s + 2 * n;
  const int lo = crp_bisect(x, n, t), hi = lo + 1;
  const double h = x[hi] - x[lo];
  const double a = (x[hi] - t) / h;
  const double b = (t - x[lo]) / h;
  return a * y[lo] + b * y[hi] + ((a * a * a - a) * m[lo] + (b * b * b - b) * m[hi]) * (h * h) / 6.0;
}

// DPL: linear outside the knots
__device__ inline double crp_dpl(const double* s, int n, double t) {
  const double* x = s;
  const double* y = s + n;
  const double* m = s + 2 * n;
  int lo = 0, hi = n;
  while (lo < hi) {  // the number of knots below t
    const int mid = (lo + hi) / 2;
    if (x[mid] < t) {
      lo = mid + 1;
    } else {
      hi = mid;
    }
  }
  int k = lo + 1;
  if (t == x[0]) k = 2;
  if (k <= 1) {
    const double e = x[1] - x[0];
    return ((y[1] - y[0]) / e - m[1] * e / 6.0) * (t - x[0]) + y[0];
  }
  if (k > n) {
    const double e = x[n - 1] - x[n - 2];
    return ((y[n - 1] - y[n - 2]) / e + m[n - 2] * e / 6.0) * (t - x[n - 1]) + y[n - 1];
  }
  const int i = k - 1;
  const double f = x[i] - t;
  const double g = t - x[i - 1];
  const double e = f + g;
  return (-g * f * (m[i - 1] * (f + e) + m[i] * (g + e)) + 6.0 * (g * y[i] + f * y[i - 1])) / (6.0 * e);
}


// SPLINT3D value weights in one direction (x**3.0 a call of pow, as there)
__device__ inline void crp_w3(const double* x, int i, double t, double& a, double& b, double& c, double& d) {
  const double h = x[i + 1] - x[i];
  a = (x[i + 1] - t) / h;
  b = 1.0 - a;
  c = (pow(a, 3.0) - a) / 6.0 * (h * h);
  d = (pow(b, 3.0) - b) / 6.0 * (h * h);
}

// An atom's position in the surface cell: ORIGEN and REGION for C4v, ORIGEN2 for the hexagonal surfaces (false: too far
// out to fold).
__device__ inline bool crp_fold(const CrpDev& s, double px, double py, double& x, double& y) {
  using namespace spo::crp_tables;
  const double a = s.a;
  const double bigx = s.square ? px : px - py * kUsq3;
  const double bigy = s.square ? py : 2.00 * py * kUsq3;
  const double o1 = bigx / a, o2 = bigy / a;
  if (!(fabs(o1) < 2.0e9) || !(fabs(o2) < 2.0e9)) return false;
  const int i1 = o1 >= 0.0 ? static_cast<int>(o1) : static_cast<int>(o1 - 1.0);
  const int i2 = o2 >= 0.0 ? static_cast<int>(o2) : static_cast<int>(o2 - 1.0);
  x = bigx - i1 * a;
  y = bigy - i2 * a;
  if (!s.square) {
    const double skewed = y;
    x = x + skewed * 0.500;
    y = kSq3 * skewed * 0.500;
    return true;
  }
  // REGION (the gradient's region is not needed for V)
  if (y <= a / 2.0) {
    if (x <= a / 2.0) {
      if (!(x >= y)) {
        const double t = x;
        x = y;
        y = t;
      }
    } else if (y >= (a - x)) {
      const double t = x;
      x = y;
      y = a - t;
    } else {
      x = a - x;
    }
  } else if (x <= a / 2.0) {
    if (y > (a - x)) {
      y = a - y;
    } else {
      const double t = x;
      x = a - y;
      y = t;
    }
  } else if (x > y) {
    const double t = x;
    x = a - y;
    y = a - t;
  } else {
    x = a - x;
    y = a - y;
  }
  return true;
}

// The C4v cell's periodic 3D spline at the folded position (SPLINT3D value).
__device__ inline double crp_cell(const CrpDev& s, double x, double y, double pz) {
  const int nz = s.cell_nz;
  const double* gx = s.cell;
  const double* gz = s.cell + 10;
  if (x < gx[0] || x > gx[4] || y < gx[5] || y > gx[9] || pz < gz[0]) {
    return __builtin_nan("");
  }
  const int i = crp_bisect(gx, 5, x), j = crp_bisect(gx + 5, 5, y), k = crp_bisect(gz, nz, pz);
  double xa, xb, xc, xd, ya, yb, yc, yd, za, zb, zc, zd;
  crp_w3(gx, i, x, xa, xb, xc, xd);
  crp_w3(gx + 5, j, y, ya, yb, yc, yd);
  crp_w3(gz, k, pz, za, zb, zc, zd);
  const long plane = 25L * nz;
  const double* f = s.cell + 10 + nz;
  auto plane_sum = [&](const double* g, const double* gxx, const double* gyy, const double* gxxyy, int kk) {
    const long p00 = i + 5L * (j + 5L * kk), p10 = p00 + 1, p01 = p00 + 5, p11 = p01 + 1;
    return ya * (xa * g[p00] + xb * g[p10] + xc * gxx[p00] + xd * gxx[p10]) +
           yb * (xa * g[p01] + xb * g[p11] + xc * gxx[p01] + xd * gxx[p11]) +
           yc * (xa * gyy[p00] + xb * gyy[p10] + xc * gxxyy[p00] + xd * gxxyy[p10]) +
           yd * (xa * gyy[p01] + xb * gyy[p11] + xc * gxxyy[p01] + xd * gxxyy[p11]);
  };
  const double *fxx = f + plane, *fyy = f + 2 * plane, *fxxyy = f + 3 * plane, *fzz = f + 4 * plane,
               *fzzxx = f + 5 * plane, *fzzyy = f + 6 * plane, *fzzxxyy = f + 7 * plane;
  const double t0 = plane_sum(f, fxx, fyy, fxxyy, k), t1 = plane_sum(f, fxx, fyy, fxxyy, k + 1);
  const double t2 = plane_sum(fzz, fzzxx, fzzyy, fzzxxyy, k), t3 = plane_sum(fzz, fzzxx, fzzyy, fzzxxyy, k + 1);
  return za * t0 + zb * t1 + zc * t2 + zd * t3;
}

// n / h for y = 1 / h rounded to nearest: two corrections by the exact remainder give the rounded quotient.
__device__ __forceinline__ double crp_quotient(double n, double h, double y) {
  double q = n * y;
  q = fma(fma(-q, h, n), y, q);
  return fma(fma(-q, h, n), y, q);
}

// The corrugation function's spline in LDS: its knots for the search (up to `size`, a power of two, +inf from the last
// knot on), then 7 doubles an interval: both knots, values and second derivatives, 1 / width. An odd stride spreads
// the lanes' intervals over the banks.
struct CrpStaged {
  const double* knots;
  const double* intervals;
  int size, last;  // last interval
};
__host__ __device__ inline int crp_staged_size(int n) {
  int size = 2;
  while (size < n) size *= 2;
  return size;
}
__host__ __device__ inline int crp_staged_doubles(int n) { return crp_staged_size(n) + 7 * (n - 1); }

// crp_splint from that table.
__device__ inline double crp_staged_splint(const CrpStaged& c, double t) {
  int lo = 0;
  for (int step = c.size >> 1; step > 0; step >>= 1) lo = c.knots[lo + step] > t ? lo : lo + step;
  lo = lo < c.last ? lo : c.last;  // t = NaN
  const double* i = c.intervals + 7 * lo;
  const double h = i[1] - i[0];
  const double a = crp_quotient(i[1] - t, h, i[6]);
  const double b = crp_quotient(t - i[0], h, i[6]);
  const double bend = ((a * a * a - a) * i[4] + (b * b * b - b) * i[5]) * (h * h);
  return a * i[2] + b * i[3] + crp_quotient(bend, 6.0, 1.0 / 6.0);
}

// The corrugation function summed over the cluster's atoms [first, last) (MURII, MURO / VREP1D values); NaN where the
// host stops. An atom beyond the function's reach adds +0 (skipped on the squared distance, with a margin that keeps
// every atom whose rounded distance could be within reach). The atoms are the same for all lanes: scalar loads.
template <bool STAGED>
__device__ __forceinline__ double crp_cluster(const CrpDev& s, const CrpStaged& staged, double x, double y, double z,
                                              int first, int last) {
  const int nc = s.n_corrugation;
  const double reach = s.corrugation[nc - 1], nearest = s.corrugation[0];
  const double reach2 = reach * reach * (1.0 + 1.0e-12);
  double rep = 0.0;
  bool bad = false;
  for (int k = first; k < last; ++k) {
    const double* at = s.cluster + 4 * k;
    const double dx = x - at[0], dy = y - at[1], dz = z - at[2];
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (r2 > reach2) continue;
    const double r = sqrt(r2);
    double vr = 0.0;
    if (!(r > reach)) {
      if (r < nearest) bad = true;
      if constexpr (STAGED)
        vr = crp_staged_splint(staged, r);
      else
        vr = crp_splint(s.corrugation, nc, r);
    }
    rep = rep + vr;
    if (!(r > 0.0) && at[3] != 0.0) bad = true;
  }
  return bad && !s.square ? __builtin_nan("") : rep;
}

// theta = 0, 45, 90, 135 degrees combined
__device__ inline double crp_four(double v0, double v45, double v90, double v135, double c2, double s2, double c4) {
  return 0.2500 * ((v0 + v45 + v90 + v135) + (v0 + v90 - v45 - v135) * c4) +
         0.500 * ((v0 - v90) * c2 + (v45 - v135) * s2);
}

// A site of the hexagonal surfaces (the top site, the bridges, the hollows, the t2 sites): its cuts start at `cut`, its
// azimuth is (phi + offset) - shift, and it needs the sine or cosine of two multiples of that.
struct CrpSite {
  int kind, cut;
  double offset, shift;
  int mid, reversed;
};
constexpr int kCrpTop = 0, kCrpBridge = 1, kCrpHollow = 2, kCrpT2 = 3;
constexpr double kCrpPi = spo::crp_tables::kPi, kCrpPi3 = kCrpPi / 3.00, kCrp2Pi3 = 2.00 * kCrpPi3;
constexpr double kCrpPi6 = kCrpPi / 6.00;
__constant__ CrpSite kCrpSites[2][12] = {
    {{kCrpTop, 0, 0, 0, 0, 0}, {kCrpBridge, 3, 0, 0, 0, 0}, {kCrpHollow, 7, 0, 0, 0, 0}, {kCrpT2, 12, 0, kCrpPi6, 5, 0},
     {kCrpBridge, 3, kCrpPi3, 0, 0, 0}, {kCrpBridge, 3, -kCrpPi3, 0, 0, 0}, {kCrpT2, 12, -kCrp2Pi3, kCrpPi6, 5, 0},
     {kCrpT2, 12, kCrp2Pi3, kCrpPi6, 5, 0}, {kCrpHollow, 7, kCrpPi, 0, 0, 0}, {kCrpT2, 12, kCrpPi, kCrpPi6, 5, 0},
     {kCrpT2, 12, kCrpPi3, kCrpPi6, 5, 0}, {kCrpT2, 12, -kCrpPi3, kCrpPi6, 5, 0}},
    {{kCrpTop, 0, 0, 0, 0, 0}, {kCrpBridge, 3, 0, 0, 0, 0}, {kCrpHollow, 7, 0, 0, 0, 0}, {kCrpT2, 12, 0, kCrpPi6, 4, 0},
     {kCrpBridge, 3, kCrpPi3, 0, 0, 0}, {kCrpBridge, 3, -kCrpPi3, 0, 0, 0}, {kCrpT2, 12, -kCrp2Pi3, kCrpPi6, 4, 0},
     {kCrpT2, 12, kCrp2Pi3, kCrpPi6, 4, 0}, {kCrpHollow, 24, 0, 0, 0, 0}, {kCrpT2, 18, kCrp2Pi3, 11.00 * kCrpPi6, 4, 1},
     {kCrpT2, 18, 0, 11.00 * kCrpPi6, 4, 1}, {kCrpT2, 18, -kCrp2Pi3, 11.00 * kCrpPi6, 4, 1}}};

// cut(k): the site's k-th cut at the point.
template <class Cut>
__device__ inline double crp_site(const CrpSite& site, double phi, double c2t, double s2t, double c4t, Cut&& cut) {
  const double ph = (phi + site.offset) - site.shift;
  const double k1 = site.kind == kCrpT2 ? 1.00 : site.kind == kCrpHollow ? 3.00 : 2.00;
  const double k2 = site.kind == kCrpT2 ? 2.00 : site.kind == kCrpBridge ? 4.00 : 6.00;
  const double t1 = site.kind == kCrpTop ? 0.0 : site.kind == kCrpHollow ? sin(k1 * ph) : cos(k1 * ph);
  const double t2 = cos(k2 * ph);
  const double c0 = cut(0), c1 = cut(1), c2 = cut(2);
  if (site.kind == kCrpTop) {
    const double v90 = 0.500 * ((c1 + c2) + (c1 - c2) * t2);
    return 0.500 * ((c0 + v90) + (c0 - v90) * c2t);
  }
  if (site.kind == kCrpBridge) {
    constexpr double u3 = 1.00 / 3.00;
    const double c3 = cut(3);
    const double v90 =
        (c1 + 2.00 * c2) * u3 - 0.500 * (c3 - c1) * t1 + (0.500 * (c3 - c1) - 2.00 * (c2 - c1) * u3) * t2;
    return 0.500 * (c0 * (1.00 + c2t) + v90 * (1.00 - c2t));
  }
  if (site.kind == kCrpHollow) {
    const double c3 = cut(3), c4 = cut(4);
    const double v45 = 0.500 * ((c3 + c4) + (c3 - c4) * t1);
    const double v135 = 0.500 * ((c3 + c4) - (c3 - c4) * t1);
    const double v90 = 0.500 * ((c1 + c2) + (c1 - c2) * t2);
    return crp_four(c0, v45, v90, v135, c2t, s2t, c4t);
  }
  // 45 cuts g, m, k around the middle one, 90 cuts c1, c2
  const double g = cut(3), k = cut(site.mid == 5 ? 4 : 5), m = cut(site.mid);
  const double odd = site.reversed ? (-g + k) : (g - k);
  const double v45 = 0.2500 * ((g + 2.00 * m + k) + (g - 2.00 * m + k) * t2) + 0.500 * odd * t1;
  const double v135 = 0.2500 * ((g + 2.00 * m + k) + (g - 2.00 * m + k) * t2) - 0.500 * odd * t1;
  const double v90 =
      site.reversed ? 0.500 * ((c1 + c2) + (-c1 + c2) * t2) : 0.500 * ((c1 + c2) + (c1 - c2) * t2);
  return crp_four(c0, v45, v90, v135, c2t, s2t, c4t);
}

// The 8 sites of C4v (RRINT): 0 and 3 top, 1 and 2 bridge (phi, phi + 90), 4 to 7 t2h (phi, -90, -180, +90).
template <class Cut>
__device__ inline double crp_site_square(int site, double phi, double c2t, double s2t, double c4t, Cut&& cut) {
  using spo::crp_tables::kPi;
  if (site == 0 || site == 3) {
    const int o = site == 0 ? 0 : 7;
    const double v90 = 0.5 * (cut(o + 1) + cut(o + 2)) + 0.5 * (cut(o + 1) - cut(o + 2)) * cos(4.0 * phi);
    return 0.5 * (cut(o) + v90) + 0.5 * (cut(o) - v90) * c2t;
  }
  if (site < 3) {
    const double ph = site == 1 ? phi : phi + kPi / 2.0;
    const double c1 = cut(4), c2 = cut(5), c3 = cut(6);
    const double v90 = (0.25 * c1 + 0.5 * c2 + 0.25 * c3) + 0.5 * (c1 - c3) * cos(2.0 * ph) +
                       (0.25 * c1 - 0.5 * c2 + 0.25 * c3) * cos(4.0 * ph);
    return 0.5 * (cut(3) + v90) + 0.5 * (cut(3) - v90) * c2t;
  }
  const double ph = site == 4 ? phi : site == 5 ? phi - kPi / 2.0 : site == 6 ? phi - kPi : phi + kPi / 2.0;
  const double p45 = ph - kPi / 4.0, p135 = ph + kPi - kPi / 4.0;
  const double c0 = cut(10), c1 = cut(11), c2 = cut(12), c3 = cut(13), c4 = cut(14), c5 = cut(15);
  const double cc0 = 0.25 * (c1 + c2 - 2.0 * c5);
  const double b0 = -c5 + c2 - 2.0 * cc0;
  const double a0 = c2 - b0 - cc0;
  const double v45 = a0 + b0 * cos(p45) + cc0 * cos(2.0 * p45);
  const double v135 = a0 + b0 * cos(p135) + cc0 * cos(2.0 * p135);
  const double v90 = 0.5 * (c3 + c4) + 0.5 * (c3 - c4) * cos(2.0 * p45);
  return 0.25 * (c0 + v45 + v90 + v135) + 0.5 * (c0 - v90) * c2t + 0.5 * (v45 - v135) * s2t +
         0.25 * (c0 + v90 - v45 - v135) * c4t;
}

// Fourier terms: a sum of `count` sines or cosines of scale (m p + n q) from kCrpAngles[first] on. Those of the two
// atoms (FOUR3II, without its first, 1; a C3v surface has the sines too), then the molecule's (FOUR6II, likewise).
struct CrpTerm {
  int first, count, sine;
};
struct CrpAngle {
  double m, n, scale, sign;
};
__constant__ CrpAngle kCrpAngles[] = {
    {1, 0, 1, 1}, {0, 1, 1, 1}, {1, 1, 1, 1},                                                     // 0
    {1, 0, 1, -1}, {0, 1, 1, -1}, {1, 1, 1, 1},                                                   // 3
    {2, 1, 1, 1}, {1, 2, 1, 1}, {1, -1, 1, 1},                                                    // 6
    {2, 0, 1, 1}, {0, 2, 1, 1}, {2, 2, 1, 1},                                                     // 9
    {2, 0, 1, -1}, {0, 2, 1, -1}, {2, 2, 1, 1},                                                   // 12
    {3, 1, 1, 1}, {1, 3, 1, 1}, {2, 3, 1, 1}, {3, 2, 1, 1}, {-1, 2, 1, 1}, {2, -1, 1, 1},         // 15
    {3, 1, 1, -1}, {1, 3, 1, -1}, {2, 3, 1, 1}, {3, 2, 1, 1}, {-1, 2, 1, -1}, {2, -1, 1, -1},     // 21
    {3, 0, 1, 1}, {0, 3, 1, 1}, {1, 1, 3, 1},                                                     // 27
    {4, 2, 1, 1}, {2, 4, 1, 1}, {2, -2, 1, 1}};                                                   // 30
__constant__ CrpTerm kCrpAtomTerms[2][9] = {
    {{0, 3, 0}, {6, 3, 0}, {9, 3, 0}, {15, 6, 0}, {27, 3, 0}, {30, 3, 0}},
    {{0, 3, 0}, {3, 3, 1}, {6, 3, 0}, {9, 3, 0}, {12, 3, 1}, {15, 6, 0}, {21, 6, 1}, {27, 3, 0}, {30, 3, 0}}};
__constant__ CrpTerm kCrpMoleculeTerms[11] = {{0, 1, 0}, {1, 1, 0}, {2, 1, 0}, {0, 1, 1}, {1, 1, 1}, {2, 1, 1},
                                              {6, 1, 0}, {7, 1, 0}, {8, 1, 0}, {9, 3, 0}, {12, 3, 1}};

__device__ inline double crp_fourier(const CrpTerm& term, double p, double q) {
  double sum = 0.0;
  for (int j = 0; j < term.count; ++j) {
    const CrpAngle& g = kCrpAngles[term.first + j];
    const double angle = g.scale * (g.m * p + g.n * q);
    sum = sum + g.sign * (term.sine ? sin(angle) : cos(angle));
  }
  return sum;
}

// The SCM correction (spo_hip_scm_correction): the pair functions of the slab's top two layers
// (src/potential/scm/scm_correction.cpp; Fortran SCM_Potential.f90), the same operand order as host/scm.cpp.
struct ScmDev {
  int on, rescale;
  double scale, cos_skew, sin_skew;
  double layers[2][18];
  int n_atoms;
  const double* atoms;
};

// -(p3 + q (p4 + q (p5 + q p6))) exp(-p2 q); t = p1..p8, C
__device__ inline double scm_unswitched(const double* t, double q) {
  const double cubic = t[2] + q * (t[3] + q * (t[4] + q * t[5]));
  return -(cubic * exp(-(t[1] * q)));
}

__device__ inline void scm_terms(const double* layer, double r, double* t) {
  double c = r;
  if (r < layer[16]) {
    c = layer[16];
  } else if (r > layer[17]) {
    c = layer[17];
  }
  for (int k = 0; k < 8; ++k) t[k] = layer[8 + k] * c + layer[k];
  t[8] = scm_unswitched(t, t[7] - t[0]);
}

__device__ inline double scm_pair(const double* t, double d) {
  if (d > t[7]) return t[8];
  const double f = scm_unswitched(t, d - t[0]);
  if (!(d > t[6])) return f;
  const double phase = ((d - t[7]) * spo::crp_tables::kPi) / (t[7] - t[6]);
  const double rho = 0.5 * cos(phase) + 0.5;
  return (1.0 - rho) * f + rho * t[8];
}

__device__ inline double scm_distance(const double* a, const double* b) {
  const double dx = a[0] - b[0], dy = a[1] - b[1], dz = a[2] - b[2];
  return sqrt((dx * dx + dy * dy) + dz * dz);
}

// The sums over the cluster (both atoms') and over the slab's atoms are made in this many runs of consecutive terms,
// whatever the number of wavefronts that share them: a point's value does not depend on the launch it is part of.
constexpr int kCrpParts = 16;

// The pair terms of the slab's atoms (hartree) with the molecule's centre at the Cartesian (x, y), z: the sums of the
// atoms [first, mid), to `head`, and [mid, last), returned. TWO: whether the first are asked for (else mid = first).
template <bool TWO>
__device__ inline double scm_pairs(const ScmDev& m, double x, double y, double z, double r, double st, double ct,
                                   double sp, double cp, int first, int mid, int last, double& head) {
  const double h = 0.5 * r;
  const double o[3] = {(h * st) * cp, (h * st) * sp, h * ct};
  double hd[2][3] = {{x - o[0], y - o[1], z - o[2]}, {x + o[0], y + o[1], z + o[2]}};
  double hi[2][3];
  if (m.rescale) {
    const double bond[3] = {hd[1][0] - hd[0][0], hd[1][1] - hd[0][1], hd[1][2] - hd[0][2]};
    const double c[3] = {((hd[0][0] + hd[1][0]) / 2.0) / m.scale, ((hd[0][1] + hd[1][1]) / 2.0) / m.scale,
                         (hd[0][2] + hd[1][2]) / 2.0};
    for (int k = 0; k < 3; ++k) {
      hi[0][k] = c[k] - 0.5 * bond[k];
      hi[1][k] = c[k] + 0.5 * bond[k];
    }
  } else {
    for (int k = 0; k < 3; ++k) {
      hi[0][k] = hd[0][k];
      hi[1][k] = hd[1][k];
    }
  }
  double t[2][9];
  scm_terms(m.layers[0], r, t[0]);
  scm_terms(m.layers[1], r, t[1]);
  double dv = +0.0;
  auto atom = [&](const double* tl, const double* at) {
    for (int a = 0; a < 2; ++a) {
      const double f_ideal = scm_pair(tl, scm_distance(hi[a], at + 3));
      const double f_distorted = scm_pair(tl, scm_distance(hd[a], at));
      dv = (dv - f_ideal) + f_distorted;
    }
  };
  for (int i = first; i < last; ++i) {
    if (TWO && i == mid) {
      head = dv;
      dv = +0.0;
    }
    const double* at = m.atoms + 7 * i;
    if (at[6] == 1.0)
      atom(t[0], at);
    else
      atom(t[1], at);
  }
  if (TWO && mid == last) {
    head = dv;
    dv = +0.0;
  }
  return dv;
}

// A workgroup's exchange in LDS: slots of 64 doubles, a lane's point in each.
constexpr int kCrpWaves = 8, kCrpWavesFew = 16;  // wavefronts of a workgroup; of one where there are few
enum CrpSlot {
  kCrpA,                            // the atoms' positions
  kCrpB = kCrpA + 3,
  kCrpR = kCrpB + 3,                // their distance
  kCrpPhi, kCrpC2, kCrpS2, kCrpC4,  // the molecule's azimuth; cos 2 theta, sin 2 theta, cos 4 theta
  kCrpRep,                          // the cluster sums, the atoms' in turn
  kCrpDv = kCrpRep + kCrpParts,     // the slab sums
  kCrpCv = kCrpDv + kCrpParts,      // the molecular cuts
  kCrpVs = kCrpCv + 29,             // the atom splines, 10 an atom (C4v: the cell's spline, the first of each)
  kCrpF = kCrpVs + 20,              // the atoms' Fourier terms, 9 an atom
  kCrpFb = kCrpF + 18,              // the molecule's
  kCrpSiteV = kCrpFb + 11,          // the sites; before them the geometry as given:
  kCrpU = kCrpSiteV, kCrpV, kCrpZ, kCrpRGiven, kCrpSt, kCrpCt, kCrpSp, kCrpCp,
  kCrpIv = kCrpSiteV + 12,          // the interpolated interaction, the atoms' potentials
  kCrpVa = kCrpIv + 1,
  kCrpSlots = kCrpVa + 2
};
// Bytes of LDS, `staged` doubles of them for the corrugation function.
constexpr std::size_t crp_lds(int staged) { return (64 * kCrpSlots + staged) * sizeof(double) + 64 * sizeof(int); }
// Two workgroups fit on a CU with a table of this many doubles; a longer one is read from memory.
constexpr int kCrpStagedMax = 1496;

// V in eV at the points of a workgroup's lanes, returned to the first wavefront: the QD wrapper, the molecule-surface V
// (POT6D value statements) and the SCM correction. point(p) writes u, v (skewed), Z, r, theta, phi of the lane's point;
// only the first wavefront calls it. NaN where the host stops.
template <int WAVES, bool STAGED, class Point>
__device__ __forceinline__ double crp_scm_block(const CrpDev& s, const ScmDev& m, Point&& point) {
  using namespace spo::crp_tables;
  extern __shared__ double crp_smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double* const slots = crp_smem + lane;
  int* const silent = reinterpret_cast<int*>(crp_smem + 64 * kCrpSlots) + lane;
  double* const table = crp_smem + 64 * kCrpSlots + 32;
  auto slot = [&](int k) -> double& { return slots[64 * k]; };
  constexpr double ev = 27.2113961;  // the CRP library's hartree in eV (to_energy: x * (1.0 * 27.2113961))

  // The geometry, by the first wavefront; the others bring the corrugation function in.
  if (wave == 0) {
    constexpr double delta = 1.0e-12;
    double g[6];
    point(g);
    const double u = m.on ? g[0] / m.scale : g[0], v = m.on ? g[1] / m.scale : g[1];
    double rr = g[3], zz = g[2];
    if (rr < s.r_min + delta) {
      rr = s.r_min + delta;
    } else if (rr > s.r_max - delta) {
      rr = s.r_max - delta;
    }
    if (zz < s.z_min + delta) zz = s.z_min + delta;
    // [[1, cos g], [0, sin g]] (u, v); cos(pi/2) as gfortran folds it for C4v
    const double cg = s.square ? 0x1.1a62633145c07p-54 : kCosPi3, sg = s.square ? 1.0 : kSinPi3;
    const double x = 1.0 * u + cg * v;
    const double y = 0.0 * u + sg * v;
    const double st = sin(g[4]), ctt = cos(g[4]), cph = cos(g[5]), sph = sin(g[5]);
    const double a[3] = {x - 0.5 * rr * st * cph, y - 0.5 * rr * st * sph, zz - 0.5 * rr * ctt};
    const double b[3] = {x + 0.5 * rr * st * cph, y + 0.5 * rr * st * sph, zz + 0.5 * rr * ctt};
    for (int k = 0; k < 3; ++k) {
      slot(kCrpA + k) = a[k];
      slot(kCrpB + k) = b[k];
    }
    slot(kCrpR) = sqrt((b[0] - a[0]) * (b[0] - a[0]) + (b[1] - a[1]) * (b[1] - a[1]) + (b[2] - a[2]) * (b[2] - a[2]));
    slot(kCrpU) = g[0];
    slot(kCrpV) = g[1];
    slot(kCrpZ) = g[2];
    slot(kCrpRGiven) = g[3];
    slot(kCrpSt) = st;
    slot(kCrpCt) = ctt;
    slot(kCrpSp) = sph;
    slot(kCrpCp) = cph;
    *silent = 0;
  } else if constexpr (STAGED) {
    const int n = s.n_corrugation, size = crp_staged_size(n);
    for (int k = threadIdx.x - 64; k < size; k += 64 * (WAVES - 1))
      table[k] = k < n - 1 ? s.corrugation[k] : __builtin_inf();
    for (int k = threadIdx.x - 64; k < n - 1; k += 64 * (WAVES - 1)) {
      const double* x = s.corrugation + k;
      double* i = table + size + 7 * k;
      i[0] = x[0];
      i[1] = x[1];
      i[2] = x[n];
      i[3] = x[n + 1];
      i[4] = x[2 * n];
      i[5] = x[2 * n + 1];
      i[6] = 1.0 / (x[1] - x[0]);
    }
  }
  __syncthreads();

  // The slab's pair terms: each wavefront's parts of its atoms.
  constexpr int kOwn = kCrpParts / WAVES;  // parts of a wavefront
  static_assert(kOwn == 1 || kOwn == 2);
  if (m.on) {
    auto start = [&](int part) { return part * m.n_atoms / kCrpParts; };
    double head = 0.0;
    slot(kCrpDv + kOwn * wave + kOwn - 1) = scm_pairs<kOwn == 2>(
        m, slot(kCrpU) + m.cos_skew * slot(kCrpV), m.sin_skew * slot(kCrpV), slot(kCrpZ), slot(kCrpRGiven), slot(kCrpSt),
        slot(kCrpCt), slot(kCrpSp), slot(kCrpCp), start(kOwn * wave), start(kOwn * wave + kOwn - 1),
        start(kOwn * wave + kOwn), head);
    if (kOwn == 2) slot(kCrpDv + kOwn * wave) = head;
  }

  // Set up only now: the slab's sums need every register.
  const CrpStaged staged{table, table + crp_staged_size(s.n_corrugation), crp_staged_size(s.n_corrugation),
                         s.n_corrugation - 2};
  const double r = slot(kCrpR);
  const double gx = slot(kCrpA) * (1.0 - 0.500) + slot(kCrpB) * 0.500;
  const double gy = slot(kCrpA + 1) * (1.0 - 0.500) + slot(kCrpB + 1) * 0.500;
  const double gz = slot(kCrpA + 2) * (1.0 - 0.500) + slot(kCrpB + 2) * 0.500;
  const bool gas_phase = !(gz < s.zso_max);  // the gas-phase potential alone
  const double fac = 2.00 * kPi / s.a;

  // The surface itself, unless every point is in the gas phase (the wavefronts hold the same points and agree).
  if (__builtin_amdgcn_ballot_w64(!gas_phase) != 0) {
    // Sums over pairs: each wavefront takes one of the atoms and its parts of the cluster.
    {
      const int h = wave & 1;
      const double px = slot(kCrpA + 3 * h), py = slot(kCrpA + 3 * h + 1), pz = slot(kCrpA + 3 * h + 2);
      double x = 0.0, y = 0.0;
      const bool in_reach = !gas_phase && !(s.square && pz >= s.cell[10 + s.cell_nz - 1]);
      const bool folded = in_reach && crp_fold(s, px, py, x, y);
#pragma unroll 1
      for (int k = 0; k < kOwn; ++k) {
        const int part = kOwn * (wave >> 1) + k;
        double rep = 0.0;
        if (in_reach)
          rep = folded ? crp_cluster<STAGED>(s, staged, x, y, pz, 2 * part * s.n_cluster / kCrpParts,
                                             2 * (part + 1) * s.n_cluster / kCrpParts)
                       : __builtin_nan("");
        slot(kCrpRep + 2 * part + h) = rep;
      }
    }
    // The cuts at (r, Z); one cell lookup per group of cuts on the same grid.
    {
      int group = -1, ci = 0, cj = 0;
      double wxa = 0, wxb = 0, wxc = 0, wxd = 0, wya = 0, wyb = 0, wyc = 0, wyd = 0;
      for (int k = wave; k < s.n_cuts; k += WAVES) {
        const int nr = s.cut_shape[3 * k], nzc = s.cut_shape[3 * k + 1], g = s.cut_shape[3 * k + 2];
        const double* blk = s.cut_data + s.cut_offsets[k];
        const double* xr = blk;
        const double* yz = blk + nr;
        if (g != group) {
          if (r < xr[0] || r > xr[nr - 1] || gz < yz[0] || gz > yz[nzc - 1]) {
            if (!gas_phase) *silent = 1;
          }
          group = g;
          ci = crp_bisect(xr, nr, r);
          cj = crp_bisect(yz, nzc, gz);
          const double hx = (xr[ci + 1] - xr[ci]) * (xr[ci + 1] - xr[ci]) / 6.0;
          wxa = (xr[ci + 1] - r) / (xr[ci + 1] - xr[ci]);
          wxb = 1.0 - wxa;
          wxc = (wxa * wxa * wxa - wxa) * hx;
          wxd = (wxb * wxb * wxb - wxb) * hx;
          const double hy = (yz[cj + 1] - yz[cj]) * (yz[cj + 1] - yz[cj]) / 6.0;
          wya = (yz[cj + 1] - gz) / (yz[cj + 1] - yz[cj]);
          wyb = 1.0 - wya;
          wyc = (wya * wya * wya - wya) * hy;
          wyd = (wyb * wyb * wyb - wyb) * hy;
        }
        const long plane = static_cast<long>(nr) * nzc;
        const double* f = blk + nr + nzc;
        const double* fxx = f + plane;
        const double* fyy = fxx + plane;
        const double* fxxyy = fyy + plane;
        const long p00 = ci + static_cast<long>(nr) * cj, p10 = p00 + 1, p01 = p00 + nr, p11 = p01 + 1;
        slot(kCrpCv + k) = wxa * (wya * f[p00] + wyb * f[p01] + wyc * fyy[p00] + wyd * fyy[p01]) +
                           wxb * (wya * f[p10] + wyb * f[p11] + wyc * fyy[p10] + wyd * fyy[p11]) +
                           wxc * (wya * fxx[p00] + wyb * fxx[p01] + wyc * fxxyy[p00] + wyd * fxxyy[p01]) +
                           wxd * (wya * fxx[p10] + wyb * fxx[p11] + wyc * fxxyy[p10] + wyd * fxxyy[p11]);
      }
    }
    if (wave == 0) {
      const double a[3] = {slot(kCrpA), slot(kCrpA + 1), slot(kCrpA + 2)};
      double ct = (slot(kCrpB + 2) - a[2]) / r;
      if (ct > 1.0) ct = 1.0;
      const double theta = acos(ct);
      const double ddx = slot(kCrpB) - a[0], ddy = slot(kCrpB + 1) - a[1];
      slot(kCrpPhi) = (ddx == 0.0 && ddy == 0.0) ? 0.0 : atan2(ddy, ddx);
      slot(kCrpC2) = cos(2.00 * theta);
      slot(kCrpS2) = sin(2.00 * theta);
      slot(kCrpC4) = cos(4.00 * theta);
    }
    if (s.square) {
      if (wave < 2) {
        const double px = slot(kCrpA + 3 * wave), py = slot(kCrpA + 3 * wave + 1), pz = slot(kCrpA + 3 * wave + 2);
        double x = 0.0, y = 0.0, cell = 0.0;  // 0 above the data
        if (!(pz >= s.cell[10 + s.cell_nz - 1]))
          cell = crp_fold(s, px, py, x, y) ? crp_cell(s, x, y, pz) : __builtin_nan("");
        slot(kCrpVs + 10 * wave) = cell;
      }
    } else {
      // The atom splines and Fourier terms, and the molecule's Fourier terms, in turn.
      const int n_terms = s.n_basis - 1;
      for (int k = wave; k < 2 * s.n_basis; k += WAVES) {
        const int h = k >= s.n_basis ? 1 : 0, i = k - h * s.n_basis;
        const int off = s.atom_offsets[i], n = s.atom_offsets[i + 1] - off;
        const double pz = slot(kCrpA + 3 * h + 2);
        double v = crp_dpl(s.atom_splines + 3 * off, n, pz);
        // z within the first site's data
        if (i == 0 && (pz < s.atom_splines[0] || pz > s.atom_splines[n - 1])) v = __builtin_nan("");
        slot(kCrpVs + 10 * h + i) = v;
      }
      for (int k = wave; k < 2 * n_terms + 11; k += WAVES) {
        const bool molecule = k >= 2 * n_terms;
        const int h = k >= n_terms ? 1 : 0;
        const double x = molecule ? gx : slot(kCrpA + 3 * h), y = molecule ? gy : slot(kCrpA + 3 * h + 1);
        const double p = fac * (x - y * kUsq3), q = fac * (2.00 * y * kUsq3);
        if (molecule)
          slot(kCrpFb + k - 2 * n_terms) = crp_fourier(kCrpMoleculeTerms[k - 2 * n_terms], p, q);
        else
          slot(kCrpF + 9 * h + k - h * n_terms) = crp_fourier(kCrpAtomTerms[s.c3v ? 1 : 0][k - h * n_terms], p, q);
      }
    }
    __syncthreads();

    // The sites (RRINTII, RRINT).
    {
      const double phi = slot(kCrpPhi), c2t = slot(kCrpC2), s2t = slot(kCrpS2), c4t = slot(kCrpC4);
      for (int k = wave; k < (s.square ? 8 : 12); k += WAVES) {
        if (s.square) {
          slot(kCrpSiteV + k) = crp_site_square(k, phi, c2t, s2t, c4t, [&](int c) { return slot(kCrpCv + c); });
        } else {
          const CrpSite& site = kCrpSites[s.c3v ? 1 : 0][k];
          slot(kCrpSiteV + k) = crp_site(site, phi, c2t, s2t, c4t, [&](int c) { return slot(kCrpCv + site.cut + c); });
        }
      }
    }
    __syncthreads();

    if (wave == 0) {
      double iv = 0.00;
      if (s.square) {  // SIS8x8
        const double p1 = slot(kCrpSiteV), p2 = slot(kCrpSiteV + 1), p5 = slot(kCrpSiteV + 2), p3 = slot(kCrpSiteV + 3);
        const double p4 = slot(kCrpSiteV + 4), p6 = slot(kCrpSiteV + 5), p7 = slot(kCrpSiteV + 6);
        const double p8 = slot(kCrpSiteV + 7);
        iv = 1.0 / 8.0 * (p1 + p2 + p5 + p3 + p4 + p6 + p7 + p8) * 1.0 +
             1.0 / 4.0 * (p1 - p2 + p5 - p3) * cos(fac * gx) + 1.0 / 4.0 * (p1 + p2 - p5 - p3) * cos(fac * gy) +
             1.0 / 4.0 * (p4 - p6 - p7 + p8) * sin(fac * gx) + 1.0 / 4.0 * (p4 + p6 - p7 - p8) * sin(fac * gy) +
             1.0 / 8.0 * (p1 - p2 - p5 + p3 - p4 + p6 - p7 + p8) * cos(fac * (gx + gy)) +
             1.0 / 8.0 * (p1 - p2 - p5 + p3 + p4 - p6 + p7 - p8) * cos(fac * (gx - gy)) +
             1.0 / 16.0 * (p1 + p2 + p5 + p3 - p4 - p6 - p7 - p8) * (cos(fac * (2.0 * gx)) + cos(fac * (2.0 * gy)));
      } else {  // SISII, FOUR6II
        for (int j = 0; j < 12; ++j) {
          double c = 0.00;
          for (int k = 0; k < 12; ++k) c = c + kCrpMolecule[k + 12 * j] * slot(kCrpSiteV + k);
          iv = iv + c * (j == 0 ? 1.00 : slot(kCrpFb + j - 1));
        }
      }
      slot(kCrpIv) = iv;
    } else if (wave < 3) {
      // An atom's potential (ATII): the Fourier interpolation of the reduced cuts, and the cluster's sum.
      const int h = wave - 1;
      double v = 0.00;
      if (s.square) {
        v = slot(kCrpVs + 10 * h);
      } else {
        const double* coefficients = s.c3v ? kCrpAtomC3v.data() : kCrpAtomC6v.data();
        for (int j = 0; j < s.n_basis; ++j) {
          double a = 0.00;
          for (int i = 0; i < s.n_basis; ++i) a = a + coefficients[i + s.n_basis * j] * slot(kCrpVs + 10 * h + i);
          v = v + a * (j == 0 ? 1.00 : slot(kCrpF + 9 * h + j - 1));
        }
      }
      double rep = slot(kCrpRep + h);
      for (int part = 1; part < kCrpParts / 2; ++part) rep = rep + slot(kCrpRep + 2 * part + h);
      slot(kCrpVa + h) = v + rep;
    }
  }
  __syncthreads();
  if (wave != 0) return 0.0;

  const int nh = s.n_h2, nz = s.n_zdep;
  double v;
  auto gas = [&] {
    const double v1 = gz <= s.zdep[nz - 1] ? crp_splint(s.zdep, nz, gz) : s.zdep[2 * nz - 1];
    return crp_splint(s.h2, nh, r) + v1;
  };
  if (r == 0.0) {
    v = __builtin_nan("");
  } else if (gas_phase) {
    v = r < s.h2[0] || r > s.h2[nh - 1] ? 0.00 : gas();  // 0: outside the data, without an error as there
  } else if (*silent) {
    v = 0.00;
  } else {
    v = slot(kCrpVa) + slot(kCrpVa + 1) + slot(kCrpIv);
    if (!(gz <= s.zso_min)) {
      const double sw = 0.500 + 0.500 * cos((gz - s.zso_min) * kPi / (s.zso_max - s.zso_min));
      v = v * sw + (1.00 - sw) * gas();
    }
  }
  v = v * (1.0 * ev) - s.h2_asymptote * (1.0 * ev);
  if (m.on) {
    double dv = slot(kCrpDv);
    for (int k = 1; k < kCrpParts; ++k) dv = dv + slot(kCrpDv + k);
    v = v + dv / 0.036749308286;
  }
  return v;
}

// V at the points (u, v, Z, r, theta, phi) from `first` on, n in all, 64 a workgroup. Two workgroups of 8 wavefronts
// share a CU, one waiting while the other works; up to a workgroup a CU, 16 wavefronts shorten the chain instead.
// 1000 points 43 us with 16 wavefronts and 60 with 8; 300 007 with the slab 1.10 ms and 0.81.
template <int WAVES, bool STAGED>
__global__ __launch_bounds__(64 * WAVES, 4) void crp_points_kernel(long first, long n, CrpDev s, ScmDev m,
                                                                       const double* points, double* values) {
  const long i = first + static_cast<long>(blockIdx.x) * 64 + (threadIdx.x & 63);
  const double v = crp_scm_block<WAVES, STAGED>(s, m, [&](double* g) {
    const double* p = points + 6 * (i < n ? i : n - 1);
    for (int k = 0; k < 6; ++k) g[k] = p[k];
  });
  if (threadIdx.x < 64 && i < n) values[i] = v;
}

}  // namespace spo_dev

#pragma clang fp contract(on)
