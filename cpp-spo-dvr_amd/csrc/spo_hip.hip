// The MI355X propagation backend behind the C ABI of include/spo_hip.h: device buffers, FFT plans and the launch
// sequence of one analysis step. Kernels: kernels_ct.hpp (compile-time shapes) and kernels.hpp (any shape); LDS
// FFT engines: fft_ct.hpp, fft_lds.hpp.
//
// The scattering wave and the tables it is multiplied with are stored in T (double, or float in the mixed mode;
// the factors are built in FP64 on the host and rounded once). The specular wave, the projection onto it, the
// Balint-Kurti coefficients and the S-matrix sums are FP64 in both modes.
#include <hip/hip_runtime.h>


#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <optional>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/spo_hip.h"
#include "kernels_ct.hpp"
#include "kernels_mfma.hpp"
#include "kernels_zr.hpp"
#include "variants.hpp"
#include "kernels_pes.hpp"
#include "kernels_mlp.hpp"

using spo_dev::cx;
using spo_dev::Variant;

namespace {

thread_local std::string g_error;

struct Status : std::runtime_error {
  int code;
  Status(int c, const std::string& what) : std::runtime_error(what), code(c) {}
};

void check(hipError_t e, const char* what) {
  if (e != hipSuccess) throw Status(SPO_HIP_E_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
}
#define HIP_CHECK(call) check((call), #call)

template <typename F>
int guarded(F&& f) {
  try {
    f();
    return SPO_HIP_OK;
  } catch (const Status& s) {
    g_error = s.what();
    return s.code;
  } catch (const std::exception& e) {
    g_error = e.what();
    return SPO_HIP_E_DEVICE;
  }
}

// Device memory owned by the backend.
class Buffer {
 public:
  Buffer() = default;
  explicit Buffer(std::size_t bytes) : bytes_(bytes) {
    if (bytes) HIP_CHECK(hipMalloc(&ptr_, bytes));
  }
  Buffer(const Buffer&) = delete;
  Buffer& operator=(const Buffer&) = delete;
  Buffer(Buffer&& o) noexcept : ptr_(o.ptr_), bytes_(o.bytes_) {
    o.ptr_ = nullptr;
    o.bytes_ = 0;
  }
  Buffer& operator=(Buffer&& o) noexcept {
    std::swap(ptr_, o.ptr_);
    std::swap(bytes_, o.bytes_);
    return *this;
  }
  ~Buffer() {
    if (ptr_) (void)hipFree(ptr_);
  }
  template <typename T>
  T* as() const { return static_cast<T*>(ptr_); }

 private:
  void* ptr_ = nullptr;
  std::size_t bytes_ = 0;
};

void require_device() {
  int devices = 0;
  if (hipGetDeviceCount(&devices) != hipSuccess || devices < 1)
    throw Status(SPO_HIP_E_NOT_SUPPORTED, "no HIP device is visible");
}

Buffer upload(const void* host, std::size_t bytes) {
  Buffer b(bytes);
  if (bytes) HIP_CHECK(hipMemcpy(b.as<void>(), host, bytes, hipMemcpyHostToDevice));
  return b;
}

// A complex factor in the storage type: FP64 as is; complex64 rounded to nearest (tables applied at every step
// also carry the remainder, factor_lo, or for twiddles a modulus correction, DevicePlan::eps).
template <typename T>
cx<T> to_storage(double x, double y) {
  if constexpr (sizeof(T) == 8) {
    return {x, y};
  } else {
    return {static_cast<float>(x), static_cast<float>(y)};
  }
}

// Complex array (interleaved doubles) -> device array of cx<T>, optionally times a real factor (in FP64 first).
// Large complex64 tables (exp(i A)) are rounded on the device.
template <typename T>
Buffer upload_complex(const double* p, std::size_t n, double factor = 1.0) {
  if (sizeof(T) == 4 && n > (std::size_t(1) << 18)) {
    Buffer full = upload(p, n * sizeof(cx<double>));
    Buffer out(n * sizeof(cx<T>));
    hipLaunchKernelGGL(spo_dev::round_to_complex64_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256),
                       0, nullptr, full.as<const double>(), out.as<float>(), static_cast<long>(n), factor);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(nullptr));
    return out;
  }
  std::vector<cx<T>> v(n);
  for (std::size_t i = 0; i < n; ++i) v[i] = to_storage<T>(p[2 * i] * factor, p[2 * i + 1] * factor);
  return upload(v.data(), n * sizeof(cx<T>));
}
// complex64: per entry of a factor table uploaded by upload_complex, the FP32 remainder z - stored z (z the FP64
// value times factor); the kernels multiply by stored z + remainder (mul_hilo). Empty in FP64.
template <typename T>
Buffer factor_lo(const double* p, std::size_t n, double factor = 1.0) {
  if constexpr (sizeof(T) == 8) {
    return Buffer();
  } else {
    std::vector<cx<float>> lo(n);
    for (std::size_t i = 0; i < n; ++i) {
      const double x = p[2 * i] * factor, y = p[2 * i + 1] * factor;
      const cx<float> w = to_storage<float>(x, y);
      lo[i] = {static_cast<float>(x - static_cast<double>(w.x)), static_cast<float>(y - static_cast<double>(w.y))};
    }
    return upload(lo.data(), n * sizeof(cx<float>));
  }
}

// The two entries (lane parity 0 and 1) of the sign-split rotation table for the factor x + i y.
template <typename T>
void set_rot_entries(spo_dev::RotEntry<T>* e, double x, double y) {
  const cx<T> w = to_storage<T>(x, y);
  e[0].x = w.x;
  e[0].y = -w.y;
  e[1].x = w.x;
  e[1].y = w.y;
  if constexpr (sizeof(T) == 4) {
    const float lo_x = static_cast<float>(x - static_cast<double>(w.x));
    const float lo_y = static_cast<float>(y - static_cast<double>(w.y));
    e[0].lo_x = lo_x;
    e[0].lo_y = -lo_y;
    e[1].lo_x = lo_x;
    e[1].lo_y = lo_y;
  }
}

template <typename T>
Buffer upload_real(const double* p, std::size_t n) {
  std::vector<T> v(p, p + n);
  return upload(v.data(), n * sizeof(T));
}

// Radices of the run-time engine: 8 while it divides, then 4, 2, 3, 5, 7, 11.
std::vector<int> radices_of(int n) {
  std::vector<int> r;
  int m = n;
  for (int p : {8, 4, 2, 3, 5, 7, 11})
    while (m % p == 0) {
      r.push_back(p);
      m /= p;
    }
  if (m != 1) throw Status(SPO_HIP_E_NOT_SUPPORTED, "FFT length " + std::to_string(n) + " has a prime factor above 11");
  if (r.size() > 12) throw Status(SPO_HIP_E_NOT_SUPPORTED, "FFT length " + std::to_string(n) + " has too many factors");
  return r;
}

// An FFT length: twiddle table W[m] = exp(-2 pi i m / n) on the device (in T) and the run-time plan.
template <typename T>
struct DevicePlan {
  Buffer table, eps;
  spo_dev::FftPlan plan{};
  explicit DevicePlan(int n) {
    const std::vector<int> r = radices_of(n);
    std::vector<cx<T>> w(n);
    std::vector<T> e(n, T(0));
    for (int m = 0; m < n; ++m) {
      const long double a = -2.0L * 3.14159265358979323846264338327950288L * m / n;
      w[m] = to_storage<T>(static_cast<double>(std::cos(a)), static_cast<double>(std::sin(a)));
      // complex64: the correction that makes the product's modulus exact (twiddle(), kernels_ct.hpp)
      const double m2 = static_cast<double>(w[m].x) * w[m].x + static_cast<double>(w[m].y) * w[m].y;
      e[m] = static_cast<T>(1.0 / std::sqrt(m2) - 1.0);
    }
    table = upload(w.data(), w.size() * sizeof(cx<T>));
    eps = upload(e.data(), e.size() * sizeof(T));
    plan.n = n;
    plan.n_stages = static_cast<int>(r.size());
    for (std::size_t i = 0; i < r.size(); ++i) plan.radix[i] = r[i];
    plan.table = table.as<void>();
    plan.eps = eps.as<void>();
  }
  const cx<T>* tw() const { return table.as<cx<T>>(); }
  // 1 / |w_m| - 1 of the stored twiddles (complex64 kernels only)
  const T* tw_eps() const { return eps.as<T>(); }
};

unsigned blocks_for(long n, int threads) { return static_cast<unsigned>((n + threads - 1) / threads); }

constexpr int kThreads = 256;
// From this many grid points on, the specular step runs on a stream of its own beside T_Zr and T_xy; below, before them
// on their stream. The two events that join the streams cost about 18 us a block and one workgroup's step 11 us (2048
// points), 20 (4200), 26 (6144) to 32 us (9504): on one stream 34 us a block instead of 46 (2048 points), 92 instead of
// 97 (4200), but 369 instead of 360 (6144) and 166 instead of 145 (9504).
constexpr int kSpecularBesidePoints = 5120;

void set_lds(const void* kernel, std::size_t bytes) {
  HIP_CHECK(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
}

// Launch through the symbol with a packed argument list (hipLaunchKernel), so one call covers every instantiation.
void launch(const void* fn, unsigned grid, unsigned threads, std::size_t lds, hipStream_t stream, void** args) {
  HIP_CHECK(hipLaunchKernel(fn, dim3(grid), dim3(threads), args, lds, stream));
}

}  // namespace

// ---------------------------------------------------------------------------------------------------------------
// Backend state, common part.
struct spo_hip_backend {
  spo_hip_shape shape{};
  spo_dev::Shape s{};
  hipStream_t stream = nullptr;
  // The specular grid's step runs on `side` (default priority, like `stream`), overlapping T_Zr and T_xy of the
  // scattering grid; `stream` waits for spec_ready before anything that touches the specular wave again.
  hipStream_t side = nullptr;
  hipEvent_t main_ready = nullptr, spec_ready = nullptr;
  // Graph mode (spo_hip_graph_enable): one analysis step captured from `stream` (with `side` joined through the
  // events) at its first use, then replayed. The step's launches and arguments do not change between steps.
  bool use_graph = false;
  hipGraphExec_t step_graph = nullptr;
  int batches = 0;  // spo_hip_batch objects this backend is a member of (it may not be destroyed before them)
  int max_lds = 65536;
  spo_hip_analysis analysis{};

  // FP64 in both modes: specular wave and its factors, the analysis.
  Buffer spec, spec_full, spec_half, spec_gas, z_spec_opt, r_opt_d, s2sc_d, sc2s_d;
  Buffer densities, partial, plane, staging, bk, sums;
  Buffer rot_index, dif_slot, radial_weight, initial_radial, energies, shift_f_d;
  std::unique_ptr<DevicePlan<double>> plan_r_d, plan_zsp, plan_x_d, plan_y_d;
  std::size_t staging_values = 0;

  // Kernel timing (spo_hip_profile_enable): one event pair per launch on `stream`.
  struct Timed {
    int kernel;
    hipEvent_t start, stop;
  };
  bool profiling = false;
  std::vector<std::string> kernel_names;
  std::vector<Timed> timed_launches;
  std::vector<hipEvent_t> event_pool;

  hipEvent_t take_event() {
    if (!event_pool.empty()) {
      hipEvent_t e = event_pool.back();
      event_pool.pop_back();
      return e;
    }
    hipEvent_t e;
    HIP_CHECK(hipEventCreate(&e));
    return e;
  }
  // Runs `launch_fn` (one kernel launch on `stream`), bracketed by events when profiling.
  // `on`: the stream launch_fn launches on (default `stream`).
  template <typename F>
  void timed(const char* name, F&& launch_fn, hipStream_t on = nullptr) {
    if (!profiling) {
      launch_fn();
      HIP_CHECK(hipGetLastError());
      return;
    }
    const hipStream_t st = on ? on : stream;
    int id = 0;
    while (id < static_cast<int>(kernel_names.size()) && kernel_names[id] != name) ++id;
    if (id == static_cast<int>(kernel_names.size())) kernel_names.emplace_back(name);
    Timed t{id, take_event(), take_event()};
    HIP_CHECK(hipEventRecord(t.start, st));
    launch_fn();
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipEventRecord(t.stop, st));
    timed_launches.push_back(t);
  }

  virtual ~spo_hip_backend() {
    for (const Timed& t : timed_launches) {
      (void)hipEventDestroy(t.start);
      (void)hipEventDestroy(t.stop);
    }
    for (hipEvent_t e : event_pool) (void)hipEventDestroy(e);
    if (step_graph) (void)hipGraphExecDestroy(step_graph);
    if (side) {
      (void)hipStreamSynchronize(side);
      (void)hipStreamDestroy(side);
    }
    if (main_ready) (void)hipEventDestroy(main_ready);
    if (spec_ready) (void)hipEventDestroy(spec_ready);
    if (stream) {
      (void)hipStreamSynchronize(stream);
      (void)hipStreamDestroy(stream);
    }
  }

  // One block of the schedule: the specular grid's kinetic step (half or full), the scattering grid's T_Zr and
  // T_xy (scattering: 0 none, 1 half, 2 full) and, unless kinetic_only, V.
  virtual void step_block(bool specular_half, int scattering, bool kinetic_only) = 0;
  void kinetic_and_potential(bool half, bool kinetic_only) { step_block(half, half ? 1 : 2, kinetic_only); }
  // Merged half steps (SPO_HIP_MERGE_HALF_STEPS=1, eager single-run steps): an analysis step leaves the scattering
  // wave's trailing T(dt/2) pending, and the next step's leading T(dt/2) applies both as one T(dt); the analysis
  // reads its plane from a T(dt/2) of the plane alone, and every other read of the wave applies the pending half
  // step first (flush_pending). Same results up to rounding; off by default, since a run split by a restart file
  // then no longer repeats the unsplit run bit for bit.
  bool merge_halves = false;
  bool pending_half = false;
  virtual void flush_pending() = 0;
  virtual void upload_wave(const double* scattering) = 0;
  virtual void download_wave(double* scattering) = 0;
  virtual void z_plane(int iz) = 0;
  virtual void block_densities() = 0;
  virtual void site_column(int ixy, double* out) = 0;
  // Every BK coefficient; from_specular: the initial state's from the specular wave at line iz_specular.
  virtual void bk_scattering(bool from_specular, int iz_specular) = 0;
  // One analysis step of the energy-resolved sums of the scattering wave (er_phase holds exp(i E t)).
  virtual void energy_resolved_scattering() = 0;

  // The specular grid's step in one launch (specular_plane_kernel), whose order the factors then have.
  const void* spec_fn = nullptr;
  spo_dev::ZrShape spec_shape = {};
  std::size_t spec_lds = 0;
  bool spec_beside = true;  // the specular step runs on `side`, beside T_Zr and T_xy

  // Energy-resolved sums: device layout [site][energy][irot][izr] and [energy][iz][ir].
  Buffer er_sums, er_specular, er_sites, er_phase;
  int er_n_sites = 0, er_n_energies = 0;
  double er_dt = 0.0;

  void specular_step(bool half, bool kinetic_only);
  void lines_d(cx<double>* data, spo_dev::Lines L, const DevicePlan<double>& p, int sign, int mode,
               const cx<double>* factor, int f_line, int f_elem);
  void analyse(int surface_fixed, int iz_specular, double t, double* coefficients);
};

void spo_hip_backend::lines_d(cx<double>* data, spo_dev::Lines L, const DevicePlan<double>& p, int sign, int mode,
                              const cx<double>* factor, int f_line, int f_elem) {
  // Few lines a workgroup: the grid has a few hundred lines in all, and they should be on many CUs.
  L.lines_per_block = std::max(1, std::min({64, 65536 / (L.n * static_cast<int>(sizeof(cx<double>))), L.count / 64}));
  const std::size_t lds = std::size_t(L.lines_per_block) * L.n * sizeof(cx<double>);
  const unsigned grid = blocks_for(L.count, L.lines_per_block);
  timed("specular_lines_fft", [&] {
    hipLaunchKernelGGL(spo_dev::lines_fft_kernel<double>, dim3(grid), dim3(kThreads), lds, side, data, L, p.plan,
                       sign, mode, factor, static_cast<const cx<double>*>(nullptr), f_line, f_elem);
  }, side);
}

// Specular grid: r lines, Z lines with the kinetic factor (FFT scales folded in), r lines back, then the gas phase
// beyond zasymp and the absorbers (src/propagation/specular_operator.cpp:40-71). FP64.
void spo_hip_backend::specular_step(bool half, bool kinetic_only) {
  // On `side`, after everything already on `stream` (the last projection wrote the specular wave).
  const hipStream_t on = spec_beside ? side : stream;
  if (spec_beside) {
    HIP_CHECK(hipEventRecord(main_ready, stream));
    HIP_CHECK(hipStreamWaitEvent(side, main_ready, 0));
  }
  cx<double>* sp = spec.as<cx<double>>();
  if (spec_fn) {
    const cx<double>* tz = plan_zsp->tw();
    const cx<double>* tr = plan_r_d->tw();
    const cx<double>* factor = (half ? spec_half : spec_full).as<cx<double>>();
    int potential = kinetic_only ? 0 : 1;
    const cx<double>* gas = spec_gas.as<cx<double>>();
    const double* zo = z_spec_opt.as<double>();
    const double* ro = r_opt_d.as<double>();
    void* args[] = {&sp, &spec_shape, const_cast<cx<double>**>(&tz), const_cast<cx<double>**>(&tr),
                    const_cast<cx<double>**>(&factor), &potential, &s.nzpot, const_cast<cx<double>**>(&gas),
                    const_cast<double**>(&zo), const_cast<double**>(&ro), &s.r_abs_first, &s.r_abs_last};
    timed("specular_plane", [&] { launch(spec_fn, 1, spo_dev::kSpecularThreads, spec_lds, on, args); }, on);
    if (spec_beside) HIP_CHECK(hipEventRecord(spec_ready, side));
    return;
  }
  spo_dev::Lines r_lines{s.nr, s.nzsp, s.nzsp, s.nr, 0, 1, 1};
  spo_dev::Lines z_lines{s.nzsp, s.nr, s.nr, 1, 0, s.nr, 1};
  lines_d(sp, r_lines, *plan_r_d, -1, 0, nullptr, 0, 0);
  lines_d(sp, z_lines, *plan_zsp, -1, 1, (half ? spec_half : spec_full).as<cx<double>>(), 1, s.nr);
  lines_d(sp, r_lines, *plan_r_d, +1, 0, nullptr, 0, 0);
  if (!kinetic_only) {
    timed("specular_potential", [&] {
      hipLaunchKernelGGL(spo_dev::specular_potential_kernel<double>, dim3(blocks_for(long(s.nr) * s.nzsp, kThreads)),
                         dim3(kThreads), 0, side, sp, s, spec_gas.as<cx<double>>(), z_spec_opt.as<double>(),
                         r_opt_d.as<double>());
    }, side);
  }
  HIP_CHECK(hipEventRecord(spec_ready, side));
}

void spo_hip_backend::analyse(int surface_fixed, int iz_specular, double t, double* coefficients) {
  const spo_hip_analysis& a = analysis;
  const std::size_t n = std::size_t(a.n_states) * a.n_v;
  if (surface_fixed && (iz_specular < 0 || iz_specular >= s.nzsp))
    throw Status(SPO_HIP_E_ARGUMENT, "specular line out of range");
  bk_scattering(surface_fixed != 0, iz_specular);
  const long total = long(n) * a.n_energies;
  timed("s_accumulate", [&] {
    hipLaunchKernelGGL(spo_dev::s_accumulate_kernel, dim3(blocks_for(total, kThreads)), dim3(kThreads), 0, stream,
                       sums.as<cx<double>>(), bk.as<cx<double>>(), static_cast<int>(n), a.n_energies,
                       energies.as<double>(), t, a.analysis_time_step);
  });
  if (coefficients)
    HIP_CHECK(hipMemcpyAsync(coefficients, bk.as<void>(), n * sizeof(cx<double>), hipMemcpyDeviceToHost, stream));
  HIP_CHECK(hipStreamSynchronize(stream));
}

// ---------------------------------------------------------------------------------------------------------------
// The part that depends on the storage type of the scattering wave.
namespace {

template <typename T>
struct State final : spo_hip_backend {
  Buffer psi, zr_full, zr_half, xy_full, xy_half, rot_half, rot_half_t, before, gas_step, z_opt;
  // complex64: the FP32 remainders of the factor tables (factor_lo); empty in FP64
  Buffer zr_full_lo, zr_half_lo, xy_full_lo, xy_half_lo, before_lo, gas_step_lo, shift_f_lo, shift_b_lo, rot_lo,
      rot_lo_t;
  Buffer shift_f, shift_b, s2sc, legendre, block_first, block_size, block_offset, rot_block, rep_of, op_of, phi_index;
  Buffer exp_table, legendre_t;
  Buffer frag_fwd, frag_bwd, fwd_offset, bwd_offset, site_order, rot_pm, lo_fwd, lo_bwd, hi_fwd, hi_bwd;
  // interaction_kernel_inplace (build_angular_plan): its tables, and the low parts' fragments of L (complex64)
  Buffer ang_tasks, ang_free, ang_phi_map, ang_sites, ang_rot;
  spo_dev::AngularPlan ang = {};
  bool build_angular_plan(const spo_hip_tables* t, const std::vector<int>& offsets, int r1, int r2);
  void run_interaction_inplace(const Variant& v);
  int max_jt = 1;
  int frag_fwd_count = 0, frag_bwd_count = 0;
  int legendre_size = 0;
  std::size_t zr_lds = 0, xy_lds = 0, v_lds = 0;
  std::unique_ptr<DevicePlan<T>> plan_z, plan_r, plan_x, plan_y, plan_phi;
  int xy_c = 1, v_c = 1;
  // Launch variants of the register-pass and MFMA kernels (identical arithmetic) and the one in use.
  std::vector<Variant> zr_variants, xy_variants, v_variants;
  int zr_pick = 0, xy_pick = 0, v_pick = 0;
  const void* v_fn = nullptr;
  bool zr_fused = false;

  // The T_Zr factors (and complex64 remainders), natural or in the order of zr_inplace_kernel's places, for the kernel in
  // use.
  void upload_zr_factors(const std::vector<double>& full, const std::vector<double>& half, const spo_dev::ZrShape* order);

  Buffer ana_row;  // the analysis row of the scattering wave at the analysis time (merged half steps)

  void run_zr(const Variant& v, bool half, cx<T>* row_out = nullptr, int row = -1);
  void run_xy(const Variant& v, bool half, bool kinetic_only, cx<T>* data = nullptr,
              const spo_dev::Shape* on = nullptr);
  void run_coupling();
  void run_interaction(const Variant& v);
  void tune();
  void scattering_kinetic(bool half, bool kinetic_only);

  void step_block(bool specular_half, int scattering, bool kinetic_only) override;
  void flush_pending() override;
  void upload_wave(const double* scattering) override;
  void download_wave(double* scattering) override;
  void z_plane(int iz) override;
  void block_densities() override;
  void site_column(int ixy, double* out) override;
  void bk_scattering(bool from_specular, int iz_specular) override;
  void energy_resolved_scattering() override;
  void lines(cx<T>* data, spo_dev::Lines L, const DevicePlan<T>& p, int sign, int mode, const cx<T>* factor,
             const cx<T>* factor_lo, int f_line, int f_elem);
};

template <typename T>
void State<T>::lines(cx<T>* data, spo_dev::Lines L, const DevicePlan<T>& p, int sign, int mode, const cx<T>* factor,
                     const cx<T>* factor_lo, int f_line, int f_elem) {
  L.lines_per_block = std::max(1, std::min(64, 65536 / (L.n * static_cast<int>(sizeof(cx<T>)))));
  const std::size_t lds = std::size_t(L.lines_per_block) * L.n * sizeof(cx<T>);
  const unsigned grid = blocks_for(L.count, L.lines_per_block);
  timed("zr_lines_fft", [&] {
    hipLaunchKernelGGL(spo_dev::lines_fft_kernel<T>, dim3(grid), dim3(kThreads), lds, stream, data, L, p.plan, sign,
                       mode, factor, factor_lo, f_line, f_elem);
  });
}

template <typename T>
void State<T>::run_zr(const Variant& v, bool half, cx<T>* row_out, int row) {
  cx<T>* ps = psi.as<cx<T>>();
  const cx<T>* tz = plan_z->tw();
  const cx<T>* tr = plan_r->tw();
  const T* ez = plan_z->tw_eps();
  const T* er = plan_r->tw_eps();
  spo_dev::ZrShape shape = v.zr;
  const cx<T>* zr = (half ? zr_half : zr_full).as<cx<T>>();
  const cx<T>* fl = (half ? zr_half_lo : zr_full_lo).as<cx<T>>();
  void* args[] = {&ps, &shape, const_cast<cx<T>**>(&tz), const_cast<cx<T>**>(&tr), const_cast<cx<T>**>(&zr),
                  const_cast<T**>(&ez), const_cast<T**>(&er), const_cast<cx<T>**>(&fl), &row_out, &row};
  launch(v.fn, s.n_rot * s.n_xy, v.threads, v.lds, stream, args);
}

template <typename T>
void State<T>::upload_zr_factors(const std::vector<double>& full, const std::vector<double>& half,
                                 const spo_dev::ZrShape* order) {
  std::vector<double> f(full), h(half);
  for (int iz = 0; order && iz < s.nz; ++iz)
    for (int ir = 0; ir < s.nr; ++ir) {
      const std::size_t to = 2 * (ir + std::size_t(s.nr) * iz), from = 2 * spo_dev::zr_factor_order(*order, iz, ir);
      for (int c = 0; c < 2; ++c) {
        f[to + c] = full[from + c];
        h[to + c] = half[from + c];
      }
    }
  zr_full = upload_complex<T>(f.data(), s.n_zr);
  zr_full_lo = factor_lo<T>(f.data(), s.n_zr);
  zr_half = upload_complex<T>(h.data(), s.n_zr);
  zr_half_lo = factor_lo<T>(h.data(), s.n_zr);
}

template <typename T>
void State<T>::run_xy(const Variant& v, bool half, bool kinetic_only, cx<T>* data, const spo_dev::Shape* on) {
  cx<T>* ps = data ? data : psi.as<cx<T>>();
  spo_dev::Shape sh = on ? *on : s;
  const int tiles = (sh.n_zr + v.param - 1) / v.param;
  const cx<T>* factor = (half ? xy_half : xy_full).as<cx<T>>();
  const cx<T>* sf = shift_f.as<cx<T>>();
  const cx<T>* sb = shift_b.as<cx<T>>();
  int needs_shift = shape.needs_shift;
  int apply_potential = kinetic_only ? 0 : 1;
  const T* zo = z_opt.as<T>();
  const cx<T>* bf = before.as<cx<T>>();
  const cx<T>* gs = gas_step.as<cx<T>>();
  spo_dev::XyLo<T> lo{(half ? xy_half_lo : xy_full_lo).as<cx<T>>(), shift_f_lo.as<cx<T>>(),
                      shift_b_lo.as<cx<T>>(), before_lo.as<cx<T>>(), gas_step_lo.as<cx<T>>()};
  void* args[] = {&ps, &sh, const_cast<cx<T>**>(&factor), const_cast<cx<T>**>(&sf), const_cast<cx<T>**>(&sb),
                  &needs_shift, &apply_potential, const_cast<T**>(&zo), const_cast<cx<T>**>(&bf),
                  const_cast<cx<T>**>(&gs), &lo};
  launch(v.fn, tiles * sh.n_rot, v.threads, v.lds, stream, args);
}

// The specular wave's part of the initial channel, ahead of an interaction kernel that does not add it itself.
template <typename T>
void State<T>::run_coupling() {
  hipLaunchKernelGGL(spo_dev::specular_coupling_kernel<T>, dim3(blocks_for(long(s.n_zr_pot) * s.n_xy, 256)), dim3(256),
                     0, stream, psi.as<cx<T>>(), spec.as<cx<double>>(), s, rot_half.as<cx<T>>(), s2sc.as<cx<T>>());
}

template <typename T>
void State<T>::run_interaction(const Variant& v) {
  cx<T>* ps = psi.as<cx<T>>();
  spo_dev::AngularTables at{legendre.as<double>(),  block_first.as<int>(), block_size.as<int>(),
                            block_offset.as<int>(), rot_block.as<int>(),   rep_of.as<int>(),
                            op_of.as<int>(),        phi_index.as<int>()};
  if (v.kind == spo_dev::InteractionKind::in_place) {
    run_interaction_inplace(v);
    return;
  }
  const int tiles = (s.n_zr_pot + 7) / 8;
  const int pair = s.n_xy % 8 == 0 ? 1 : 0;
  const cx<double>* sp = spec.as<cx<double>>();
  const cx<T>* et = exp_table.as<cx<T>>();
  const cx<T>* rh = rot_half_t.as<cx<T>>();
  const cx<T>* rl = rot_lo_t.as<cx<T>>();
  const cx<T>* ssc = s2sc.as<cx<T>>();
  const cx<T>* tp = plan_phi->tw();
  const T* ep = plan_phi->tw_eps();
  spo_dev::MfmaTables mt{fwd_offset.as<int>(), bwd_offset.as<int>(), site_order.as<int>(), pair};
  const T* ff = frag_fwd.as<T>();
  const T* fb = frag_bwd.as<T>();
  int mj = max_jt;
  const int grid = pair ? 2 * ((tiles + 1) / 2) * s.n_xy : tiles * s.n_xy;
  if (v.kind == spo_dev::InteractionKind::buffer) {
    const cx<T>* rp = rot_pm.as<cx<T>>();
    const unsigned* lf = lo_fwd.as<unsigned>();
    const unsigned* lb = lo_bwd.as<unsigned>();
    const unsigned* hf = hi_fwd.as<unsigned>();
    const unsigned* hb = hi_bwd.as<unsigned>();
    int nf = frag_fwd_count, nbw = frag_bwd_count;
    void* args[] = {&ps, &s, const_cast<cx<T>**>(&tp), &at, &mt, const_cast<T**>(&ff), const_cast<T**>(&fb),
                    &nf, &nbw, const_cast<cx<T>**>(&et), const_cast<cx<T>**>(&rp), const_cast<unsigned**>(&lf),
                    const_cast<unsigned**>(&lb), const_cast<T**>(&ep), const_cast<unsigned**>(&hf),
                    const_cast<unsigned**>(&hb)};
    launch(v.fn, grid, v.threads, v.lds, stream, args);
    return;
  }
  void* args[] = {&ps, const_cast<cx<double>**>(&sp), &s, const_cast<cx<T>**>(&tp), &at, &mt,
                  const_cast<T**>(&ff), const_cast<T**>(&fb), &mj, const_cast<cx<T>**>(&et),
                  const_cast<cx<T>**>(&rh), const_cast<cx<T>**>(&ssc), const_cast<T**>(&ep),
                  const_cast<cx<T>**>(&rl)};
  launch(v.fn, grid, v.threads, v.lds, stream, args);
}

template <typename T>
void State<T>::run_interaction_inplace(const Variant& v) {
  cx<T>* ps = psi.as<cx<T>>();
  const cx<double>* sp = spec.as<cx<double>>();
  spo_dev::AngularPlan plan = ang;
  plan.rows = s.n_theta * v.columns;
  plan.inv_rows = spo_dev::inverse_of(plan.rows);
  const int tiles = (s.n_zr_pot + v.columns - 1) / v.columns;
  const unsigned grid = 8u * plan.sites_per_xcd * 2u * ((tiles + 1) / 2);
  const int* rep = rep_of.as<int>();
  const int* op = op_of.as<int>();
  const T* ff = frag_fwd.as<T>();
  const T* fb = frag_bwd.as<T>();
  const unsigned* lf = lo_fwd.as<unsigned>();
  const unsigned* lb = lo_bwd.as<unsigned>();
  const cx<T>* et = exp_table.as<cx<T>>();
  const cx<T>* rp = ang_rot.as<cx<T>>();
  const cx<T>* rh = rot_half.as<cx<T>>();
  const cx<T>* ssc = s2sc.as<cx<T>>();
  const cx<T>* tp = plan_phi->tw();
  const T* ep = plan_phi->tw_eps();
  void* args[] = {&ps, const_cast<cx<double>**>(&sp), &s, &plan, const_cast<int**>(&rep), const_cast<int**>(&op),
                  const_cast<T**>(&ff), const_cast<T**>(&fb), const_cast<unsigned**>(&lf),
                  const_cast<unsigned**>(&lb), const_cast<cx<T>**>(&et), const_cast<cx<T>**>(&rp),
                  const_cast<cx<T>**>(&rh), const_cast<cx<T>**>(&ssc), const_cast<cx<T>**>(&tp),
                  const_cast<T**>(&ep)};
  launch(v.fn, grid, v.threads, v.lds, stream, args);
}

// The tables of interaction_kernel_inplace (the fragments themselves are frag_fwd and frag_bwd); false where the blocks
// m and -m do not share their Legendre matrix up to the sign and their rotation factors, which the kernel relies on.
template <typename T>
bool State<T>::build_angular_plan(const spo_hip_tables* t, const std::vector<int>& offsets, int r1, int r2) {
  const int mm = s.mj_max, n_tt = (s.n_theta + 15) / 16, k_bwd = (s.n_theta + 3) / 4;
  std::vector<int> fo(s.n_blocks), bo(s.n_blocks);
  int nf = 0, nb_count = 0, base = mm;
  for (int b = 0; b < s.n_blocks; ++b) {
    fo[b] = nf;
    nf += n_tt * ((t->block_size[b] + 3) / 4);
    bo[b] = nb_count;
    nb_count += ((t->block_size[b] + 15) / 16) * k_bwd;
    if (t->block_size[b] > t->block_size[base]) base = b;
  }
  // Rotation factors: one row per row of the longest block where every block's rows are a run of those (the rows of
  // one J are the same for every mJ), else one per basis function.
  auto same_row = [&](int i, int j) {
    for (int ir = 0; ir < s.nr; ++ir)
      for (int c = 0; c < 2; ++c)
        if (t->rotation_half[2 * (i + std::size_t(s.n_rot) * ir) + c] !=
            t->rotation_half[2 * (j + std::size_t(s.n_rot) * ir) + c])
          return false;
    return true;
  };
  std::vector<int> rot_first(s.n_blocks, -1);
  const int bf = t->block_first[base], bn = t->block_size[base];
  bool shared = true;
  for (int b = 0; b < s.n_blocks && shared; ++b) {
    for (int o = 0; o + t->block_size[b] <= bn && rot_first[b] < 0; ++o) {
      bool all = true;
      for (int j = 0; j < t->block_size[b] && all; ++j) all = same_row(t->block_first[b] + j, bf + o + j);
      if (all) rot_first[b] = o;
    }
    shared = rot_first[b] >= 0;
  }
  const int rot_rows = shared ? bn : s.n_rot, rot_from = shared ? bf : 0;
  if (!shared)
    for (int b = 0; b < s.n_blocks; ++b) rot_first[b] = t->block_first[b];
  std::vector<spo_dev::RotEntry<T>> pm(2 * std::size_t(rot_rows) * s.nr, spo_dev::RotEntry<T>{});
  for (int row = 0; row < rot_rows; ++row)
    for (int ir = 0; ir < s.nr; ++ir) {
      const std::size_t from = 2 * (row + rot_from + std::size_t(s.n_rot) * ir);
      set_rot_entries(pm.data() + spo_dev::rot_pm_index(row, ir, s.nr, 0), t->rotation_half[from],
                      t->rotation_half[from + 1]);
    }
  std::vector<spo_dev::AngularTask> tasks;
  std::vector<char> used(s.n_phi, 0);
  const int cb = sizeof(cx<T>), fragment = 64 * sizeof(T);
  for (int m = 0; m <= mm; ++m) {
    const int b[2] = {mm + m, mm - m}, nb = t->block_size[b[0]];
    bool plus = t->block_size[b[1]] == nb && rot_first[b[1]] == rot_first[b[0]], minus = plus;
    for (int k = 0; k < s.n_theta * nb && (plus || minus); ++k) {
      plus = plus && t->legendre[offsets[b[0]] + k] == t->legendre[offsets[b[1]] + k];
      minus = minus && t->legendre[offsets[b[0]] + k] == -t->legendre[offsets[b[1]] + k];
    }
    if (!plus && !minus) return false;
    spo_dev::AngularTask task{};
    for (int side = 0; side < 2; ++side) {
      const int place = spo_dev::phi_place(side && m ? s.n_phi - m : m, r1, r2), first = t->block_first[b[side]];
      used[place] = 1;
      task.psi[side] = first * s.n_zr * cb;
      task.place[side] = place * cb;
      if (s.ichn >= first && s.ichn < first + nb && !(side && m == 0)) {
        ang.task_initial = m;
        ang.side_initial = side;
        ang.j_initial = s.ichn - first;
      }
    }
    task.nb = nb;
    task.fwd = fo[b[0]] * fragment;
    task.bwd = bo[b[0]] * fragment;
    task.negate = plus ? 0 : 1;
    task.rot = rot_first[b[0]] * s.nr * 32;
    tasks.push_back(task);
  }
  std::vector<int> free_places;
  for (int p = 0; p < s.n_phi; ++p)
    if (!used[p]) free_places.push_back(p);
  ang.n_free = static_cast<int>(free_places.size());
  free_places.push_back(0);  // never empty
  std::vector<int> map;
  for (int op = 0; op < shape.n_operations; ++op)
    for (int p = 0; p < s.n_phi; ++p) map.push_back(t->phi_index[spo_dev::phi_frequency(p, r1, r2) + s.n_phi * op]);
  // Sites sorted by representative, an eighth to each XCD (rounded up; the rest of the positions hold none).
  std::vector<int> sorted(s.n_xy);
  for (int i = 0; i < s.n_xy; ++i) sorted[i] = i;
  std::stable_sort(sorted.begin(), sorted.end(),
                   [&](int x, int y) { return t->representative_of[x] < t->representative_of[y]; });
  const int per = (s.n_xy + 7) / 8;
  std::vector<int> sites(8 * std::size_t(per), -1);
  for (int x = 0; x < 8; ++x)
    for (int k = 0; k < per; ++k)
      if (per * x + k < s.n_xy) sites[8 * k + x] = sorted[per * x + k];
  ang_tasks = upload(tasks.data(), tasks.size() * sizeof(spo_dev::AngularTask));
  ang_free = upload(free_places.data(), free_places.size() * sizeof(int));
  ang_phi_map = upload(map.data(), map.size() * sizeof(int));
  ang_sites = upload(sites.data(), sites.size() * sizeof(int));
  ang_rot = upload(pm.data(), pm.size() * sizeof(spo_dev::RotEntry<T>));
  ang.tasks = ang_tasks.as<spo_dev::AngularTask>();
  ang.n_tasks = static_cast<int>(tasks.size());
  ang.free_places = ang_free.as<int>();
  ang.phi_map = ang_phi_map.as<int>();
  ang.site_order = ang_sites.as<int>();
  ang.sites_per_xcd = per;
  ang.inv_nr = spo_dev::inverse_of(s.nr);
  ang.rot_rows = rot_rows;
  ang.frag_fwd = nf;
  ang.frag_bwd = nb_count;
  return true;
}

// The launch tuner. The variants of one family compute the same transforms with other block sizes, tiles and FFT
// radices (interaction: in other kernels), so their results can differ in the last bits, and the default is therefore
// fixed: the first variant of each family (ordered by what measured fastest on MI355X for the shape), which keeps
// repeated runs bitwise identical. SPO_HIP_TUNE=auto makes the first backend of a process with a given shape, precision
// and list of variants time every one on the scattering wave's memory (cleared afterwards), one warm-up and two timed
// launches each, and keep the fastest for the process. The list belongs to the key because its order and length depend
// on more than the shape: the tables, SPO_HIP_INTERACTION and SPO_HIP_CONTRACTION. SPO_HIP_TUNE="zr=384,xy=8,
// interaction=16" forces variants by thread count (zr), izr per tile (xy) or wavefronts (interaction), and
// "interaction=#2" the variant at that place in the family's list (0 = the default).
struct TuneCache {
  std::mutex mutex;
  std::map<std::string, int> picks;  // shape and list -> place in that list
};
TuneCache& tune_cache() {
  static TuneCache cache;
  return cache;
}

// The variant SPO_HIP_TUNE selects for a family, or -1 to time them (SPO_HIP_TUNE=auto).
int forced_variant(const std::vector<Variant>& v, const char* family, bool by_threads) {
  const char* env = std::getenv("SPO_HIP_TUNE");
  if (!env) return 0;
  const std::string spec = env;
  if (spec == "auto") return -1;
  const std::string key = std::string(family) + "=";
  const std::size_t at = spec.find(key);
  if (at == std::string::npos) return 0;
  const char* value = spec.c_str() + at + key.size();
  if (*value == '#') {  // "family=#k": the k-th variant of the family's list (0 = the default)
    const int k = std::atoi(value + 1);
    if (k < 0 || k >= static_cast<int>(v.size()))
      throw Status(SPO_HIP_E_ARGUMENT, std::string("SPO_HIP_TUNE: ") + family + " has " + std::to_string(v.size()) +
                                           " variants, no #" + std::to_string(k));
    return k;
  }
  const int want = std::atoi(value);
  for (std::size_t i = 0; i < v.size(); ++i)
    if ((by_threads ? v[i].threads : v[i].param) == want) return static_cast<int>(i);
  throw Status(SPO_HIP_E_ARGUMENT, std::string("SPO_HIP_TUNE: no ") + family + " variant " + std::to_string(want));
}

template <typename T>
void State<T>::tune() {
  int dev = 0;
  HIP_CHECK(hipGetDevice(&dev));
  bool ran = false;  // kernels ran on the scattering wave
  auto pick = [&](const std::vector<Variant>& v, const char* family, bool by_threads, auto&& run) -> int {
    if (v.size() < 2) return 0;
    const int forced = forced_variant(v, family, by_threads);
    if (forced >= 0) return forced;
    std::string key = std::string(family) + ":";
    for (int n : {s.nz, s.nr, s.nx, s.ny, s.nzpot, s.n_rot, s.n_theta, s.n_phi, s.n_rep}) key += std::to_string(n) + "x";
    key.back() = ':';
    key += std::to_string(sizeof(T)) + ":" + std::to_string(dev);
    std::string list = key;
    for (const Variant& one : v)
      list += ":" + std::to_string(reinterpret_cast<std::uintptr_t>(one.fn)) + "/" + std::to_string(one.threads);
    {
      const std::lock_guard<std::mutex> lock(tune_cache().mutex);
      const auto hit = tune_cache().picks.find(list);
      if (hit != tune_cache().picks.end()) return hit->second;
    }
    ran = true;
    hipEvent_t e0, e1;
    HIP_CHECK(hipEventCreate(&e0));
    HIP_CHECK(hipEventCreate(&e1));
    int best = 0;
    float best_ms = 0.0f;
    for (std::size_t i = 0; i < v.size(); ++i) {
      run(v[i]);
      HIP_CHECK(hipEventRecord(e0, stream));
      run(v[i]);
      run(v[i]);
      HIP_CHECK(hipEventRecord(e1, stream));
      HIP_CHECK(hipEventSynchronize(e1));
      float ms = 0.0f;
      HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
      if (i == 0 || ms < best_ms) {
        best = static_cast<int>(i);
        best_ms = ms;
      }
    }
    HIP_CHECK(hipEventDestroy(e0));
    HIP_CHECK(hipEventDestroy(e1));
    {
      const std::lock_guard<std::mutex> lock(tune_cache().mutex);
      tune_cache().picks[list] = best;
    }
    if (std::getenv("SPO_HIP_TUNE_LOG"))
      std::fprintf(stderr, "spo_hip tune %s: %s=%d (#%d of %zu, %.3f ms for two launches)\n", key.c_str(), family,
                   by_threads ? v[best].threads : v[best].param, best, v.size(), best_ms);
    return best;
  };
  zr_pick = pick(zr_variants, "zr", true, [&](const Variant& v) { run_zr(v, false); });
  xy_pick = pick(xy_variants, "xy", false, [&](const Variant& v) { run_xy(v, false, false); });
  // Each kernel with what it needs for the same work: those that read the wave as it is, after the specular coupling.
  v_pick = pick(v_variants, "interaction", false, [&](const Variant& v) {
    if (v.kind != spo_dev::InteractionKind::in_place) run_coupling();
    run_interaction(v);
  });
  // The interaction adds the specular wave's part to the scattering wave, which is zero again when this returns.
  if (ran)
    HIP_CHECK(hipMemsetAsync(psi.as<void>(), 0, std::size_t(s.n_zr) * s.n_rot * s.n_xy * sizeof(cx<T>), stream));
  HIP_CHECK(hipStreamSynchronize(stream));
}

template <typename T>
void State<T>::scattering_kinetic(bool half, bool kinetic_only) {
  cx<T>* ps = psi.as<cx<T>>();
  // T_Zr.
  const cx<T>* zr = (half ? zr_half : zr_full).as<cx<T>>();
  const cx<T>* zr_lo = (half ? zr_half_lo : zr_full_lo).as<cx<T>>();
  const int n_planes = s.n_rot * s.n_xy;
  if (!zr_variants.empty()) {
    timed("zr_plane", [&] { run_zr(zr_variants[zr_pick], half); });
  } else if (zr_fused) {
    timed("zr_plane_generic", [&] {
      hipLaunchKernelGGL(spo_dev::zr_plane_kernel<T>, dim3(n_planes), dim3(kThreads), std::size_t(s.n_zr) * sizeof(cx<T>),
                         stream, ps, s, plan_z->plan, plan_r->plan, zr, zr_lo);
    });
  } else {
    spo_dev::Lines r_lines{s.nr, s.nz * n_planes, s.nz, s.nr, s.n_zr, 1, 1};
    spo_dev::Lines z_lines{s.nz, s.nr * n_planes, s.nr, 1, s.n_zr, s.nr, 1};
    lines(ps, r_lines, *plan_r, -1, 0, nullptr, nullptr, 0, 0);
    lines(ps, z_lines, *plan_z, -1, 1, zr, zr_lo, 1, s.nr);
    lines(ps, r_lines, *plan_r, +1, 0, nullptr, nullptr, 0, 0);
  }
  // T_xy and the diagonal part of V.
  if (!xy_variants.empty()) {
    timed("xy_tile", [&] { run_xy(xy_variants[xy_pick], half, kinetic_only); });
  } else {
    const int tiles = (s.n_zr + xy_c - 1) / xy_c;
    const cx<T>* factor = (half ? xy_half : xy_full).as<cx<T>>();
    const T* zo = z_opt.as<T>();
    const spo_dev::XyLo<T> lo{(half ? xy_half_lo : xy_full_lo).as<cx<T>>(), shift_f_lo.as<cx<T>>(),
                              shift_b_lo.as<cx<T>>(), before_lo.as<cx<T>>(), gas_step_lo.as<cx<T>>()};
    timed("xy_tile_generic", [&] {
      hipLaunchKernelGGL(spo_dev::xy_kernel<T>, dim3(tiles * s.n_rot), dim3(kThreads), xy_lds, stream, ps, s, xy_c,
                         plan_x->plan, plan_y->plan, factor, shift_f.as<cx<T>>(), shift_b.as<cx<T>>(),
                         shape.needs_shift, kinetic_only ? 0 : 1, zo, before.as<cx<T>>(), gas_step.as<cx<T>>(), lo);
    });
  }
}

template <typename T>
void State<T>::flush_pending() {
  if (!pending_half) return;
  pending_half = false;
  scattering_kinetic(true, true);
}

template <typename T>
void State<T>::step_block(bool specular_half, int scattering, bool kinetic_only) {
  if (scattering == 0 && !kinetic_only) throw Status(SPO_HIP_E_ARGUMENT, "a potential step without its kinetic step");
  specular_step(specular_half, kinetic_only);
  if (scattering != 0) scattering_kinetic(scattering == 1, kinetic_only);
  cx<T>* ps = psi.as<cx<T>>();
  // The specular step (on `side`) is complete before the specular wave is read or written on `stream` again.
  if (spec_beside) HIP_CHECK(hipStreamWaitEvent(stream, spec_ready, 0));
  if (kinetic_only || s.n_zr_pot == 0) return;
  // V in the interaction region, then the projection onto the specular grid.
  spo_dev::AngularTables at{legendre.as<double>(),  block_first.as<int>(), block_size.as<int>(),
                            block_offset.as<int>(), rot_block.as<int>(),   rep_of.as<int>(),
                            op_of.as<int>(),        phi_index.as<int>()};
  const int tiles = (s.n_zr_pot + v_c - 1) / v_c;
  const std::size_t lds = v_lds;
  const cx<double>* sp = spec.as<cx<double>>();
  const cx<T>* et = exp_table.as<cx<T>>();
  const cx<T>* rh = rot_half.as<cx<T>>();
  const cx<T>* ssc = s2sc.as<cx<T>>();
  if (!v_variants.empty()) {
    if (v_variants[v_pick].kind != spo_dev::InteractionKind::in_place)
      timed("specular_coupling", [&] { run_coupling(); });
    timed("interaction", [&] { run_interaction(v_variants[v_pick]); });
  } else if (v_fn) {
    const cx<T>* tp = plan_phi->tw();
    const T* lt = legendre_t.as<T>();
    int c = v_c;
    int ls = legendre_size;
    const cx<T>* rl = rot_lo.as<cx<T>>();
    const T* ep = plan_phi->tw_eps();
    void* args[] = {&ps, const_cast<cx<double>**>(&sp), &s, &c, const_cast<cx<T>**>(&tp), &at,
                    const_cast<cx<T>**>(&et), const_cast<cx<T>**>(&rh), const_cast<cx<T>**>(&ssc),
                    const_cast<T**>(&lt), &ls, const_cast<cx<T>**>(&rl), const_cast<T**>(&ep)};
    timed("interaction", [&] { launch(v_fn, tiles * s.n_xy, kThreads, lds, stream, args); });
  } else {
    timed("interaction_generic", [&] {
      hipLaunchKernelGGL(spo_dev::interaction_kernel<T>, dim3(tiles * s.n_xy), dim3(kThreads), lds, stream, ps, sp, s,
                         v_c, plan_phi->plan, at, et, rh, ssc, rot_lo.as<cx<T>>());
    });
  }
  timed("projection", [&] {
    hipLaunchKernelGGL(spo_dev::projection_kernel<T>, dim3(blocks_for(s.n_zr_pot, 64)),
                       dim3(64 * spo_dev::kProjectionWaves), 0,
                       stream, ps, spec.as<cx<double>>(), s, sc2s_d.as<cx<double>>(), s2sc_d.as<cx<double>>());
  });
}

template <typename T>
void State<T>::upload_wave(const double* scattering) {
  pending_half = false;  // a new wave at the analysis time
  const std::size_t per_izr = std::size_t(s.n_rot) * s.n_xy;
  const int chunk = static_cast<int>(std::max<std::size_t>(1, staging_values / per_izr));
  for (int izr0 = 0; izr0 < s.n_zr; izr0 += chunk) {
    const int count = std::min(chunk, s.n_zr - izr0);
    HIP_CHECK(hipMemcpyAsync(staging.as<void>(), scattering + 2 * per_izr * izr0, per_izr * count * sizeof(cx<double>),
                             hipMemcpyHostToDevice, stream));
    hipLaunchKernelGGL(spo_dev::host_to_device_kernel<T>, dim3(blocks_for(long(per_izr) * count, kThreads)),
                       dim3(kThreads), 0, stream, psi.as<cx<T>>(), s, staging.as<cx<double>>(), izr0, count);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(stream));
  }
}

template <typename T>
void State<T>::download_wave(double* scattering) {
  flush_pending();
  const std::size_t per_izr = std::size_t(s.n_rot) * s.n_xy;
  const int chunk = static_cast<int>(std::max<std::size_t>(1, staging_values / per_izr));
  for (int izr0 = 0; izr0 < s.n_zr; izr0 += chunk) {
    const int count = std::min(chunk, s.n_zr - izr0);
    hipLaunchKernelGGL(spo_dev::device_to_host_kernel<T>, dim3(blocks_for(long(per_izr) * count, kThreads)),
                       dim3(kThreads), 0, stream, psi.as<cx<T>>(), s, staging.as<cx<double>>(), izr0, count);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipMemcpyAsync(scattering + 2 * per_izr * izr0, staging.as<void>(), per_izr * count * sizeof(cx<double>),
                             hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
  }
}

template <typename T>
void State<T>::z_plane(int iz) {
  flush_pending();
  const long n = long(s.n_rot) * s.n_xy * s.nr;
  hipLaunchKernelGGL(spo_dev::z_plane_kernel<T>, dim3(blocks_for(n, kThreads)), dim3(kThreads), 0, stream,
                     psi.as<cx<T>>(), s, iz, plane.as<cx<double>>());
  HIP_CHECK(hipGetLastError());
}

template <typename T>
void State<T>::block_densities() {
  flush_pending();
  // One part per site (n_zr x n_xy partial sums over irot), then the parts added in site order: enough workgroups
  // to cover the device, where a few long per-thread loops over sites left it latency-bound.
  const int chunk = 1;
  const int parts = s.n_xy;
  timed("densities", [&] {
    hipLaunchKernelGGL(spo_dev::densities_partial_kernel<T>, dim3(blocks_for(s.n_zr, kThreads), parts), dim3(kThreads),
                       0, stream, psi.as<cx<T>>(), s, chunk, partial.as<double>());
  });
  timed("densities_sum", [&] {
    hipLaunchKernelGGL(spo_dev::densities_sum_kernel, dim3(blocks_for(s.n_zr, kThreads)), dim3(kThreads), 0, stream,
                       partial.as<double>(), s.n_zr, parts, densities.as<double>());
  });
}

template <typename T>
void State<T>::site_column(int ixy, double* out) {
  flush_pending();
  const std::size_t n = std::size_t(s.n_zr) * s.n_rot;
  if constexpr (sizeof(T) == sizeof(double)) {
    HIP_CHECK(hipMemcpyAsync(out, psi.as<cx<T>>() + n * ixy, n * sizeof(cx<T>), hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
  } else {
    std::vector<cx<T>> tmp(n);
    HIP_CHECK(hipMemcpyAsync(tmp.data(), psi.as<cx<T>>() + n * ixy, n * sizeof(cx<T>), hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
    for (std::size_t i = 0; i < n; ++i) {
      out[2 * i] = tmp[i].x;
      out[2 * i + 1] = tmp[i].y;
    }
  }
}

template <typename T>
void State<T>::bk_scattering(bool from_specular, int iz_specular) {
  const spo_hip_analysis& a = analysis;
  const cx<T>* src = psi.as<cx<T>>();
  spo_dev::Shape sh = s;
  int iz = a.iz_analysis;
  if (pending_half && (zr_variants.empty() || xy_variants.empty())) flush_pending();
  if (pending_half) {
    // The analysis plane at the analysis time without advancing the wave: T_Zr(dt/2) of every (irot, ixy) plane
    // with only row iz_analysis written out, then T_xy(dt/2) of those rows (layout of psi with one Z point).
    if (!ana_row.as<void>()) ana_row = Buffer(std::size_t(s.nr) * s.n_rot * s.n_xy * sizeof(cx<T>));
    cx<T>* row = ana_row.as<cx<T>>();
    timed("zr_row", [&] { run_zr(zr_variants[zr_pick], true, row, a.iz_analysis); });
    sh.nz = 1;
    sh.n_zr = s.nr;
    sh.nzpot = 0;
    sh.n_zr_pot = 0;
    timed("xy_row", [&] { run_xy(xy_variants[xy_pick], true, true, row, &sh); });
    src = row;
    iz = 0;
  }
  timed("bk_scattering", [&] {
    hipLaunchKernelGGL(spo_dev::bk_scattering_kernel<T>, dim3(a.n_v * a.n_rotation), dim3(kThreads),
                       std::size_t(s.n_xy) * sizeof(cx<double>), stream, src, sh, iz,
                       a.n_rotation, a.n_diffraction, a.n_states, rot_index.as<int>(), dif_slot.as<int>(),
                       radial_weight.as<double>(), shift_f_d.as<cx<double>>(), a.xy_scale, plan_x_d->plan,
                       plan_y_d->plan, bk.as<cx<double>>(),
                       static_cast<const cx<double>*>(from_specular ? spec.as<cx<double>>() : nullptr), iz_specular,
                       a.initial_state, initial_radial.as<double>(), a.dr);
  });
}

template <typename T>
void State<T>::energy_resolved_scattering() {
  flush_pending();
  const long block = long(s.n_zr) * s.n_rot;
  timed("energy_resolved", [&] {
    hipLaunchKernelGGL(spo_dev::energy_resolved_kernel<T>, dim3(blocks_for(block, 256), er_n_sites), dim3(256), 0,
                       stream, psi.as<cx<T>>(), block, er_sites.as<int>(), er_n_energies,
                       er_phase.as<cx<double>>(), er_dt, er_sums.as<cx<double>>());
  });
}

spo_dev::Shape make_shape(const spo_hip_shape* shape) {
  spo_dev::Shape s{};
  s.n_rot = shape->n_rot;
  s.nx = shape->nx;
  s.ny = shape->ny;
  s.n_xy = shape->nx * shape->ny;
  s.nr = shape->nr;
  s.nz = shape->nz;
  s.n_zr = shape->nr * shape->nz;
  s.nzsp = shape->nz_specular;
  s.nzpot = shape->nz_potential;
  s.n_zr_pot = shape->nz_potential * shape->nr;
  s.n_theta = shape->n_theta;
  s.n_phi = shape->n_phi;
  s.n_tp = shape->n_theta * shape->n_phi;
  s.n_rep = shape->n_representatives;
  s.ichn = shape->initial_channel;
  s.mj_max = shape->mj_max;
  s.n_blocks = 2 * shape->mj_max + 1;
  s.r_abs_first = shape->r_absorber_first;
  s.r_abs_last = shape->r_absorber_last;
  return s;
}

template <typename T>
std::unique_ptr<spo_hip_backend> create_state(const spo_hip_shape* shape, const spo_hip_tables* t,
                                              const spo_hip_analysis* a, const double* initial_specular) {
  auto b = std::make_unique<State<T>>();
  b->shape = *shape;
  b->s = make_shape(shape);
  const spo_dev::Shape& s = b->s;
  if (s.n_rot < 1 || s.nx < 2 || s.ny < 2 || s.nr < 2 || s.nz < 2 || s.nzsp < s.nz || s.nzpot < 0 || s.nzpot > s.nz ||
      s.n_theta < 1 || s.n_phi < 1 || s.n_rep < 1 || s.ichn < 0 || s.ichn >= s.n_rot || shape->n_operations < 1 ||
      shape->steps_per_analysis < 1 || s.r_abs_first < 0 || s.r_abs_last >= s.nr)
    throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_create: inconsistent shape");

  int device = 0;
  HIP_CHECK(hipGetDevice(&device));
  HIP_CHECK(hipDeviceGetAttribute(&b->max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, device));
  const std::size_t psi_values = std::size_t(s.n_zr) * s.n_rot * s.n_xy;
  const std::size_t exp_values = std::size_t(s.n_tp) * s.n_rep * s.n_zr_pot;
  std::size_t free_bytes = 0, total_bytes = 0;
  HIP_CHECK(hipMemGetInfo(&free_bytes, &total_bytes));
  const std::size_t need = (psi_values + exp_values) * sizeof(cx<T>) + (std::size_t(1) << 28);
  if (need > free_bytes)
    throw Status(SPO_HIP_E_NOT_SUPPORTED, "not enough device memory: need " + std::to_string(need >> 20) +
                                              " MiB, free " + std::to_string(free_bytes >> 20) + " MiB");
  HIP_CHECK(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
  HIP_CHECK(hipStreamCreateWithFlags(&b->side, hipStreamNonBlocking));
  HIP_CHECK(hipEventCreateWithFlags(&b->main_ready, hipEventDisableTiming));
  HIP_CHECK(hipEventCreateWithFlags(&b->spec_ready, hipEventDisableTiming));

  const std::size_t cT = sizeof(cx<T>), c16 = sizeof(cx<double>);
  // Zero slack behind the last site: the interaction kernels' phase-1 loads of a partial k step or of a column past
  // the interaction region read values past a site column without a branch (their products vanish: the matching
  // Legendre fragments are zero, or the column is never stored), at most 15 n_zr + 7 values past the end.
  const std::size_t psi_slack = 16 * std::size_t(s.n_zr) + 64;
  b->psi = Buffer((psi_values + psi_slack) * cT);
  HIP_CHECK(hipMemsetAsync(b->psi.template as<void>(), 0, (psi_values + psi_slack) * cT, b->stream));
  b->spec = upload(initial_specular, std::size_t(s.nr) * s.nzsp * c16);
  b->densities = Buffer(std::size_t(s.n_zr) * sizeof(double));
  b->partial = Buffer(std::size_t(s.n_zr) * s.n_xy * sizeof(double));
  b->plane = Buffer(std::size_t(s.n_rot) * s.n_xy * s.nr * c16);
  b->staging_values = std::max<std::size_t>(std::size_t(s.n_rot) * s.n_xy, std::size_t(4) << 20);
  b->staging = Buffer(b->staging_values * c16);

  // Kinetic factors with the forward and backward FFT scales folded in (multiplied in FP64, then stored).
  const double zr_f = t->fft_scale_z * t->fft_scale_r;
  const double zr_b = (1.0 / (s.nz * t->fft_scale_z)) * (1.0 / (s.nr * t->fft_scale_r));
  const double sp_b = (1.0 / (s.nzsp * t->fft_scale_z)) * (1.0 / (s.nr * t->fft_scale_r));
  const double xy_f = t->fft_scale_x * t->fft_scale_y;
  const double xy_b = (1.0 / (s.nx * t->fft_scale_x)) * (1.0 / (s.ny * t->fft_scale_y));
  auto fold = [](const double* p, std::size_t n, double f1, double f2) {
    std::vector<double> v(p, p + 2 * n);
    for (double& x : v) x = x * f1 * f2;
    return v;
  };
  const std::vector<double> zr_full_values = fold(t->zr_full, s.n_zr, zr_f, zr_b);
  const std::vector<double> zr_half_values = fold(t->zr_half, s.n_zr, zr_f, zr_b);
  {
    const auto sf = fold(t->specular_full, std::size_t(s.nr) * s.nzsp, zr_f, sp_b);
    const auto sh = fold(t->specular_half, std::size_t(s.nr) * s.nzsp, zr_f, sp_b);
    b->spec_lds = spo_dev::zr_plane_lds<double>(s.nzsp, s.nr);
    if (b->spec_lds <= static_cast<std::size_t>(b->max_lds))
      b->spec_fn = spo_dev::specular_plane(s.nzsp, s.nr, b->spec_shape);
    if (b->spec_fn) set_lds(b->spec_fn, b->max_lds);  // one kernel serves grids of many sizes
    auto specular_factor = [&](const std::vector<double>& f) {
      if (!b->spec_fn) return upload(f.data(), f.size() * sizeof(double));
      std::vector<double> p(f.size());
      for (int iz = 0; iz < s.nzsp; ++iz)
        for (int ir = 0; ir < s.nr; ++ir)
          for (int c = 0; c < 2; ++c)
            p[2 * (ir + std::size_t(s.nr) * iz) + c] = f[2 * spo_dev::zr_factor_order(b->spec_shape, iz, ir) + c];
      return upload(p.data(), p.size() * sizeof(double));
    };
    b->spec_full = specular_factor(sf);
    b->spec_half = specular_factor(sh);
    b->spec_beside = !b->spec_fn || s.nzsp * s.nr >= kSpecularBesidePoints;
    const auto xf = fold(t->xy_full, s.n_xy, xy_f, xy_b), xh = fold(t->xy_half, s.n_xy, xy_f, xy_b);
    b->xy_full = upload_complex<T>(xf.data(), s.n_xy);
    b->xy_full_lo = factor_lo<T>(xf.data(), s.n_xy);
    b->xy_half = upload_complex<T>(xh.data(), s.n_xy);
    b->xy_half_lo = factor_lo<T>(xh.data(), s.n_xy);
  }
  b->rot_half = upload_complex<T>(t->rotation_half, std::size_t(s.n_rot) * s.nr);
  b->rot_lo = factor_lo<T>(t->rotation_half, std::size_t(s.n_rot) * s.nr);
  {
    // (irot, ir) -> (ir, irot), ir fastest, for the MFMA interaction kernel
    std::vector<double> rt(2 * std::size_t(s.n_rot) * s.nr);
    for (int ir = 0; ir < s.nr; ++ir)
      for (int irot = 0; irot < s.n_rot; ++irot)
        for (int c = 0; c < 2; ++c)
          rt[2 * (ir + std::size_t(s.nr) * irot) + c] = t->rotation_half[2 * (irot + std::size_t(s.n_rot) * ir) + c];
    b->rot_half_t = upload_complex<T>(rt.data(), rt.size() / 2);
    b->rot_lo_t = factor_lo<T>(rt.data(), rt.size() / 2);
  }
  b->before = upload_complex<T>(t->before_interaction, std::size_t(s.n_rot) * s.nr);
  b->gas_step = upload_complex<T>(t->gas_phase_step, std::size_t(s.n_rot) * s.nr);
  b->before_lo = factor_lo<T>(t->before_interaction, std::size_t(s.n_rot) * s.nr);
  b->gas_step_lo = factor_lo<T>(t->gas_phase_step, std::size_t(s.n_rot) * s.nr);
  b->spec_gas = upload(t->specular_gas_phase, std::size_t(s.nr) * c16);
  b->z_opt = upload_real<T>(t->z_optical, s.nz);
  b->r_opt_d = upload(t->r_optical, std::size_t(s.nr) * sizeof(double));
  b->z_spec_opt = upload(t->z_specular_optical, std::size_t(s.nzsp) * sizeof(double));
  b->shift_f = upload_complex<T>(t->shift_forward, s.n_xy);
  b->shift_b = upload_complex<T>(t->shift_backward, s.n_xy);
  b->shift_f_lo = factor_lo<T>(t->shift_forward, s.n_xy);
  b->shift_b_lo = factor_lo<T>(t->shift_backward, s.n_xy);
  b->shift_f_d = upload(t->shift_forward, std::size_t(s.n_xy) * c16);
  b->s2sc = upload_complex<T>(t->specular_to_scattering, s.n_xy);
  b->s2sc_d = upload(t->specular_to_scattering, std::size_t(s.n_xy) * c16);
  b->sc2s_d = upload(t->scattering_to_specular, std::size_t(s.n_xy) * c16);

  // Angular transform tables (the Legendre matrix stays FP64 and is rounded at use).
  std::vector<int> offsets(s.n_blocks), rot_block(s.n_rot, -1);
  int total = 0, covered = 0;
  for (int blk = 0; blk < s.n_blocks; ++blk) {
    offsets[blk] = total;
    const int first = t->block_first[blk], size = t->block_size[blk];
    if (first < 0 || size < 0 || first + size > s.n_rot) throw Status(SPO_HIP_E_ARGUMENT, "bad mJ block");
    for (int j = 0; j < size; ++j) rot_block[first + j] = blk;
    total += s.n_theta * size;
    covered += size;
  }
  if (covered != s.n_rot) throw Status(SPO_HIP_E_ARGUMENT, "the mJ blocks do not cover the basis");
  if (2 * s.mj_max + 1 > s.n_phi) throw Status(SPO_HIP_E_ARGUMENT, "nphi < 2 MJMax + 1");
  b->legendre = upload(t->legendre, std::size_t(total) * sizeof(double));
  b->legendre_t = upload_real<T>(t->legendre, std::size_t(total));
  b->legendre_size = total;
  b->block_first = upload(t->block_first, std::size_t(s.n_blocks) * sizeof(int));
  b->block_size = upload(t->block_size, std::size_t(s.n_blocks) * sizeof(int));
  b->block_offset = upload(offsets.data(), offsets.size() * sizeof(int));
  b->rot_block = upload(rot_block.data(), rot_block.size() * sizeof(int));
  for (int ixy = 0; ixy < s.n_xy; ++ixy)
    if (t->representative_of[ixy] < 0 || t->representative_of[ixy] >= s.n_rep || t->operation_of[ixy] < 0 ||
        t->operation_of[ixy] >= shape->n_operations)
      throw Status(SPO_HIP_E_ARGUMENT, "bad symmetry map");
  for (int k = 0; k < s.n_phi * shape->n_operations; ++k)
    if (t->phi_index[k] < 0 || t->phi_index[k] >= s.n_phi) throw Status(SPO_HIP_E_ARGUMENT, "bad phi map");
  b->rep_of = upload(t->representative_of, std::size_t(s.n_xy) * sizeof(int));
  b->op_of = upload(t->operation_of, std::size_t(s.n_xy) * sizeof(int));
  b->phi_index = upload(t->phi_index, std::size_t(s.n_phi) * shape->n_operations * sizeof(int));
  b->exp_table = upload_complex<T>(t->exp_potential, exp_values);

  // Analysis (FP64).
  b->analysis = *a;
  if (a->n_states != a->n_rotation * a->n_diffraction || a->n_v < 1 || a->n_energies < 1 || a->iz_analysis < 0 ||
      a->iz_analysis >= s.nz || a->initial_state < 0 || a->initial_state >= a->n_states || a->n_diffraction > s.n_xy)
    throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_create: inconsistent analysis");
  for (int k = 0; k < a->n_rotation; ++k)
    if (a->rotation_index[k] < 0 || a->rotation_index[k] >= s.n_rot) throw Status(SPO_HIP_E_ARGUMENT, "bad rotation index");
  for (int k = 0; k < a->n_diffraction; ++k)
    if (a->diffraction_slot[k] < 0 || a->diffraction_slot[k] >= s.n_xy) throw Status(SPO_HIP_E_ARGUMENT, "bad slot");
  b->rot_index = upload(a->rotation_index, std::size_t(a->n_rotation) * sizeof(int));
  b->dif_slot = upload(a->diffraction_slot, std::size_t(a->n_diffraction) * sizeof(int));
  b->radial_weight = upload(a->radial_weight, std::size_t(s.nr) * a->n_rotation * a->n_v * sizeof(double));
  b->initial_radial = upload(a->initial_radial, std::size_t(s.nr) * a->n_v * sizeof(double));
  b->energies = upload(a->total_energy_hartree, std::size_t(a->n_energies) * sizeof(double));
  b->analysis.rotation_index = nullptr;
  b->analysis.diffraction_slot = nullptr;
  b->analysis.radial_weight = nullptr;
  b->analysis.initial_radial = nullptr;
  b->analysis.total_energy_hartree = nullptr;
  b->bk = Buffer(std::size_t(a->n_states) * a->n_v * c16);
  const std::size_t n_sums = std::size_t(a->n_states) * a->n_v * a->n_energies;
  b->sums = Buffer(n_sums * c16);
  HIP_CHECK(hipMemsetAsync(b->sums.template as<void>(), 0, n_sums * c16, b->stream));

  // Plans, tile widths and the kernels for this shape.
  b->plan_z = std::make_unique<DevicePlan<T>>(s.nz);
  b->plan_r = std::make_unique<DevicePlan<T>>(s.nr);
  b->plan_x = std::make_unique<DevicePlan<T>>(s.nx);
  b->plan_y = std::make_unique<DevicePlan<T>>(s.ny);
  b->plan_phi = std::make_unique<DevicePlan<T>>(s.n_phi);
  b->plan_r_d = std::make_unique<DevicePlan<double>>(s.nr);
  b->plan_zsp = std::make_unique<DevicePlan<double>>(s.nzsp);
  b->plan_x_d = std::make_unique<DevicePlan<double>>(s.nx);
  b->plan_y_d = std::make_unique<DevicePlan<double>>(s.ny);
  const std::size_t lds_limit = static_cast<std::size_t>(b->max_lds);
  // T_Zr: the register-pass kernel where the axes are products of two radices and the plane fits in LDS, else the
  // run-time engine on the plane, else lines.
  if (spo_dev::zr_plane_lds<T>(s.nz, s.nr) <= lds_limit) b->zr_variants = spo_dev::zr_variants<T>(s.nz, s.nr);
  if (!b->zr_variants.empty()) {
    for (const Variant& v : b->zr_variants) set_lds(v.fn, lds_limit);  // one kernel serves planes of many sizes
  } else if (std::size_t(s.n_zr) * cT <= lds_limit) {
    b->zr_fused = true;
    b->zr_lds = std::size_t(s.n_zr) * cT;
    set_lds(reinterpret_cast<const void*>(spo_dev::zr_plane_kernel<T>), b->zr_lds);
  }
  b->upload_zr_factors(zr_full_values, zr_half_values, b->zr_variants.empty() ? nullptr : &b->zr_variants[0].zr);
  // T_xy.
  for (const Variant& v : spo_dev::xy_reg_variants<T>(s.nx, s.ny))
    if (v.lds <= lds_limit) b->xy_variants.push_back(v);
  if (!b->xy_variants.empty()) {
    for (const Variant& v : b->xy_variants) set_lds(v.fn, v.lds);
  } else {
    b->xy_c = std::max(1, std::min(64, 4096 / s.n_xy));
    b->xy_lds = std::size_t(b->xy_c) * s.n_xy * cT;
    if (b->xy_lds > lds_limit) throw Status(SPO_HIP_E_NOT_SUPPORTED, "the (x, y) tile does not fit in LDS");
    set_lds(reinterpret_cast<const void*>(spo_dev::xy_kernel<T>), b->xy_lds);
  }
  // Interaction tile: the largest power of two of columns (at most 32) whose LDS fits in 80 KiB (two per CU).
  b->v_fn = s.n_theta <= spo_dev::kMaxTheta ? spo_dev::interaction_ct_symbol<T>(s.n_phi) : nullptr;
  auto v_bytes = [&](int c) {
    return b->v_fn ? spo_dev::interaction_ct_lds<T>(c, s.n_theta, s.n_phi, b->legendre_size)
                   : std::size_t(c) * (s.n_rot + s.n_tp) * cT;
  };
  int p2 = 1;
  while (p2 < 32 && v_bytes(2 * p2) <= 81920) p2 *= 2;
  b->v_c = p2;
  b->v_lds = v_bytes(p2);
  if (b->v_lds > lds_limit) throw Status(SPO_HIP_E_NOT_SUPPORTED, "an angular column does not fit in LDS");
  set_lds(b->v_fn ? b->v_fn : reinterpret_cast<const void*>(spo_dev::interaction_kernel<T>), b->v_lds);
  // Interaction with the theta contractions on MFMA: Legendre fragments in lane order, XCD-grouped site order. The
  // default is interaction_kernel_inplace where its conditions hold (an instantiated phi length, at most 16 theta
  // points and 16 J per block, 32-bit offsets within a site, one Legendre matrix for m and -m), followed in the list by
  // the kernels below for the launch tuner.
  // SPO_HIP_INTERACTION selects one of the others for comparisons: "buf" (the buffer-addressed MFMA kernel where its
  // shape conditions hold, else "mfma"), "mfma" (MFMA contractions, fused register phi step), "mfma_staged" (MFMA
  // contractions, staged LDS phi FFTs), "lds" (contractions on the vector units).
  {
    const char* env = std::getenv("SPO_HIP_INTERACTION");
    const std::string choice = env ? env : (sizeof(T) == 8 ? "mfma" : "buf");
    if (choice != "buf" && choice != "mfma" && choice != "mfma_staged" && choice != "lds")
      throw Status(SPO_HIP_E_ARGUMENT, "SPO_HIP_INTERACTION must be buf, mfma, mfma_staged or lds");
    const bool fused = (choice == "mfma" || choice == "buf") && s.n_theta <= 16;
    // SPO_HIP_CONTRACTION=bf16x3: the complex64 theta contractions as split-BF16x3 products (buffer kernel, 48-point
    // phi step); the default "fp32" is FP32 MFMA with the bf16 low part of L. FP64 ignores it.
    const char* contraction = std::getenv("SPO_HIP_CONTRACTION");
    if (contraction && std::string(contraction) != "fp32" && std::string(contraction) != "bf16x3")
      throw Status(SPO_HIP_E_ARGUMENT, "SPO_HIP_CONTRACTION must be fp32 or bf16x3");
    const bool bf16x3 = sizeof(T) == 4 && contraction && std::string(contraction) == "bf16x3";
    std::vector<Variant> variants;
    for (const Variant& v : spo_dev::interaction_mfma_variants<T>(s.n_phi, s.n_theta, fused))
      if (v.lds <= lds_limit) variants.push_back(v);
    // phi lengths with a buffer-kernel instantiation only (the reduced-JMax batch members' 28 and 40 points)
    const bool buf_candidate =
        choice == "buf" && !spo_dev::interaction_buf_variants<T>(s.n_phi, s.n_theta, s.n_blocks, bf16x3).empty();
    int longest_block = 0;
    for (int blk = 0; blk < s.n_blocks; ++blk) longest_block = std::max(longest_block, t->block_size[blk]);
    std::vector<Variant> in_place;
    if (!env && !bf16x3 && longest_block <= 16 && std::size_t(s.n_zr) * s.n_rot * cT < (std::size_t(1) << 31))
      for (const Variant& v : spo_dev::interaction_inplace_variants<T>(s.n_phi, s.n_theta, long(s.n_zr_pot) * s.n_xy))
        if (v.lds <= lds_limit) in_place.push_back(v);
    if ((!variants.empty() || buf_candidate || !in_place.empty()) && choice != "lds") {
      const int n_tt = (s.n_theta + 15) / 16, k_bwd = (s.n_theta + 3) / 4;
      std::vector<int> fo(s.n_blocks), bo(s.n_blocks);
      int nf = 0, nbw = 0, max_nb = 0;
      for (int blk = 0; blk < s.n_blocks; ++blk) {
        const int nb = t->block_size[blk];
        fo[blk] = nf;
        nf += n_tt * ((nb + 3) / 4);
        bo[blk] = nbw;
        nbw += ((nb + 15) / 16) * k_bwd;
        max_nb = std::max(max_nb, nb);
      }
      std::vector<double> ff(64 * std::size_t(std::max(nf, 1)), 0.0), fb(64 * std::size_t(std::max(nbw, 1)), 0.0);
      for (int blk = 0; blk < s.n_blocks; ++blk) {
        const int nb = t->block_size[blk], ks = (nb + 3) / 4;
        const double* L = t->legendre + offsets[blk];  // (theta, J)
        for (int lane = 0; lane < 64; ++lane) {
          const int i = lane % 16, kk = lane / 16;
          for (int tt = 0; tt < n_tt; ++tt)
            for (int k = 0; k < ks; ++k) {
              const int th = 16 * tt + i, j = 4 * k + kk;
              if (th < s.n_theta && j < nb) ff[64 * std::size_t(fo[blk] + tt * ks + k) + lane] = L[th * nb + j];
            }
          for (int jt = 0; jt < (nb + 15) / 16; ++jt)
            for (int k = 0; k < k_bwd; ++k) {
              const int th = 4 * k + kk, j = 16 * jt + i;
              if (th < s.n_theta && j < nb) fb[64 * std::size_t(bo[blk] + jt * k_bwd + k) + lane] = L[th * nb + j];
            }
        }
      }
      std::vector<int> order(s.n_xy);
      for (int i = 0; i < s.n_xy; ++i) order[i] = i;
      if (s.n_xy % 8 == 0) {
        std::vector<int> sorted(order);
        std::stable_sort(sorted.begin(), sorted.end(), [&](int x, int y) {
          return t->representative_of[x] < t->representative_of[y];
        });
        const int per = s.n_xy / 8;
        for (int x = 0; x < 8; ++x)
          for (int k = 0; k < per; ++k) order[8 * k + x] = sorted[per * x + k];
      }
      b->frag_fwd = upload_real<T>(ff.data(), ff.size());
      b->frag_bwd = upload_real<T>(fb.data(), fb.size());
      b->fwd_offset = upload(fo.data(), fo.size() * sizeof(int));
      b->bwd_offset = upload(bo.data(), bo.size() * sizeof(int));
      b->site_order = upload(order.data(), order.size() * sizeof(int));
      b->max_jt = (max_nb + 15) / 16;
      b->frag_fwd_count = nf;
      b->frag_bwd_count = nbw;
      auto low_fragments = [&] {
        if (sizeof(T) != 4 || b->lo_fwd.template as<void>()) return;
        // bf16 fragments of a function of L, lane (i, q) element t = contraction row 4 t + q
        // (legendre_low_product): forward A = L (theta = i, J = row), backward A = L^T (J = i, theta = row).
        auto bf16 = [](double x) -> std::uint16_t {
          const float f = static_cast<float>(x);
          std::uint32_t u;
          std::memcpy(&u, &f, 4);
          u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even (the values are finite and small)
          return static_cast<std::uint16_t>(u >> 16);
        };
        auto bf16_value = [&](double x) {
          const std::uint32_t u = std::uint32_t(bf16(x)) << 16;
          float f;
          std::memcpy(&f, &u, 4);
          return static_cast<double>(f);
        };
        auto fragments = [&](auto&& piece, Buffer& fwd, Buffer& bwd) {
          std::vector<std::uint16_t> lf(256 * std::size_t(s.n_blocks), 0), lb(256 * std::size_t(s.n_blocks), 0);
          for (int blk = 0; blk < s.n_blocks; ++blk) {
            const int nb = t->block_size[blk];
            const double* L = t->legendre + offsets[blk];  // (theta, J)
            for (int lane = 0; lane < 64; ++lane)
              for (int e = 0; e < 4; ++e) {
                const int i = lane % 16, q = lane / 16, row = 4 * e + q;
                if (i < s.n_theta && row < nb) lf[256 * std::size_t(blk) + 4 * lane + e] = bf16(piece(L[i * nb + row]));
                if (row < s.n_theta && i < nb) lb[256 * std::size_t(blk) + 4 * lane + e] = bf16(piece(L[row * nb + i]));
              }
          }
          fwd = upload(lf.data(), lf.size() * sizeof(std::uint16_t));
          bwd = upload(lb.data(), lb.size() * sizeof(std::uint16_t));
        };
        if (bf16x3) {
          // split-BF16x3: A_hi = bf16(L), A_lo = bf16(L - A_hi)
          fragments([&](double l) { return l; }, b->hi_fwd, b->hi_bwd);
          fragments([&](double l) { return l - bf16_value(l); }, b->lo_fwd, b->lo_bwd);
        } else {
          // the low part L - float(L) of the FP32 contraction
          fragments([](double l) { return l - static_cast<double>(static_cast<float>(l)); }, b->lo_fwd, b->lo_bwd);
        }
      };
      // The buffer-addressed kernel where its shape conditions hold: one theta tile, blocks of at most 16 J, a
      // site column addressable with 32-bit offsets.
      if (choice == "buf" && s.n_theta <= 16 && max_nb <= 16 &&
          std::size_t(s.n_zr) * s.n_rot * cT < (std::size_t(1) << 31)) {
        std::vector<Variant> buf;
        for (const Variant& v : spo_dev::interaction_buf_variants<T>(s.n_phi, s.n_theta, s.n_blocks, bf16x3))
          if (v.lds <= lds_limit) buf.push_back(v);
        if (bf16x3 && buf.empty())
          throw Status(SPO_HIP_E_NOT_SUPPORTED, "SPO_HIP_CONTRACTION=bf16x3: instantiated for the 48-point phi step only");
        if (!buf.empty()) {
          // Sign-split rotation factors, 16 zero rows past the last irot (the loads of a block's rows past the
          // basis stay inside the table).
          std::vector<spo_dev::RotEntry<T>> pm(2 * (std::size_t(s.n_rot) + 16) * s.nr, spo_dev::RotEntry<T>{});
          for (int irot = 0; irot < s.n_rot; ++irot)
            for (int ir = 0; ir < s.nr; ++ir) {
              const double x = t->rotation_half[2 * (irot + std::size_t(s.n_rot) * ir)];
              const double y = t->rotation_half[2 * (irot + std::size_t(s.n_rot) * ir) + 1];
              set_rot_entries(pm.data() + spo_dev::rot_pm_index(irot, ir, s.nr, 0), x, y);
            }
          b->rot_pm = upload(pm.data(), pm.size() * sizeof(spo_dev::RotEntry<T>));
          low_fragments();
          variants = buf;
        }
      }
      if (!in_place.empty() && b->build_angular_plan(t, offsets, in_place[0].r1, in_place[0].r2)) {
        low_fragments();
        variants.insert(variants.begin(), in_place.begin(), in_place.end());
      }
      if (!variants.empty()) {  // else the kernels chosen above (v_fn or the run-time-shaped one) stay
        b->v_variants = variants;
        b->v_c = 8;
        for (const Variant& v : variants) set_lds(v.fn, lds_limit);
      }
    }
  }
  set_lds(reinterpret_cast<const void*>(spo_dev::lines_fft_kernel<T>), 65536);
  set_lds(reinterpret_cast<const void*>(spo_dev::lines_fft_kernel<double>), 65536);
  set_lds(reinterpret_cast<const void*>(spo_dev::bk_scattering_kernel<T>), std::size_t(s.n_xy) * c16);
  // SPO_HIP_MERGE_HALF_STEPS=1: merged half steps between analysis steps (see spo_hip_backend::merge_halves).
  if (const char* m = std::getenv("SPO_HIP_MERGE_HALF_STEPS")) {
    const std::string v = m;
    if (v != "0" && v != "1") throw Status(SPO_HIP_E_ARGUMENT, "SPO_HIP_MERGE_HALF_STEPS must be 0 or 1");
    b->merge_halves = v == "1";
  }
  HIP_CHECK(hipStreamSynchronize(b->stream));
  b->tune();
  if (b->zr_pick != 0)
    b->upload_zr_factors(zr_full_values, zr_half_values, &b->zr_variants[b->zr_pick].zr);
  return b;
}

}  // namespace

extern "C" {

const char* spo_hip_last_error(void) { return g_error.c_str(); }

int spo_hip_device_count(int* count) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
  *count = n;
  return SPO_HIP_OK;
}

int spo_hip_create(const spo_hip_shape* shape, const spo_hip_tables* t, const spo_hip_analysis* a,
                   const double* initial_specular, spo_hip_backend** out) {
  return guarded([&] {
    if (!shape || !t || !a || !initial_specular || !out) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_create: NULL argument");
    *out = nullptr;
    require_device();
    std::unique_ptr<spo_hip_backend> b;
    if (shape->precision == SPO_HIP_FP64)
      b = create_state<double>(shape, t, a, initial_specular);
    else if (shape->precision == SPO_HIP_MIXED)
      b = create_state<float>(shape, t, a, initial_specular);
    else
      throw Status(SPO_HIP_E_NOT_SUPPORTED, "unsupported precision");
    *out = b.release();
  });
}

int spo_hip_destroy(spo_hip_backend* b) {
  return guarded([&] {
    if (b && b->batches > 0)
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_destroy: the backend is still a member of a batch (destroy the batch first)");
    delete b;
  });
}

int spo_hip_upload_wave(spo_hip_backend* b, const double* scattering, const double* specular) {
  return guarded([&] {
    if (scattering) b->upload_wave(scattering);
    if (specular)
      HIP_CHECK(hipMemcpyAsync(b->spec.as<void>(), specular, std::size_t(b->s.nr) * b->s.nzsp * sizeof(cx<double>),
                               hipMemcpyHostToDevice, b->stream));
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

int spo_hip_download_wave(spo_hip_backend* b, double* scattering, double* specular) {
  return guarded([&] {
    if (scattering) b->download_wave(scattering);
    if (specular)
      HIP_CHECK(hipMemcpyAsync(specular, b->spec.as<void>(), std::size_t(b->s.nr) * b->s.nzsp * sizeof(cx<double>),
                               hipMemcpyDeviceToHost, b->stream));
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

int spo_hip_kinetic_and_potential(spo_hip_backend* b, int half_step, int kinetic_only) {
  return guarded([&] {
    b->flush_pending();
    b->kinetic_and_potential(half_step != 0, kinetic_only != 0);
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

}  // extern "C"

namespace {

// The blocks of one analysis step, [T/2 V], (n - 1) [T V], [T/2], enqueued on the backend's streams.
void enqueue_blocks(spo_hip_backend* b) {
  // Merged half steps only on eager steps (a captured graph replays the plain schedule).
  const bool merge = b->merge_halves && !b->use_graph;
  if (!merge) b->flush_pending();
  b->step_block(true, merge && b->pending_half ? 2 : 1, false);
  for (int k = 1; k < b->shape.steps_per_analysis; ++k) b->kinetic_and_potential(false, false);
  if (merge) {
    b->step_block(true, 0, true);  // the specular grid's trailing half step; the scattering grid's waits
    b->pending_half = true;
  } else {
    b->kinetic_and_potential(true, true);
  }
}

// One analysis step on the backend's stream: the blocks, or in graph mode the captured step (captured here the
// first time).
void enqueue_analysis_step(spo_hip_backend* b) {
  if (!b->use_graph) {
    enqueue_blocks(b);
    return;
  }
  if (!b->step_graph) {
    hipGraph_t graph = nullptr;
    HIP_CHECK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    enqueue_blocks(b);
    HIP_CHECK(hipStreamEndCapture(b->stream, &graph));
    const hipError_t e = hipGraphInstantiate(&b->step_graph, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    HIP_CHECK(e);
  }
  HIP_CHECK(hipGraphLaunch(b->step_graph, b->stream));
}

}  // namespace

extern "C" {

int spo_hip_graph_enable(spo_hip_backend* b, int on) {
  return guarded([&] {
    if (!b) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_graph_enable: NULL backend");
    if (on && b->profiling) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_graph_enable: kernel timing is on");
    b->flush_pending();
    HIP_CHECK(hipStreamSynchronize(b->stream));
    if (b->step_graph) {
      HIP_CHECK(hipGraphExecDestroy(b->step_graph));
      b->step_graph = nullptr;
    }
    b->use_graph = on != 0;
  });
}

int spo_hip_propagate_analysis_step(spo_hip_backend* b) {
  return guarded([&] {
    enqueue_analysis_step(b);
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

int spo_hip_propagate_batch(spo_hip_backend* const* backends, int n) {
  return guarded([&] {
    if (n < 0 || (n > 0 && !backends)) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_propagate_batch: bad arguments");
    for (int i = 0; i < n; ++i) {
      if (!backends[i]) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_propagate_batch: NULL backend");
      for (int j = 0; j < i; ++j)
        if (backends[j] == backends[i]) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_propagate_batch: a backend twice");
    }
    // Block r of every run's schedule [T/2 V], (n - 1) [T V], [T/2], round robin over the runs: each run's launches
    // stay in its own order on its own streams, and the runs' kernels overlap where one alone does not fill the GPU.
    // Runs in graph mode launch their captured step; the others' blocks go round robin. A batch step runs the plain
    // schedule: a pending half step is applied first.
    for (int i = 0; i < n; ++i) backends[i]->flush_pending();
    for (int i = 0; i < n; ++i)
      if (backends[i]->use_graph) enqueue_analysis_step(backends[i]);
    int longest = 0;
    for (int i = 0; i < n; ++i)
      if (!backends[i]->use_graph) longest = std::max(longest, backends[i]->shape.steps_per_analysis + 1);
    for (int r = 0; r < longest; ++r)
      for (int i = 0; i < n; ++i) {
        spo_hip_backend* b = backends[i];
        const int blocks = b->shape.steps_per_analysis + 1;
        if (b->use_graph || r >= blocks) continue;
        b->kinetic_and_potential(r == 0 || r == blocks - 1, r == blocks - 1);
      }
    for (int i = 0; i < n; ++i) HIP_CHECK(hipStreamSynchronize(backends[i]->stream));
  });
}

}  // extern "C"

// A batch of backends stepped together through one hipGraph: at its first step, block r of every member's schedule
// is enqueued round robin on the members' streams (as spo_hip_propagate_batch does) inside one capture that starts
// on the first member's stream, forks to the others through an event and joins them back; later steps replay the
// graph with one launch. Each member's launches keep their order on its own streams, so a member's results are
// bitwise those of the member stepped alone.
struct spo_hip_batch {
  std::vector<spo_hip_backend*> members;
  hipEvent_t fork = nullptr;
  std::vector<hipEvent_t> joins;
  hipGraphExec_t graph = nullptr;
  ~spo_hip_batch() {
    if (graph) (void)hipGraphExecDestroy(graph);
    if (fork) (void)hipEventDestroy(fork);
    for (hipEvent_t e : joins) (void)hipEventDestroy(e);
    for (spo_hip_backend* b : members) --b->batches;
  }
};

namespace {

void enqueue_round_robin(spo_hip_backend* const* backends, int n) {
  int longest = 0;
  for (int i = 0; i < n; ++i) longest = std::max(longest, backends[i]->shape.steps_per_analysis + 1);
  for (int r = 0; r < longest; ++r)
    for (int i = 0; i < n; ++i) {
      spo_hip_backend* b = backends[i];
      const int blocks = b->shape.steps_per_analysis + 1;
      if (r >= blocks) continue;
      b->kinetic_and_potential(r == 0 || r == blocks - 1, r == blocks - 1);
    }
}

}  // namespace

extern "C" {

int spo_hip_batch_create(spo_hip_backend* const* backends, int n, spo_hip_batch** out) {
  return guarded([&] {
    if (!out || n < 1 || !backends) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_batch_create: bad arguments");
    *out = nullptr;
    for (int i = 0; i < n; ++i) {
      if (!backends[i]) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_batch_create: NULL backend");
      if (backends[i]->profiling) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_batch_create: kernel timing is on");
      for (int j = 0; j < i; ++j)
        if (backends[j] == backends[i]) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_batch_create: a backend twice");
    }
    for (int i = 0; i < n; ++i) backends[i]->flush_pending();
    auto batch = std::make_unique<spo_hip_batch>();
    HIP_CHECK(hipEventCreateWithFlags(&batch->fork, hipEventDisableTiming));
    for (int i = 0; i < n; ++i) {
      hipEvent_t e = nullptr;
      HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      batch->joins.push_back(e);
    }
    for (int i = 0; i < n; ++i) {
      batch->members.push_back(backends[i]);
      ++backends[i]->batches;
    }
    *out = batch.release();
  });
}

int spo_hip_batch_step(spo_hip_batch* batch) {
  return guarded([&] {
    if (!batch) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_batch_step: NULL batch");
    std::vector<spo_hip_backend*>& m = batch->members;
    hipStream_t origin = m[0]->stream;
    for (spo_hip_backend* b : m)
      if (b->profiling) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_batch_step: kernel timing is on");
    for (spo_hip_backend* b : m) {  // the graph replays the plain schedule: pending half steps are applied first
      if (!b->pending_half) continue;
      b->flush_pending();
      HIP_CHECK(hipStreamSynchronize(b->stream));
    }
    if (!batch->graph) {
      // Every member's earlier work is complete before the capture (the members' streams join the capture only
      // through the fork event).
      for (spo_hip_backend* b : m) HIP_CHECK(hipStreamSynchronize(b->stream));
      hipGraph_t graph = nullptr;
      HIP_CHECK(hipStreamBeginCapture(origin, hipStreamCaptureModeThreadLocal));
      HIP_CHECK(hipEventRecord(batch->fork, origin));
      for (std::size_t i = 1; i < m.size(); ++i) HIP_CHECK(hipStreamWaitEvent(m[i]->stream, batch->fork, 0));
      enqueue_round_robin(m.data(), static_cast<int>(m.size()));
      for (std::size_t i = 1; i < m.size(); ++i) {
        HIP_CHECK(hipEventRecord(batch->joins[i], m[i]->stream));
        HIP_CHECK(hipStreamWaitEvent(origin, batch->joins[i], 0));
      }
      HIP_CHECK(hipStreamEndCapture(origin, &graph));
      const hipError_t e = hipGraphInstantiate(&batch->graph, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      HIP_CHECK(e);
    }
    HIP_CHECK(hipGraphLaunch(batch->graph, origin));
    HIP_CHECK(hipStreamSynchronize(origin));
  });
}

int spo_hip_batch_destroy(spo_hip_batch* batch) {
  return guarded([&] {
    if (!batch) return;
    HIP_CHECK(hipStreamSynchronize(batch->members[0]->stream));
    delete batch;
  });
}

int spo_hip_get_specular(spo_hip_backend* b, double* out) {
  return guarded([&] {
    HIP_CHECK(hipMemcpyAsync(out, b->spec.as<void>(), std::size_t(b->s.nr) * b->s.nzsp * sizeof(cx<double>),
                             hipMemcpyDeviceToHost, b->stream));
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

int spo_hip_get_z_plane(spo_hip_backend* b, int iz, double* out) {
  return guarded([&] {
    const spo_dev::Shape& s = b->s;
    if (iz < 0 || iz >= s.nz) throw Status(SPO_HIP_E_ARGUMENT, "z plane index out of range");
    b->z_plane(iz);
    const long n = long(s.n_rot) * s.n_xy * s.nr;
    HIP_CHECK(hipMemcpyAsync(out, b->plane.as<void>(), n * sizeof(cx<double>), hipMemcpyDeviceToHost, b->stream));
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

int spo_hip_block_densities(spo_hip_backend* b, double* out) {
  return guarded([&] {
    b->block_densities();
    HIP_CHECK(hipMemcpyAsync(out, b->densities.as<void>(), std::size_t(b->s.n_zr) * sizeof(double),
                             hipMemcpyDeviceToHost, b->stream));
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

int spo_hip_site_column(spo_hip_backend* b, int ixy, double* out) {
  return guarded([&] {
    if (ixy < 0 || ixy >= b->s.n_xy) throw Status(SPO_HIP_E_ARGUMENT, "site index out of range");
    b->site_column(ixy, out);
  });
}

int spo_hip_analyse(spo_hip_backend* b, int surface_fixed, int iz_specular, double t, double* coefficients) {
  return guarded([&] { b->analyse(surface_fixed, iz_specular, t, coefficients); });
}

int spo_hip_get_s_sums(spo_hip_backend* b, double* out) {
  return guarded([&] {
    const spo_hip_analysis& a = b->analysis;
    const std::size_t n = std::size_t(a.n_states) * a.n_v * a.n_energies;
    HIP_CHECK(hipMemcpyAsync(out, b->sums.as<void>(), n * sizeof(cx<double>), hipMemcpyDeviceToHost, b->stream));
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

int spo_hip_energy_resolved_start(spo_hip_backend* b, int n_sites, const int* site_ixy, int n_energies,
                                  double analysis_time_step) {
  return guarded([&] {
    if (n_sites < 1 || n_energies < 1 || !site_ixy)
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_energy_resolved_start: no sites or no energies");
    for (int i = 0; i < n_sites; ++i)
      if (site_ixy[i] < 0 || site_ixy[i] >= b->s.n_xy) throw Status(SPO_HIP_E_ARGUMENT, "site outside the (x, y) grid");
    const std::size_t block = std::size_t(b->s.n_zr) * b->s.n_rot;
    const std::size_t spec_n = std::size_t(b->s.nzsp) * b->s.nr;
    b->er_sums = Buffer(std::size_t(n_sites) * n_energies * block * sizeof(cx<double>));
    b->er_specular = Buffer(std::size_t(n_energies) * spec_n * sizeof(cx<double>));
    b->er_sites = upload(site_ixy, std::size_t(n_sites) * sizeof(int));
    b->er_phase = Buffer(std::size_t(n_energies) * sizeof(cx<double>));
    b->er_n_sites = n_sites;
    b->er_n_energies = n_energies;
    b->er_dt = analysis_time_step;
    HIP_CHECK(hipMemsetAsync(b->er_sums.as<void>(), 0, std::size_t(n_sites) * n_energies * block * sizeof(cx<double>),
                             b->stream));
    HIP_CHECK(hipMemsetAsync(b->er_specular.as<void>(), 0, std::size_t(n_energies) * spec_n * sizeof(cx<double>),
                             b->stream));
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

int spo_hip_energy_resolved_add(spo_hip_backend* b, const double* phase_factors) {
  return guarded([&] {
    if (b->er_n_sites == 0) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_energy_resolved_add before _start");
    HIP_CHECK(hipMemcpyAsync(b->er_phase.as<void>(), phase_factors, std::size_t(b->er_n_energies) * sizeof(cx<double>),
                             hipMemcpyHostToDevice, b->stream));
    b->energy_resolved_scattering();
    const int spec_n = b->s.nzsp * b->s.nr;
    b->timed("energy_resolved_specular", [&] {
      hipLaunchKernelGGL(spo_dev::energy_resolved_specular_kernel, dim3(blocks_for(spec_n, 256)), dim3(256), 0,
                         b->stream, b->spec.as<cx<double>>(), spec_n, b->er_n_energies, b->er_phase.as<cx<double>>(),
                         b->er_dt, b->er_specular.as<cx<double>>());
    });
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

int spo_hip_energy_resolved_read(spo_hip_backend* b, double* sums, double* specular_sums) {
  return guarded([&] {
    if (b->er_n_sites == 0) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_energy_resolved_read before _start");
    const std::size_t n_zr = b->s.n_zr, n_rot = b->s.n_rot, block = n_zr * n_rot;
    const std::size_t pairs = std::size_t(b->er_n_sites) * b->er_n_energies;
    std::vector<cx<double>> dev(pairs * block);
    HIP_CHECK(hipMemcpyAsync(dev.data(), b->er_sums.as<void>(), dev.size() * sizeof(cx<double>), hipMemcpyDeviceToHost,
                             b->stream));
    HIP_CHECK(hipMemcpyAsync(specular_sums, b->er_specular.as<void>(),
                             std::size_t(b->er_n_energies) * b->s.nzsp * b->s.nr * sizeof(cx<double>),
                             hipMemcpyDeviceToHost, b->stream));
    HIP_CHECK(hipStreamSynchronize(b->stream));
    // [pair][irot][izr] -> [pair][izr][irot]
    // (the caller's buffer is only guaranteed 8-byte aligned: copy components)
    for (std::size_t pr = 0; pr < pairs; ++pr)
      for (std::size_t irot = 0; irot < n_rot; ++irot)
        for (std::size_t izr = 0; izr < n_zr; ++izr) {
          const cx<double> v = dev[pr * block + izr + n_zr * irot];
          double* o = sums + 2 * (pr * block + irot + n_rot * izr);
          o[0] = v.x;
          o[1] = v.y;
        }
  });
}

int spo_hip_profile_enable(spo_hip_backend* b, int on) {
  return guarded([&] {
    if (on && b->use_graph) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_profile_enable: graph mode is on");
    HIP_CHECK(hipStreamSynchronize(b->stream));
    for (const auto& t : b->timed_launches) {
      b->event_pool.push_back(t.start);
      b->event_pool.push_back(t.stop);
    }
    b->timed_launches.clear();
    b->profiling = on != 0;
  });
}

int spo_hip_profile_read(spo_hip_backend* b, spo_hip_kernel_time* out, int capacity, int* count) {
  return guarded([&] {
    HIP_CHECK(hipStreamSynchronize(b->stream));
    std::vector<spo_hip_kernel_time> agg(b->kernel_names.size());
    for (std::size_t k = 0; k < agg.size(); ++k) {
      std::memset(&agg[k], 0, sizeof(agg[k]));
      std::strncpy(agg[k].name, b->kernel_names[k].c_str(), sizeof(agg[k].name) - 1);
    }
    for (const auto& t : b->timed_launches) {
      float ms = 0.0f;
      HIP_CHECK(hipEventElapsedTime(&ms, t.start, t.stop));
      agg[t.kernel].launches += 1;
      agg[t.kernel].total_ms += ms;
    }
    *count = static_cast<int>(agg.size());
    for (int k = 0; k < *count && k < capacity; ++k) out[k] = agg[k];
  });
}

int spo_hip_accumulate(spo_hip_backend* b, double time, const double* coefficients) {
  return guarded([&] {
    if (!b || !coefficients) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_accumulate: NULL argument");
    const spo_hip_analysis& a = b->analysis;
    const std::size_t n = std::size_t(a.n_states) * a.n_v;
    HIP_CHECK(hipMemcpyAsync(b->bk.as<void>(), coefficients, n * sizeof(cx<double>), hipMemcpyHostToDevice,
                             b->stream));
    const long total = long(n) * a.n_energies;
    hipLaunchKernelGGL(spo_dev::s_accumulate_kernel, dim3(blocks_for(total, kThreads)), dim3(kThreads), 0, b->stream,
                       b->sums.as<cx<double>>(), b->bk.as<cx<double>>(), static_cast<int>(n), a.n_energies,
                       b->energies.as<double>(), time, a.analysis_time_step);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipStreamSynchronize(b->stream));
  });
}

}  // extern "C"

// The potential surrogate's device state: FP32 master parameters, the hidden layers' bf16 fragments, Adam moments, what
// a training pass leaves for the gradient (made at the first one), and the rows of a call (grown to the largest one so
// far).
struct spo_hip_mlp {
  int batch = 0;
  int adam_step = 0;
  Buffer params, frag, grad, m, v;
  Buffer operands, values, errors;
  spo_dev::MlpTape tape{};
  Buffer x, t, y, losses;
  long x_values = 0, t_values = 0, y_values = 0, loss_values = 0;
};

namespace {

// `b`, holding at least `count` floats; `have` is its size.
float* at_least(Buffer& b, long& have, long count) {
  if (have < count) {
    have = 0;
    b = Buffer();  // the old memory first
    b = Buffer(std::size_t(count) * sizeof(float));
    have = count;
  }
  return b.as<float>();
}

void mlp_make_tape(spo_hip_mlp& n) {
  if (n.tape.a1) return;
  const std::size_t rows = n.batch, cells = rows * spo_dev::kMlpWidth;
  n.operands = Buffer(4 * cells * sizeof(short));
  n.values = Buffer(4 * cells * sizeof(float));
  n.errors = Buffer(2 * rows * sizeof(float));
  short* o = n.operands.as<short>();
  float* f = n.values.as<float>();
  float* e = n.errors.as<float>();
  n.tape = {o, o + cells, o + 2 * cells, o + 3 * cells, f, f + cells, f + 2 * cells, f + 3 * cells, e, e + rows};
}

// One pass over the batch at x, t, then Adam, or the gradient to grad_out.
void mlp_step(spo_hip_mlp& n, const float* x, const float* t, float* loss, float* grad_out, float lr) {
  spo_dev::MlpAdam adam{n.params.as<float>(), n.m.as<float>(), n.v.as<float>(), grad_out, lr, 0.9f, 0.999f, 1e-8f,
                        1.0f, 1.0f};
  if (!grad_out) {
    ++n.adam_step;
    adam.c1 = 1.0f - std::pow(adam.beta1, static_cast<float>(n.adam_step));
    adam.c2 = 1.0f - std::pow(adam.beta2, static_cast<float>(n.adam_step));
  }
  hipLaunchKernelGGL(spo_dev::mlp_pass_kernel, dim3(n.batch / spo_dev::kMlpRows), dim3(256), 0, nullptr, x, t,
                     long(n.batch), n.params.as<float>(), n.frag.as<short>(), n.tape);
  HIP_CHECK(hipGetLastError());
  hipLaunchKernelGGL(spo_dev::mlp_update_kernel, dim3(spo_dev::kMlpUpdateBlocks), dim3(256), 0, nullptr, adam,
                     n.frag.as<short>(), n.tape, x, long(n.batch), loss);
  HIP_CHECK(hipGetLastError());
}

}  // namespace

extern "C" {

int spo_hip_mlp_create(int batch, spo_hip_mlp** out) {
  return guarded([&] {
    if (!out) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_mlp_create: NULL out");
    if (batch < 16 || batch % 16 != 0 || batch > (1 << 22))
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_mlp_create: batch must be a multiple of 16 (16 .. 4194304)");
    require_device();
    auto n = std::make_unique<spo_hip_mlp>();
    n->batch = batch;
    const std::size_t pb = spo_dev::kMlpParams * sizeof(float), fb = spo_dev::kMlpFragments * sizeof(short);
    n->params = Buffer(pb);
    n->frag = Buffer(fb);
    n->grad = Buffer(pb);
    n->m = Buffer(pb);
    n->v = Buffer(pb);
    HIP_CHECK(hipMemset(n->params.as<void>(), 0, pb));
    HIP_CHECK(hipMemset(n->frag.as<void>(), 0, fb));
    HIP_CHECK(hipMemset(n->m.as<void>(), 0, pb));
    HIP_CHECK(hipMemset(n->v.as<void>(), 0, pb));
    *out = n.release();
  });
}

int spo_hip_mlp_destroy(spo_hip_mlp* mlp) {
  delete mlp;
  return SPO_HIP_OK;
}

int spo_hip_mlp_set_params(spo_hip_mlp* mlp, const float* params) {
  return guarded([&] {
    if (!mlp || !params) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_mlp_set_params: NULL argument");
    HIP_CHECK(hipMemcpy(mlp->params.as<void>(), params, spo_dev::kMlpParams * sizeof(float), hipMemcpyHostToDevice));
    const std::size_t pb = spo_dev::kMlpParams * sizeof(float);
    HIP_CHECK(hipMemset(mlp->m.as<void>(), 0, pb));
    HIP_CHECK(hipMemset(mlp->v.as<void>(), 0, pb));
    mlp->adam_step = 0;
    hipLaunchKernelGGL(spo_dev::mlp_fragment_kernel, dim3(blocks_for(2L * spo_dev::kMlpWidth * spo_dev::kMlpWidth, 256)),
                       dim3(256), 0, nullptr, mlp->params.as<float>(), mlp->frag.as<short>());
    HIP_CHECK(hipGetLastError());
  });
}

int spo_hip_mlp_get_params(const spo_hip_mlp* mlp, float* params) {
  return guarded([&] {
    if (!mlp || !params) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_mlp_get_params: NULL argument");
    HIP_CHECK(hipMemcpy(params, mlp->params.as<void>(), spo_dev::kMlpParams * sizeof(float), hipMemcpyDeviceToHost));
  });
}

int spo_hip_mlp_gradient(spo_hip_mlp* mlp, const float* x, const float* t, float* loss, float* grad) {
  return guarded([&] {
    if (!mlp || !x || !t || !loss || !grad) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_mlp_gradient: NULL argument");
    const long rows = mlp->batch;
    float* dx = at_least(mlp->x, mlp->x_values, rows * spo_dev::kMlpIn);
    float* dt = at_least(mlp->t, mlp->t_values, rows);
    float* dl = at_least(mlp->losses, mlp->loss_values, 1);
    HIP_CHECK(hipMemcpy(dx, x, rows * spo_dev::kMlpIn * sizeof(float), hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(dt, t, rows * sizeof(float), hipMemcpyHostToDevice));
    mlp_make_tape(*mlp);
    mlp_step(*mlp, dx, dt, dl, mlp->grad.as<float>(), 0.0f);
    HIP_CHECK(hipMemcpy(loss, dl, sizeof(float), hipMemcpyDeviceToHost));
    HIP_CHECK(hipMemcpy(grad, mlp->grad.as<void>(), spo_dev::kMlpParams * sizeof(float), hipMemcpyDeviceToHost));
  });
}

int spo_hip_mlp_train(spo_hip_mlp* mlp, long n, const float* x, const float* t, int steps, float lr, float* losses) {
  return guarded([&] {
    if (!mlp || !x || !t || !losses) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_mlp_train: NULL argument");
    if (n < mlp->batch || n % mlp->batch != 0 || steps < 0)
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_mlp_train: n must be a positive multiple of the batch");
    if (steps == 0) return;
    // Only the rows that these steps reach.
    const long rows = mlp->batch, used = std::min(n, steps * rows);
    float* dx = at_least(mlp->x, mlp->x_values, used * spo_dev::kMlpIn);
    float* dt = at_least(mlp->t, mlp->t_values, used);
    float* dl = at_least(mlp->losses, mlp->loss_values, steps);
    HIP_CHECK(hipMemcpy(dx, x, std::size_t(used) * spo_dev::kMlpIn * sizeof(float), hipMemcpyHostToDevice));
    HIP_CHECK(hipMemcpy(dt, t, std::size_t(used) * sizeof(float), hipMemcpyHostToDevice));
    mlp_make_tape(*mlp);
    for (int s = 0; s < steps; ++s) {
      const long off = (static_cast<long>(s) * rows) % n;
      mlp_step(*mlp, dx + off * spo_dev::kMlpIn, dt + off, dl + s, nullptr, lr);
    }
    HIP_CHECK(hipMemcpy(losses, dl, steps * sizeof(float), hipMemcpyDeviceToHost));
  });
}

int spo_hip_mlp_predict(spo_hip_mlp* mlp, long n, const float* x, float* y) {
  return guarded([&] {
    if (!mlp || (n > 0 && (!x || !y)) || n < 0) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_mlp_predict: bad arguments");
    constexpr long kChunk = 1L << 20;  // rows per launch: 28 MB of device memory
    for (long done = 0; done < n;) {
      const long rows = std::min(kChunk, n - done);
      float* dx = at_least(mlp->x, mlp->x_values, rows * spo_dev::kMlpIn);
      float* dy = at_least(mlp->y, mlp->y_values, rows);
      HIP_CHECK(hipMemcpy(dx, x + done * spo_dev::kMlpIn, rows * spo_dev::kMlpIn * sizeof(float), hipMemcpyHostToDevice));
      const long tiles = (rows + spo_dev::kMlpRows - 1) / spo_dev::kMlpRows;
      hipLaunchKernelGGL(spo_dev::mlp_predict_kernel, dim3(static_cast<unsigned>(std::min(tiles, 2048L))), dim3(256), 0,
                         nullptr, dx, mlp->params.as<float>(), mlp->frag.as<short>(), rows, dy);
      HIP_CHECK(hipGetLastError());
      HIP_CHECK(hipMemcpy(y + done, dy, rows * sizeof(float), hipMemcpyDeviceToHost));
      done += rows;
    }
  });
}

int spo_hip_pes_values(int pes, long n, const double* points, double* values) {
  return guarded([&] {
    if (pes != SPO_HIP_PES_HARDWALL && pes != SPO_HIP_PES_DAILIGHT)
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_pes_values: unknown surface " + std::to_string(pes));
    if (n < 0 || (n > 0 && (!points || !values))) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_pes_values: bad arrays");
    if (n == 0) return;
    require_device();
    Buffer p = upload(points, std::size_t(n) * 6 * sizeof(double));
    Buffer out(std::size_t(n) * sizeof(double));
    hipLaunchKernelGGL(spo_dev::pes_points_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, nullptr, pes, n,
                       p.as<double>(), out.as<double>());
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipMemcpy(values, out.as<void>(), std::size_t(n) * sizeof(double), hipMemcpyDeviceToHost));
  });
}

}  // extern "C"

// Scratch of spo_hip_pes_values_static, one copy per device for the life of the process: the points (6 doubles
// each) of up to kPesStaticMax points, then their values. 3.5 MiB.
constexpr long kPesStaticMax = 1L << 16;
static __device__ __align__(256) double scratch[7 * kPesStaticMax];

namespace {

// The device address of `scratch` on each device, looked up once per device with that device current. In host
// code the name `scratch` is only a stand-in for the symbol; kernels and copies get this address instead.
constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
double* scratch_address[kMaxDevices] = {};

double* scratch_on_current_device() {
  int dev = 0;
  HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) throw Status(SPO_HIP_E_NOT_SUPPORTED, "device index beyond the scratch table");
  std::lock_guard<std::mutex> lock(scratch_mutex);
  if (!scratch_address[dev]) {
    void* p = nullptr;
    HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    scratch_address[dev] = static_cast<double*>(p);
  }
  return scratch_address[dev];
}

}  // namespace

extern "C" {

int spo_hip_pes_values_static(int pes, long n, const double* points, double* values) {
  return guarded([&] {
    if (pes != SPO_HIP_PES_HARDWALL && pes != SPO_HIP_PES_DAILIGHT)
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_pes_values_static: unknown surface " + std::to_string(pes));
    if (n < 0 || (n > 0 && (!points || !values)))
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_pes_values_static: bad arrays");
    if (n > kPesStaticMax)
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_pes_values_static: " + std::to_string(n) + " points, at most " +
                                           std::to_string(kPesStaticMax) + " per call");
    if (n == 0) return;
    require_device();
    double* p = scratch_on_current_device();
    double* out = p + 6 * kPesStaticMax;
    // Every value of the call is written by the kernel, so nothing of an earlier call's contents is read.
    HIP_CHECK(hipMemcpy(p, points, std::size_t(n) * 6 * sizeof(double), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(spo_dev::pes_points_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, nullptr, pes, n, p, out);
    HIP_CHECK(hipGetLastError());
    HIP_CHECK(hipMemcpy(values, out, std::size_t(n) * sizeof(double), hipMemcpyDeviceToHost));
  });
}

}  // extern "C"

namespace {

// A packed CRP surface, checked against its own offsets, and an SCM correction (or NULL; the atoms' layers 1 or 2, a
// positive scale) on the device, with `room` bytes after them: one allocation and one copy. An array each (10 and the
// slab's) cost a call 13 us apiece in allocations, copies and frees: 265 us for 1000 points, of them 44 in the kernel,
// and now 107.
struct CrpUpload {
  Buffer memory;
  spo_dev::CrpDev view{};
  spo_dev::ScmDev correction{};
  void* room = nullptr;

  CrpUpload(const spo_hip_crp_surface& s, const spo_hip_scm_correction* m, std::size_t room_bytes = 0) {
    const int n_basis = s.square ? 0 : (s.c3v ? 10 : 7), n_cuts = s.square ? 16 : (s.c3v ? 29 : 18);
    auto bad = [](const char* what) { throw Status(SPO_HIP_E_ARGUMENT, std::string("CRP surface: ") + what); };
    if (s.n_cuts != n_cuts) bad("the number of molecular cuts does not match the symmetry");
    if (s.n_corrugation < 4 || s.n_cluster < 1 || s.n_h2 < 4 || s.n_z_dependence < 4) bad("too few points");
    if (!s.corrugation || !s.cluster || !s.atom_offsets || !s.cut_shape || !s.cut_offsets || !s.cut_data || !s.h2 ||
        !s.z_dependence || (!s.square && !s.atom_splines) || (s.square && !s.cell_spline))
      bad("NULL array");
    if (s.square && s.cell_nz < 4) bad("the C4v cell spline needs at least 4 z points");
    if (s.atom_offsets[0] != 0) bad("atom offsets");
    for (int i = 0; i < n_basis; ++i)
      if (s.atom_offsets[i + 1] - s.atom_offsets[i] < 4) bad("an atom cut with fewer than 4 knots");
    if (s.cut_offsets[0] != 0) bad("cut offsets");
    for (int k = 0; k < n_cuts; ++k) {
      const long nr = s.cut_shape[3 * k], nz = s.cut_shape[3 * k + 1], g = s.cut_shape[3 * k + 2];
      if (nr < 4 || nz < 4 || g < 0 || g > k) bad("cut shape");
      if (g != k && (s.cut_shape[3 * g] != nr || s.cut_shape[3 * g + 1] != nz)) bad("cut group of another shape");
      if (s.cut_offsets[k + 1] - s.cut_offsets[k] != nr + nz + 4 * nr * nz) bad("cut block size");
    }
    if (m) {
      if (m->n_atoms < 1 || !m->atoms) throw Status(SPO_HIP_E_ARGUMENT, "SCM correction: no atoms");
      if (!(m->scale > 0.0)) throw Status(SPO_HIP_E_ARGUMENT, "SCM correction: the scale must be positive");
      for (int i = 0; i < m->n_atoms; ++i)
        if (m->atoms[7 * i + 6] != 1.0 && m->atoms[7 * i + 6] != 2.0)
          throw Status(SPO_HIP_E_ARGUMENT, "SCM correction: an atom outside layers 1 and 2");
    }
    struct Part {
      const void* from;
      std::size_t bytes, at;
    };
    std::vector<Part> parts;
    std::size_t total = 0;
    auto add = [&](const void* from, std::size_t bytes) {
      parts.push_back({from, bytes, total});
      total += (bytes + 15) / 16 * 16;
      return parts.back().at;
    };
    auto doubles = [&](const double* from, std::size_t n) { return add(from, n * sizeof(double)); };
    const std::size_t corrugation = doubles(s.corrugation, 3 * std::size_t(s.n_corrugation));
    const std::size_t cluster = doubles(s.cluster, 4 * std::size_t(s.n_cluster));
    const std::size_t atom_offsets = add(s.atom_offsets, (n_basis + 1) * sizeof(int));
    const std::size_t atom_splines =
        doubles(s.atom_splines, s.square ? 0 : 3 * std::size_t(s.atom_offsets[n_basis]));
    const std::size_t cell =
        doubles(s.cell_spline, s.square ? 10 + std::size_t(s.cell_nz) + 8 * 25 * std::size_t(s.cell_nz) : 0);
    const std::size_t cut_shape = add(s.cut_shape, 3 * std::size_t(n_cuts) * sizeof(int));
    const std::size_t cut_offsets = add(s.cut_offsets, (n_cuts + 1) * sizeof(long));
    const std::size_t cut_data = doubles(s.cut_data, std::size_t(s.cut_offsets[n_cuts]));
    const std::size_t h2 = doubles(s.h2, 3 * std::size_t(s.n_h2));
    const std::size_t zdep = doubles(s.z_dependence, 3 * std::size_t(s.n_z_dependence));
    const std::size_t atoms = doubles(m ? m->atoms : nullptr, m ? 7 * std::size_t(m->n_atoms) : 0);
    std::vector<unsigned char> packed(total);
    for (const Part& part : parts)
      if (part.bytes) std::memcpy(packed.data() + part.at, part.from, part.bytes);
    memory = Buffer(total + room_bytes);
    unsigned char* base = memory.as<unsigned char>();
    HIP_CHECK(hipMemcpy(base, packed.data(), total, hipMemcpyHostToDevice));
    room = base + total;
    auto on = [&](std::size_t at) { return reinterpret_cast<const double*>(base + at); };
    view = spo_dev::CrpDev{s.c3v, n_basis, n_cuts, s.n_corrugation, s.n_cluster, s.n_h2, s.n_z_dependence,
                           s.lattice_constant, s.zso_min, s.zso_max, s.r_min, s.r_max, s.z_min, s.h2_asymptote,
                           on(corrugation), on(cluster), reinterpret_cast<const int*>(base + atom_offsets),
                           on(atom_splines), reinterpret_cast<const int*>(base + cut_shape),
                           reinterpret_cast<const long*>(base + cut_offsets), on(cut_data), on(h2), on(zdep), s.square,
                           s.cell_nz, s.square ? on(cell) : nullptr};
    if (!m) return;
    correction.on = 1;
    correction.rescale = m->rescale;
    correction.scale = m->scale;
    correction.cos_skew = m->cos_skew;
    correction.sin_skew = m->sin_skew;
    for (int l = 0; l < 2; ++l)
      for (int k = 0; k < 18; ++k) correction.layers[l][k] = m->layers[l][k];
    correction.n_atoms = m->n_atoms;
    correction.atoms = on(atoms);
  }
};

using CrpPointsKernel = decltype(&spo_dev::crp_points_kernel<8, true>);
constexpr CrpPointsKernel kCrpPointsKernels[2][2] = {
    {spo_dev::crp_points_kernel<spo_dev::kCrpWaves, false>, spo_dev::crp_points_kernel<spo_dev::kCrpWaves, true>},
    {spo_dev::crp_points_kernel<spo_dev::kCrpWavesFew, false>, spo_dev::crp_points_kernel<spo_dev::kCrpWavesFew, true>}};
using CrpGridKernel = decltype(&spo_dev::crp_grid_kernel<8, true>);
constexpr CrpGridKernel kCrpGridKernels[2][2] = {
    {spo_dev::crp_grid_kernel<spo_dev::kCrpWaves, false>, spo_dev::crp_grid_kernel<spo_dev::kCrpWaves, true>},
    {spo_dev::crp_grid_kernel<spo_dev::kCrpWavesFew, false>, spo_dev::crp_grid_kernel<spo_dev::kCrpWavesFew, true>}};

// A CRP kernel over n points, 64 a workgroup: kernels[few][staged], few workgroups (at most one a CU) of 16 wavefronts
// and the corrugation function in LDS or read from memory.
template <class... P, class... A>
void launch_crp(const spo_dev::CrpDev& s, void (*const (&kernels)[2][2])(long, long, P...), long n, const A&... args) {
  int dev = 0, units = 0;
  HIP_CHECK(hipGetDevice(&dev));
  HIP_CHECK(hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, dev));
  const bool few = n <= 64L * units;
  const int doubles = spo_dev::crp_staged_doubles(s.n_corrugation);
  const bool staged = doubles <= spo_dev::kCrpStagedMax;
  const auto kernel = kernels[few][staged];
  const int threads = 64 * (few ? spo_dev::kCrpWavesFew : spo_dev::kCrpWaves);
  const std::size_t lds = spo_dev::crp_lds(staged ? doubles : 0);
  // The kernel's limit is one for the process: the same for every table, so that threads with other surfaces agree.
  set_lds(reinterpret_cast<const void*>(kernel), spo_dev::crp_lds(spo_dev::kCrpStagedMax));
  constexpr long kLaunch = 1L << 28;  // a launch has at most 2^32 threads, 8 a point here
  for (long first = 0; first < n; first += kLaunch) {
    const dim3 grid(blocks_for(std::min(n - first, kLaunch), 64));
    hipLaunchKernelGGL(kernel, grid, dim3(threads), lds, nullptr, first, n, args...);
    HIP_CHECK(hipGetLastError());
  }
}

void check_finite(const double* v, long n, const char* where) {
  for (long i = 0; i < n; ++i)
    if (std::isnan(v[i]))
      throw Status(SPO_HIP_E_ARGUMENT, std::string(where) + ": the CRP surface cannot be evaluated at point " +
                                           std::to_string(i) + " (an atom on a surface atom or outside the data)");
}

}  // namespace

extern "C" {

int spo_hip_crp_values(const spo_hip_crp_surface* surface, long n, const double* points, double* values) {
  return spo_hip_scm_values(surface, nullptr, n, points, values);
}

int spo_hip_scm_values(const spo_hip_crp_surface* surface, const spo_hip_scm_correction* scm, long n,
                       const double* points, double* values) {
  return guarded([&] {
    if (!surface) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_crp_values: NULL surface");
    if (n < 0 || (n > 0 && (!points || !values))) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_crp_values: bad arrays");
    if (n == 0) return;
    require_device();
    const CrpUpload crp(*surface, scm, std::size_t(n) * 7 * sizeof(double));
    double* const p = static_cast<double*>(crp.room);
    double* const out = p + 6 * n;
    HIP_CHECK(hipMemcpy(p, points, std::size_t(n) * 6 * sizeof(double), hipMemcpyHostToDevice));
    launch_crp(crp.view, kCrpPointsKernels, n, crp.view, crp.correction, static_cast<const double*>(p), out);
    HIP_CHECK(hipMemcpy(values, out, std::size_t(n) * sizeof(double), hipMemcpyDeviceToHost));
    check_finite(values, n, "spo_hip_crp_values");
  });
}

int spo_hip_potential_grid(const spo_hip_pes_grid* grid, double* values) {
  return guarded([&] {
    if (!grid || !values) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_potential_grid: NULL argument");
    const spo_hip_pes_grid& g = *grid;
    if (g.pes != SPO_HIP_PES_HARDWALL && g.pes != SPO_HIP_PES_DAILIGHT && g.pes != SPO_HIP_PES_CRP)
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_potential_grid: unknown surface " + std::to_string(g.pes));
    if (g.pes == SPO_HIP_PES_CRP && !g.crp) throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_potential_grid: no CRP surface");
    if (g.nx <= 0 || g.ny <= 0 || g.nr <= 0 || g.nz_potential < 0 || g.n_theta <= 0 || g.n_phi <= 0 ||
        g.n_representatives <= 0 || g.n_representatives > g.nx * g.ny)
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_potential_grid: bad extents");
    if (!g.x || !g.y || !g.r || !g.theta || !g.phi || !g.representatives || (g.nz_potential > 0 && !g.z) ||
        (g.use_switching && !g.gas_phase))
      throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_potential_grid: NULL table");
    for (int k = 0; k < g.n_representatives; ++k)
      if (g.representatives[k] < 0 || g.representatives[k] >= g.nx * g.ny)
        throw Status(SPO_HIP_E_ARGUMENT, "spo_hip_potential_grid: representative outside the (x, y) grid");
    const long n_zr = long(g.nz_potential) * g.nr;
    const long n = long(g.n_theta) * g.n_phi * g.n_representatives * n_zr;
    if (n == 0) return;
    require_device();
    auto up = [](const void* h, std::size_t bytes) { return upload(h, bytes); };
    Buffer x = up(g.x, g.nx * sizeof(double)), y = up(g.y, g.ny * sizeof(double));
    Buffer z = up(g.z, g.nz_potential * sizeof(double)), r = up(g.r, g.nr * sizeof(double));
    Buffer th = up(g.theta, g.n_theta * sizeof(double)), ph = up(g.phi, g.n_phi * sizeof(double));
    Buffer reps = up(g.representatives, g.n_representatives * sizeof(int));
    Buffer gas = g.use_switching ? up(g.gas_phase, g.nr * sizeof(double)) : Buffer();
    Buffer out(std::size_t(n) * sizeof(double));
    std::optional<CrpUpload> crp;
    if (g.pes == SPO_HIP_PES_CRP) crp.emplace(*g.crp, g.scm);
    spo_dev::PesGrid d{g.pes, g.ny, g.nr, g.n_theta, g.n_phi, g.n_representatives, static_cast<int>(n_zr),
                       x.as<double>(), y.as<double>(), z.as<double>(), r.as<double>(), th.as<double>(),
                       ph.as<double>(), reps.as<int>(), g.use_switching, g.z_min_switch, g.z_max_switch,
                       g.use_switching ? gas.as<double>() : nullptr, g.impose_v_min, g.impose_v_max, g.v_min,
                       g.v_max, crp ? crp->view : spo_dev::CrpDev{}, crp ? crp->correction : spo_dev::ScmDev{}};
    if (g.pes == SPO_HIP_PES_CRP) {
      launch_crp(d.crp, kCrpGridKernels, n, d, out.as<double>());
    } else {
      hipLaunchKernelGGL(spo_dev::potential_grid_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, nullptr, d,
                         out.as<double>());
      HIP_CHECK(hipGetLastError());
    }
    HIP_CHECK(hipMemcpy(values, out.as<void>(), std::size_t(n) * sizeof(double), hipMemcpyDeviceToHost));
    if (g.pes == SPO_HIP_PES_CRP) check_finite(values, n, "spo_hip_potential_grid");
  });
}

}  // extern "C"
