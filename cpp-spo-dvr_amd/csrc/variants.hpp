// The launch variants of the shape-specialised kernels: which instantiations serve a shape, in order of preference.
// The instantiations are compiled in translation units of their own (variants_*.hip).
#pragma once

#include <cstddef>
#include <vector>

#include "kernels_angular.hpp"
#include "kernels_zr.hpp"

namespace spo_dev {

enum class InteractionKind { none, mfma, buffer, in_place };

// A launch variant of a kernel family: the kernel, its block size, its tile parameter (T_xy: izr per tile;
// interaction: wavefronts) and its LDS bytes.
struct Variant {
  const void* fn;
  int threads;
  int param;
  std::size_t lds;
  ZrShape zr = {};  // T_Zr: the radices
  InteractionKind kind = InteractionKind::none;  // interaction: the kernel
  int columns = 0, r1 = 0, r2 = 0;  // interaction_kernel_inplace: columns of a tile, phi radices
};

// T_Zr of a whole plane in LDS; empty for an axis that is not a product of two radices.
template <typename T>
std::vector<Variant> zr_variants(int nz, int nr);
// specular_plane_kernel for a grid of this shape (its radices to shape), or NULL where an axis is not a product of two
// radices.
constexpr int kSpecularThreads = 512;
const void* specular_plane(int nz, int nr, ZrShape& shape);
template <typename T>
std::vector<Variant> xy_reg_variants(int nx, int ny);
// fused: the phi step in three register passes (phi_step_fused) rather than the staged LDS FFTs (8 wavefronts).
template <typename T>
std::vector<Variant> interaction_mfma_variants(int nphi, int n_theta, bool fused);
// The buffer-addressed interaction kernel: every MFMA shape with at most 8 mJ blocks per wavefront; bf16x3: the
// complex64 split-BF16x3 contraction variant (instantiated for the 48-point phi step).
template <typename T>
std::vector<Variant> interaction_buf_variants(int nphi, int n_theta, int n_blocks, bool bf16x3);
// interaction_kernel_inplace for a phi length that is instantiated and at most 16 theta points; columns: the (Z, r, x, y)
// points of a launch.
template <typename T>
std::vector<Variant> interaction_inplace_variants(int nphi, int n_theta, long columns);
// The interaction kernel with the contractions on the vector units, or NULL.
template <typename T>
const void* interaction_ct_symbol(int nphi);

}  // namespace spo_dev
