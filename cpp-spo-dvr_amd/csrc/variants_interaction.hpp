// The interaction kernels' instantiations, for the translation unit of each storage type.
#pragma once

#include <algorithm>

#include "kernels_mfma.hpp"
#include "variants.hpp"

namespace spo_dev {

constexpr int kLdsInteractionThreads = 256;

// Phi lengths of the interaction kernel with the contractions on the vector units.
#define SPO_PHI_LENGTHS(X) X(48) X(22) X(10) X(12) X(8) X(56)
// Interaction with the theta contractions on MFMA (phi length, wavefronts, phi radices R1 x R2 of the fused phi
// step); the staged-FFT variant is instantiated with 8 wavefronts.
#define SPO_MFMA_SHAPES(X)                                                                                   \
  X(48, 8, 12, 4) X(48, 4, 12, 4) X(48, 16, 12, 4) X(22, 8, 11, 2) X(12, 8, 4, 3) X(10, 8, 5, 2)             \
  X(8, 8, 4, 2) X(56, 8, 8, 7) X(56, 4, 8, 7)
// The buffer-addressed interaction kernel (phi length, wavefronts, phi radices): the MFMA shapes, the phi steps of
// the reduced-JMax batch members (28 and 40 points) and two more factorisations of the 48-point step (16 x 3,
// 8 x 6) for the launch tuner.
#define SPO_BUF_SHAPES(X) SPO_MFMA_SHAPES(X) X(28, 8, 7, 4) X(40, 8, 10, 4) X(48, 8, 16, 3) X(48, 8, 8, 6)


// fused: the phi step in three register passes (phi_step_fused) rather than the staged LDS FFTs (8 wavefronts).
template <typename T>
std::vector<Variant> interaction_mfma_variants(int nphi, int n_theta, bool fused) {
  constexpr int NT = 1;  // 8 columns: one 128-byte line of an irot row in FP64 (two complex64 tiles ran slower)
  std::vector<Variant> out;
  const std::size_t lds = spo_dev::interaction_mfma_lds<T>(8 * NT, n_theta, nphi, fused);
#define X(A, W, R1, R2)                                                                                      \
  if (nphi == A && (fused || W == 8))                                                                        \
    out.push_back({fused ? reinterpret_cast<const void*>(spo_dev::interaction_mfma_kernel<T, A, NT, W, R1, R2>) \
                         : reinterpret_cast<const void*>(spo_dev::interaction_mfma_kernel<T, A, NT, W>),     \
                   64 * W, W, lds, {}, InteractionKind::mfma});
  SPO_MFMA_SHAPES(X)
#undef X
  return out;
}

// The buffer-addressed interaction kernel: every MFMA shape with at most 8 mJ blocks per wavefront; bf16x3: the
// complex64 split-BF16x3 contraction variant (instantiated for the 48-point phi step).
template <typename T>
std::vector<Variant> interaction_buf_variants(int nphi, int n_theta, int n_blocks, bool bf16x3) {
  std::vector<Variant> out;
  const std::size_t lds = spo_dev::interaction_buf_lds<T>(n_theta, nphi);
  if (bf16x3) {
    if constexpr (sizeof(T) == 4) {
      if (nphi == 48 && n_blocks <= 64)
        out.push_back({reinterpret_cast<const void*>(spo_dev::interaction_buf_kernel<T, 48, 8, 12, 4, true>), 512,
                       8, lds, {}, InteractionKind::buffer});
    }
    return out;
  }
#define X(A, W, R1, R2)                                                                                         \
  if (nphi == A && n_blocks <= 8 * W)                                                                           \
    out.push_back({reinterpret_cast<const void*>(spo_dev::interaction_buf_kernel<T, A, W, R1, R2>), 64 * W, W, lds, {}, InteractionKind::buffer});
  SPO_BUF_SHAPES(X)
#undef X
  return out;
}

template <typename T>
const void* interaction_ct_symbol(int nphi) {
#define X(A) \
  if (nphi == A) return reinterpret_cast<const void*>(spo_dev::interaction_ct_kernel<T, A, kLdsInteractionThreads>);
  SPO_PHI_LENGTHS(X)
#undef X
  return nullptr;
}

}  // namespace spo_dev
