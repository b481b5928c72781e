// Instantiations of the interaction kernels for fp64 storage.
#include <hip/hip_runtime.h>

#include "variants_interaction.hpp"

namespace spo_dev {

template std::vector<Variant> interaction_mfma_variants<double>(int, int, bool);
template std::vector<Variant> interaction_buf_variants<double>(int, int, int, bool);
template const void* interaction_ct_symbol<double>(int);

}  // namespace spo_dev
