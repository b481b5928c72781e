// Instantiations of the interaction kernels for complex64 storage.
#include <hip/hip_runtime.h>

#include "variants_interaction.hpp"

namespace spo_dev {

template std::vector<Variant> interaction_mfma_variants<float>(int, int, bool);
template std::vector<Variant> interaction_buf_variants<float>(int, int, int, bool);
template const void* interaction_ct_symbol<float>(int);

}  // namespace spo_dev
