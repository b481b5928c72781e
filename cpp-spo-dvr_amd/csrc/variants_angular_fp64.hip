// Instantiations of the in-place interaction kernel for fp64 storage.
#include <hip/hip_runtime.h>

#include "variants_angular.hpp"

namespace spo_dev {

template std::vector<Variant> interaction_inplace_variants<double>(int, int, long);

}  // namespace spo_dev
