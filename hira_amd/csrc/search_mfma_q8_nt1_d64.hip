// MFMA search kernel instantiations for D = 64, keys scanned through their 8-bit shadow, its tiles non-temporal.
#include "search_mfma_kernel.h"

namespace hira {
void launch_mfma_q8_nt1_d64(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s) {
    launch_mfma_mt<2, true, 1>(plan, p, grid, s);
}
}  // namespace hira
