// MFMA search kernel instantiations for D = 128, keys scanned through their 8-bit shadow, its tiles non-temporal.
#include "search_mfma_kernel.h"

namespace hira {
void launch_mfma_q8_nt1_d128(const SearchPlan& plan, const SearchParams& p, dim3 grid, hipStream_t s) {
    launch_mfma_mt<4, true, 1>(plan, p, grid, s);
}
}  // namespace hira
