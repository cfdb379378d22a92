// The fused stage kernels of the parity path (mose_stage.hpp) for one (MOSE_NS, MOSE_NR), given by the build: one
// translation unit per species and RANS count, so that they compile side by side.
#include <hip/hip_runtime.h>

#include "mose_flat.hpp"

namespace mose {

template void launch_stage_tiles<MOSE_NS, MOSE_NR>(const CaseDev&, const StageArgs&, int, bool, unsigned, size_t,
                                                   hipStream_t);

template <int NS, int NR>
const void* stage_kernel_parity() {
  return (const void*)k_stage<NS, NR, false, MOSE_RS_HLLC, 256, 0>;
}
template const void* stage_kernel_parity<MOSE_NS, MOSE_NR>();

#if MOSE_NS == 1 && MOSE_NR == 0
void launch_flat_parity(const CaseDev& D, const StageArgs& A, int rs, bool two, int threads, unsigned grid, hipStream_t s) {
  launch_flat<false>(D, A, rs, two, threads, grid, s);
}
#endif

}  // namespace mose
