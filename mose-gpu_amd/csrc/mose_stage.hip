// The fused stage kernels of the parity path (mose_stage.hpp) for one (MOSE_NS, MOSE_NR), given by the build: one
// translation unit per species and RANS count, so that they compile side by side.
#include <hip/hip_runtime.h>

#include "mose_stage.hpp"

namespace mose {

template void launch_stage_tiles<MOSE_NS, MOSE_NR>(const CaseDev&, const StageArgs&, int, bool, unsigned, size_t,
                                                   hipStream_t);

}  // namespace mose
