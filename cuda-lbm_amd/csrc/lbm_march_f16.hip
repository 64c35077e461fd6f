// lbm_march_f16.hip — the marching multi-step kernels, f16 storage.
#include "lbm_march_kernels.hpp"

namespace lbm {

hipError_t launch_march_f16(int coll, int steps, const StepParams& p, const MarchGrid& m, bool edge, bool wide, hipStream_t s) {
    return launch_march_s<LBM_F16_SHIFTED>(coll, steps, p, m, edge, wide, s);
}

}  // namespace lbm
