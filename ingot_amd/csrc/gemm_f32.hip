// Tile configurations of the f32 MFMA GEMM (indices of its gemm_configs table).

#include "gemm_mfma.hpp"

namespace ingot {

hipError_t launch_gemm_f32(int cfg, const GemmArgs& a, int batch, hipStream_t st) {
    switch (cfg) {
        case 0: return launch_one<KIND_F32, 128, 128, 2, 2, 2>(a, batch, st);
        case 1: return launch_one<KIND_F32, 128, 64, 2, 2, 2>(a, batch, st);
        case 2: return launch_one<KIND_F32, 64, 64, 2, 2, 3>(a, batch, st);
        case 3: return launch_one<KIND_F32, 32, 96, 2, 2, 2>(a, batch, st);
        case 4: return launch_one<KIND_F32, 32, 32, 2, 2, 4>(a, batch, st);
        case 5: return launch_one<KIND_F32, 32, 96, 2, 2, 4>(a, batch, st);
        case 6: return launch_one<KIND_F32, 64, 96, 2, 2, 3>(a, batch, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace ingot
