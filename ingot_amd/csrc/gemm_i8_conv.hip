// The int8 tile configurations (indices of the kind's gemm_configs table) over a convolution's pixels (gemm_kernel's CONV).

#include "gemm_mfma.hpp"

namespace ingot {

hipError_t launch_gemm_i8_conv(int cfg, const GemmArgs& a, int batch, hipStream_t st) {
    switch (cfg) {
        case 0: return launch_one<KIND_I8, 256, 256, 2, 4, 2, 0, true>(a, batch, st);
        case 1: return launch_one<KIND_I8, 128, 128, 4, 2, 4, 0, true>(a, batch, st);
        case 2: return launch_one<KIND_I8, 128, 64, 2, 2, 2, 0, true>(a, batch, st);
        case 3: return launch_one<KIND_I8, 64, 64, 2, 2, 2, 0, true>(a, batch, st);
        case 4: return launch_one<KIND_I8, 64, 96, 2, 2, 2, 0, true>(a, batch, st);
        case 5: return launch_one<KIND_I8, 32, 32, 2, 2, 4, 0, true>(a, batch, st);
        case 6: return launch_one<KIND_I8, 64, 64, 2, 2, 4, 0, true>(a, batch, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace ingot
