// One translation unit per (16-bit element type, product) of the persistent grouped GEMM; the build
// compiles this file with -DFMOE_GEMM_TYPE=<1 bf16|2 f16> and -DFMOE_GEMM_PRODUCT=<0 fwd|1 dgrad|2 wgrad>.
#include "gemm_ring.hpp"

#if FMOE_GEMM_TYPE == 1
#define FMOE_T __bf16
#define FMOE_TNAME bf16
#elif FMOE_GEMM_TYPE == 2
#define FMOE_T _Float16
#define FMOE_TNAME f16
#else
#error "FMOE_GEMM_TYPE must be 1 or 2"
#endif

#define FMOE_CAT_(a, b, c) launch_ring_##a##_##b
#define FMOE_CAT(a, b) FMOE_CAT_(a, b, )

namespace fmoe {
using namespace gemm;

#if FMOE_GEMM_PRODUCT == 0
int FMOE_CAT(FMOE_TNAME, fwd)(const RingParams &prm, int epilogue, int activation, hipStream_t stream) {
    if (epilogue == kEpiBiasAct) {
        const bool aux = prm.aux != nullptr;
        if (activation == FMOE_ACT_GELU && aux)
            return launch_ring<FMOE_T, kKC, kKC, kRaggedRows, kEpiBiasAct, FMOE_ACT_GELU, true>(prm, stream);
        if (activation == FMOE_ACT_GELU)
            return launch_ring<FMOE_T, kKC, kKC, kRaggedRows, kEpiBiasAct, FMOE_ACT_GELU, false>(prm, stream);
        if (activation == FMOE_ACT_RELU && !aux)
            return launch_ring<FMOE_T, kKC, kKC, kRaggedRows, kEpiBiasAct, FMOE_ACT_RELU, false>(prm, stream);
        return fail(FMOE_EINVAL, "activation %d is not built for the persistent kernel", activation);
    }
    return launch_ring<FMOE_T, kKC, kKC, kRaggedRows, kEpiStore>(prm, stream);
}
#elif FMOE_GEMM_PRODUCT == 1
int FMOE_CAT(FMOE_TNAME, dgrad)(const RingParams &prm, int epilogue, int activation, hipStream_t stream) {
    if (epilogue == kEpiDAct) {
        if (activation == FMOE_ACT_GELU) return launch_ring<FMOE_T, kMC, kKC, kRaggedRows, kEpiDAct, FMOE_ACT_GELU, true>(prm, stream);
        if (activation == FMOE_ACT_RELU) return launch_ring<FMOE_T, kMC, kKC, kRaggedRows, kEpiDAct, FMOE_ACT_RELU, true>(prm, stream);
        return fail(FMOE_EINVAL, "activation %d is not built for the persistent kernel", activation);
    }
    return launch_ring<FMOE_T, kMC, kKC, kRaggedRows, kEpiStore>(prm, stream);
}
#elif FMOE_GEMM_PRODUCT == 2
int FMOE_CAT(FMOE_TNAME, wgrad)(const RingParams &prm, int, int, hipStream_t stream) {
    return launch_ring<FMOE_T, kMC, kMC, kRaggedK, kEpiStore>(prm, stream);
}
#else
#error "FMOE_GEMM_PRODUCT must be 0, 1 or 2"
#endif

}  // namespace fmoe
