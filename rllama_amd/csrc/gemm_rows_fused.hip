// gemm_rows_fused.hip -- the kernel of gemm_rows_device.h with the epilogues of w1|w3 (both products and SiLU * gate) and wq|wk|wv (RoPE, cache
// rows, V^T).
#include "gemm_rows_device.h"

namespace rlh {

hipError_t launch_gemm_f16_rows_fused(const GemmParams &p, int epilogue, hipStream_t s) {
    if (epilogue == kGemmEpiSiluGateF16) return launch_rows_epi<kGemmEpiSiluGateF16>(p, s);
    return epilogue == kGemmEpiRopeQkv ? launch_rows_epi<kGemmEpiRopeQkv>(p, s) : hipErrorInvalidValue;
}

} // namespace rlh
