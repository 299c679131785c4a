// gemm_rows.hip -- products of a model's short prompts and of the op-level tensors (at most 160 rows): which ones, in how many pieces along K,
// and the plain epilogues.  The kernel is in gemm_rows_device.h; gemm_rows_fused.hip holds w1|w3 and wq|wk|wv.
#include "gemm_rows_device.h"

namespace rlh {

hipError_t launch_gemm_f16_rows_fused(const GemmParams &p, int epilogue, hipStream_t s); // gemm_rows_fused.hip

// Microseconds of a product in `pieces` pieces with what has to follow it: a launch, then what one compute unit stages at 45 GB/s or all of
// the weights at 5.6 TB/s.  The kernel that adds the pieces brings the RMSNorm behind a residual product along.
static double rows_us(const GemmParams &p, int epilogue, int pieces) {
    const double k = ((p.k / 128 + pieces - 1) / pieces) * 128.0;
    const double staged = k / 1024 * rows_us_k(p, pieces, rows_columns(p, pieces)), weights = 2.0 * p.n * (double)p.k * (p.b2 != nullptr ? 2 : 1) / 5.6e6;
    double us = 3.0 + (staged > weights ? staged : weights);
    if (pieces > 1) us += 4.0 + 4.0 * pieces * (double)p.m * p.n / 4.7e6;
    if (epilogue == kGemmEpiResAddF32 && p.norm_w != nullptr) us += pieces > 1 ? 1.2 : 4.5;
    return us;
}

int gemm_f16_rows_pieces(const GemmParams &p, int epilogue) {
    if (p.tune.no_rows || p.tune.dual_plus1 != 0 || p.tune.tile_plus1 != 0 || p.tune.split_k != 0 || p.f32_operands || p.k_seg != 0 || p.causal != 0 || p.accumulate) return 0;
    if (p.keep_order && p.m > 16) return 0;
    if (p.batch != 1 || p.split_k > 1 || p.m < 1 || p.m > kRowsMax) return 0;
    if (p.n < 8 || p.n % 8 != 0 || p.k < 128 || p.k % 128 != 0 || p.lda % 8 != 0 || p.ldb % 8 != 0 || p.ldc % 8 != 0) return 0;
    const uintptr_t all = reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.b) | reinterpret_cast<uintptr_t>(p.b2) | reinterpret_cast<uintptr_t>(p.c) |
                          reinterpret_cast<uintptr_t>(p.residual);
    if (all % 16 != 0) return 0;
    if ((uint64_t)kRowsMax * 2 * (uint64_t)(p.lda > p.ldb ? p.lda : p.ldb) >> 32) return 0; // byte offsets within a tile are 32 bits
    switch (epilogue) {
    case kGemmEpiSiluGateF16:
        // (long rows of few columns are faster as two cut products: gemm_f16_gate_cut has the figures)
        return p.b2 != nullptr && !gemm_f16_gate_cut(p) ? 1 : 0;
    case kGemmEpiRopeQkv: return p.b2 == nullptr ? 1 : 0;
    case kGemmEpiF16:
    case kGemmEpiResAddF32: break;
    default: return 0;
    }
    if (p.b2 != nullptr || (epilogue == kGemmEpiResAddF32 && p.residual == nullptr)) return 0;
    const size_t per = (size_t)p.m * p.n * sizeof(float);
    const size_t room = p.workspace == nullptr ? 0 : p.workspace_bytes < kGemmPartialBytes ? p.workspace_bytes : kGemmPartialBytes;
    int best = 1;
    double best_us = rows_us(p, epilogue, 1);
    for (int pieces = 2; pieces <= 8 && pieces * 4 <= p.k / 128 && pieces * per <= room && reinterpret_cast<uintptr_t>(p.workspace) % 16 == 0; pieces++) {
        const double us = rows_us(p, epilogue, pieces);
        if (us < best_us) {
            best = pieces;
            best_us = us;
        }
    }
    return best;
}

hipError_t launch_gemm_f16_rows(const GemmParams &p, int epilogue, hipStream_t s) {
    switch (epilogue) {
    case kGemmEpiF16: return launch_rows_epi<kGemmEpiF16>(p, s);
    case kGemmEpiF32: return p.split_k > 1 ? launch_rows_epi<kGemmEpiF32>(p, s) : hipErrorInvalidValue;
    case kGemmEpiResAddF32: return launch_rows_epi<kGemmEpiResAddF32>(p, s);
    case kGemmEpiSiluGateF16:
    case kGemmEpiRopeQkv: return launch_gemm_f16_rows_fused(p, epilogue, s);
    default: return hipErrorInvalidValue;
    }
}

} // namespace rlh
