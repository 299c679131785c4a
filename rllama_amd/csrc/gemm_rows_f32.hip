// gemm_rows_f32.hip -- fp32 products of a model's short prompts (f32 mode) on the kernel of gemm_rows_device.h and the fp32 matrix instruction.
//
// With few rows the weights are read at the rate of the memory whatever the arithmetic, so the fp32 instruction (a sixteenth of the f16
// rate) is fast enough, and nothing has to be decomposed, cut along K for lack of workgroups or added up by kernels of their own:
// w1 and w3 with SiLU * gate are one launch, wo and w2 add to the residual stream where it lies.
//
// Time to the first token, the kernels for any number of rows -> this, us, 2 / 16 / 32 / 64 rows: dim 1024, 16 layers 1911 / 1831 / 1973 / 2459 ->
// 1111 / 1078 / 1281 / 1542; dim 2048, 12 layers 1774 / 1854 / 1962 / 2410 -> 1150 / 1223 / 1466 / 1922; dim 4096, 6 layers 1801 / 1785 / 1847 /
// 2255 ->
// 1341 / 1263 / 1414 / 1994.
#include "gemm_rows_device.h"
#include "split3_plan.h"

namespace rlh {

// Microseconds of a product in `pieces` pieces with the kernel that adds them: a launch, then the longest of staging or arithmetic of a compute
// unit and all weights at 5.6 TB/s.
static double rows_f32_us(const GemmParams &p, int pieces) {
    const double k = ((p.k / 64 + pieces - 1) / pieces) * 64.0;
    const double work = k / 1024 * rows_us_k(p, pieces, rows_columns(p, pieces)), weights = 4.0 * p.n * (double)p.k * (p.b2 != nullptr ? 2 : 1) / 5.6e6;
    return 3.0 + (work > weights ? work : weights) + (pieces > 1 ? 4.0 + 4.0 * pieces * (double)p.m * p.n / 4.7e6 : 0.0);
}

int gemm_f32_rows_pieces(const GemmParams &p, int epilogue) {
    if (p.tune.no_rows || p.tune.split3_plus1 != 0 || p.tune.tile_plus1 != 0 || p.tune.split_k != 0 || p.keep_order || !p.f32_operands || p.k_seg != 0 || p.causal != 0) return 0;
    if (p.batch != 1 || p.split_k > 1 || p.m < 1 || p.m > kRowsF32Max || p.n < 4 || p.n % 4 != 0 || p.k < 64 || p.k % 64 != 0 || p.lda % 4 != 0 || p.ldb % 4 != 0 || p.ldc % 4 != 0) return 0;
    const uintptr_t all = reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.b) | reinterpret_cast<uintptr_t>(p.b2) | reinterpret_cast<uintptr_t>(p.c);
    if (all % 16 != 0 || (uint64_t)kRowsF32Max * 4 * (uint64_t)(p.lda > p.ldb ? p.lda : p.ldb) >> 32) return 0; // byte offsets within a tile are 32 bits
    if (epilogue == kGemmEpiSiluGateF32 ? p.b2 == nullptr || p.accumulate : epilogue != kGemmEpiF32 || p.b2 != nullptr) return 0;
    // What the other kernels take for the same: the fp32 instruction stops being fast enough at 48 to 96 rows, depending on how evenly the
    // columns divide (prompt of 64 rows, others -> this: dim 4096, 6 layers 2255 -> 2005 us, dim 5120, 4 layers 1866 -> 1991).
    double others = gemm_f32_instruction_us(p);
    const double parts = p.workspace == nullptr ? -1.0 : split3_us(p.m, p.n, p.k, p.ldc, p.workspace_bytes, p.compute_units);
    if (parts >= 0.0 && parts < others) others = parts;
    const double weights = 4.0 * p.n * (double)p.k / 5.6e6 + 10.0; // (neither estimate knows the memory; 4096 x 11008 of 16 rows: 53 us)
    if (others < weights) others = weights;
    if (p.b2 != nullptr) others = 2.0 * others + 5.0;
    const size_t per = (size_t)p.m * p.n * sizeof(float);
    const size_t room = p.workspace == nullptr ? 0 : p.workspace_bytes < kGemmPartialBytes ? p.workspace_bytes : kGemmPartialBytes;
    int best = 1;
    double best_us = rows_f32_us(p, 1);
    for (int pieces = 2; p.b2 == nullptr && pieces <= 8 && pieces * 4 <= p.k / 64 && pieces * per <= room && reinterpret_cast<uintptr_t>(p.workspace) % 16 == 0; pieces++) {
        const double us = rows_f32_us(p, pieces);
        if (us < best_us) {
            best = pieces;
            best_us = us;
        }
    }
    return best_us < 0.97 * others ? best : 0;
}

template <int kEpi>
static hipError_t launch_rows_f32_epi(const GemmParams &p, hipStream_t s) {
    switch (rows_fragments(p)) {
    case 1: return launch_rows_mf<kEpi, 1, true>(p, s);
    case 2: return launch_rows_mf<kEpi, 2, true>(p, s);
    case 3: return launch_rows_mf<kEpi, 3, true>(p, s);
    case 4: return launch_rows_mf<kEpi, 4, true>(p, s);
    case 6: return launch_rows_mf<kEpi, 6, true>(p, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_gemm_f32_rows(const GemmParams &p, int epilogue, hipStream_t s) {
    const int pieces = gemm_f32_rows_pieces(p, epilogue);
    if (pieces == 0) return hipErrorInvalidValue;
    if (epilogue == kGemmEpiSiluGateF32) return launch_rows_f32_epi<kGemmEpiSiluGateF32>(p, s);
    if (pieces == 1) return launch_rows_f32_epi<kGemmEpiF32>(p, s);
    GemmParams q = p; // partial sums: piece z into slice z of the work memory
    q.c = p.workspace;
    q.accumulate = 0;
    q.split_k = q.batch = pieces;
    q.ldc = p.n;
    q.stride_c = (size_t)p.m * p.n;
    const hipError_t e = launch_rows_f32_epi<kGemmEpiF32>(q, s);
    return e != hipSuccess ? e : launch_gemm_split_finish_f32(p, reinterpret_cast<const float *>(p.workspace), pieces, s);
}

} // namespace rlh
