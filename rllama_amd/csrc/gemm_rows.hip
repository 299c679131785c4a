// gemm_rows.hip -- products of a model's short prompts and of the op-level tensors (at most 160 rows): which ones, in how many pieces along K,
// and the plain epilogues.  The kernel is in gemm_rows_device.h; gemm_rows_fused.hip holds w1|w3 and wq|wk|wv.
#include "gemm_rows_device.h"

namespace rlh {

hipError_t launch_gemm_f16_rows_fused(const GemmParams &p, int epilogue, hipStream_t s); // gemm_rows_fused.hip

// Whether what of A the pieces of one round read (all of K: workgroups start all over it) is more than one XCD's L2 of 4 MB keeps beside the
// weights that pass through.
static bool rows_beyond_l2(const GemmParams &p, int pieces, long rounds) { return 2.0 * p.m * p.k * ((pieces + rounds - 1) / rounds) / pieces > 3.25 * (1 << 20); }

// Microseconds of a product in `pieces` pieces with what has to follow it: a launch, then what one compute unit stages at 45 GB/s (twice that
// where at most an eighth of them work) or all of the weights at 5.6 TB/s.  Units of 128 halves are staged slower where A is beyond the L2
// (8192 x 22016, 128 rows: one round of 2 pieces 149 us, two rounds of 4 pieces 108).  Partial sums are written and read back at 2.5 TB/s, all in
// all (taken as 4.7, 12288 x 6144 of 160 rows ran in 4 pieces, 65 us, and 512 x 4096 of 2 rows in 8, 9.2 us; 47 and 5.0 in one).
// The kernel that adds the pieces brings the RMSNorm behind a residual product along.
static double rows_us(const GemmParams &p, int epilogue, int pieces) {
    const double k = ((p.k / 128 + pieces - 1) / pieces) * 128.0;
    const int nf = rows_columns(p, pieces);
    const long blocks = (long)((p.n + 16 * nf - 1) / (16 * nf)) * pieces, rounds = (blocks + p.compute_units - 1) / p.compute_units;
    double staged = k / 1024 * rows_us_k(p, pieces, nf);
    if (rows_fragments(p) + nf <= kRowsFrags128 && rows_beyond_l2(p, pieces, rounds)) staged *= 1.4;
    if (blocks <= p.compute_units / 8) staged *= 0.5;
    const double weights = 2.0 * p.n * (double)p.k * (p.b2 != nullptr ? 2 : 1) / 5.6e6;
    double us = 3.0 + (staged > weights ? staged : weights);
    if (pieces > 1) us += 4.0 + 4.0 * pieces * (double)p.m * p.n / 2.5e6;
    if (epilogue == kGemmEpiResAddF32 && p.norm_w != nullptr) us += pieces > 1 ? 1.2 : 4.8;
    return us;
}

// What the kernels for any number of rows do better from 65 rows on, among 2500 plain products of 2 to 160 rows, 512 to 65536 columns, K = 128 to
// 22016 and the products of prompts of ten dims (us, this kernel -> those):
static bool rows_other_kernels(const GemmParams &p, int epilogue, int pieces) {
    if (p.m <= 64 || p.b2 != nullptr) return false;
    const long n_cu = p.compute_units, blocks64 = (p.n + 63) / 64, rounds = (blocks64 + n_cu - 1) / n_cu;
    // More than one round of the widest workgroups: every round stages all rows again, and a last one that is partly empty takes as long (128 rows:
    // 18432 x 4096 70 -> 50, 22016 x 1024 20.1 -> 17.0, 32000 x 2048 38 -> 35; 96 rows, 32000 x 5120 80 -> 71).  This kernel stays the better one where the
    // rounds are full and K is long, the sooner if their 128-column tiles need a second round too (65 rows, 32000 x 8192: 97 against 111; 49152 x 1536: 39
    // against 43; 128 rows, 49152 x 8192 186 against 220) or beyond 128 rows, where they need a second row tile (131 rows, 32000 x 4096 70 against 81, 24576 x 8192
    // 118 against 126); with RoPE their tiles are wide (wq|wk|wv of dim 8192, 65 / 112 / 131 rows: 90 / 107 / 124 against 96 / 100 / 134).
    if (rounds > 1) {
        const double full = (double)blocks64 / (rounds * n_cu);
        bool worth;
        if (epilogue == kGemmEpiRopeQkv) worth = full >= 0.75 && p.k >= 6144 && (p.m <= 96 || p.m > 128);
        else if (p.m <= 96) worth = full >= 0.9 && p.k >= (rounds > 2 ? 1536 : 8192) && p.k <= 11008;
        else if (p.m <= 128) worth = full >= 0.9 && rounds > 2 && p.k >= 6144;
        else if (p.m <= 144) worth = p.k >= 8192 || (full >= 0.9 && p.k >= 4096);
        else worth = full >= 0.9 && p.k >= 8192;
        if (!worth) return true;
    }
    // Cut, where their 64-column tiles make one round whole: the second kernel costs more than the wider staging saves (128 rows: 4096 x 2048 15.0 -> 11.4, 3072 x 1536
    // 12.8 -> 9.4, 3072 x 2560 15.1 -> 13.4, 1536 x 1536 10.6 -> 8.5; but 512 x 2048 7.8 against 10.1, 1536 x 2560 11 against 13).  Products that the RMSNorm follows
    // need a second kernel either way.
    if (epilogue == kGemmEpiF16 && pieces > 1 && p.n >= 1024 && p.k <= (p.n >= 3072 ? 2560 : 2048) &&
        p.m > (p.k <= 1536 || (p.n >= 3072 && p.k <= 2048) ? 64 : 96) && gemm_f16_narrow(p)) return true;
    // One round with A beyond the L2, against cut products of few columns that divide the compute units evenly (K = 22016, 128 rows, 2048 / 4096 columns:
    // 47 / 82 -> 37 / 61, w2 of the 7B shape, 160 rows: 42 -> 37; but 3072 columns 64 against 73, 8192 columns of 131 rows 111 against 122).
    const int nf = rows_columns(p, pieces);
    return p.n >= 1024 && blocks64 <= n_cu / 4 && n_cu % blocks64 == 0 && (long)((p.n + 16 * nf - 1) / (16 * nf)) * pieces <= n_cu &&
           rows_beyond_l2(p, pieces, 1);
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
    case kGemmEpiRopeQkv: return p.b2 == nullptr && !rows_other_kernels(p, epilogue, 1) ? 1 : 0;
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
    return rows_other_kernels(p, epilogue, best) ? 0 : best;
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
