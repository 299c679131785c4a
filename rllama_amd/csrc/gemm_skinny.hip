// gemm_skinny.hip -- C = A * B^T (f16 operands, fp32 accumulate) for prompts of at most 16 rows (one fragment; more would not be
// stored), where the product is one pass over the weights B and everything else should stay out of its way.
//
// The tiled kernels (gemm_dma.hip) stage B through LDS on 64 columns per workgroup: 172 workgroups for 11008 columns, 64 for
// 4096, so wo and w2 are cut along K and a second kernel adds the pieces.  Here a workgroup owns 16 columns (of one product, or
// of w1 and w3 alike) and its 16, 8 or 4 wavefronts split K among them; B goes from memory straight into the registers that feed
// v_mfma_f32_16x16x32_f16 (lane l: row l % 16, 8 values of k, 16 bytes), a burst of four K-steps in flight while the previous one
// is consumed, sixteen wavefronts per compute unit, and A -- a few rows, resident in L2 -- comes the same way.  The wavefronts'
// partial sums are added through LDS in the order of the wavefronts, so the result does not depend on timing, and the epilogue has
// whole sums: no second kernel.
//
// Products whose K is a multiple of 128 and whose columns are a multiple of 8 go to gemm_rows_device.h instead, which sweeps whole
// 256-byte pieces of rows and is faster (dim 2304, 10 layers, 8 rows: 754 -> 564 us to the first token).  Left here are other K, such as an odd
// number of heads of 64 (f16 prompts of dim 1088), other numbers of columns, and what GEMM_ROWS=0 sends here; the figures below, taken in part at multiples of
// 128, compare this kernel with the tiled ones.
//
// What bounds it: small products by the latency of their launches, larger ones by what the memory path takes in 64-byte pieces.
// Time to the first token at 2 / 8 / 16 rows, ms, tiled kernels -> this: dim 1024, 8 layers 0.50 / 0.52 / 0.53 -> 0.41 / 0.43 / 0.44; dim 2048,
// 16 layers 1.30 / 1.28 / 1.32 -> 0.99 / 1.05 / 1.16; 7B shape (wo only) 1 to 2 %.  At 17 to 32 rows the second
// fragment of A per fragment of B costs more than it saves (dim 2048, 32 rows: 1.44 against 1.54).
#include "kernels.h"
#include "device_utils.h"
#include "gemm_epilogue.h"

namespace rlh {

constexpr int kSkCols = 16;

template <int kEpi, bool kDual, int kSkWaves>
__global__ __launch_bounds__(64 * kSkWaves, 4) void gemm_f16_skinny_kernel(GemmParams p) {
    static_assert(kDual == (kEpi == kGemmEpiSiluGateF16), "two products share the SiLU-gate epilogue only");
    constexpr int kP = kDual ? 2 : 1;                     // products
    constexpr int kSkBurst = 4;                           // K-steps per burst: two bursts of B and A fragments fit 128 registers
    __shared__ float red[kSkWaves][kP][256];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int frow = lane & 15, fk = (lane >> 4) * 8;
    const int n0 = blockIdx.x * kSkCols;
    const int steps = p.k / 32, q = steps / kSkWaves, r = steps % kSkWaves;
    const int first = wave * q + min(wave, r), count = q + (wave < r ? 1 : 0); // this wavefront's K-steps

    // thread tid < 256 finishes the element that lane tid % 64 holds in accumulator register tid / 64
    const int o_row = (lane >> 4) * 4 + wave, o_col = n0 + frow;
    const bool o_in = tid < 256 && o_row < p.m && o_col < p.n;
    [[maybe_unused]] float res = 0.0f; // what the residual epilogue adds to, requested ahead of everything else
    if constexpr (kEpi == kGemmEpiResAddF32) res = o_in ? p.residual[(size_t)o_row * p.ldc + o_col] : 0.0f;

    // rows past the edges are clamped to a valid row; what they produce is not stored
    const half_t *bp[kP];
#pragma unroll
    for (int b = 0; b < kP; b++) bp[b] = (b ? p.b2 : p.b) + (size_t)min(n0 + frow, p.n - 1) * p.ldb + first * 32 + fk;
    const half_t *ap = p.a + (size_t)min(frow, p.m - 1) * p.lda + first * 32 + fk;

    float4_t acc[kP];
#pragma unroll
    for (int b = 0; b < kP; b++) acc[b] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    uint4_t wv[2][kP][kSkBurst], xv[2][kSkBurst];
    auto load = [&](int set, int s, int j) { // K-step s of this wavefront
#pragma unroll
        for (int b = 0; b < kP; b++) wv[set][b][j] = load16<true>(bp[b] + s * 32);
        xv[set][j] = load16<false>(ap + s * 32);
    };
    auto mma = [&](int set, int j) {
#pragma unroll
        for (int b = 0; b < kP; b++)
            acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, xv[set][j]), __builtin_bit_cast(half8_t, wv[set][b][j]), acc[b], 0, 0, 0);
    };
    // bursts of kSkBurst K-steps, the next one requested before the current one is consumed; in a partial one the last K-step is
    // requested again in place of those that do not exist
    auto request = [&](int set, int s) {
        if (s + kSkBurst <= count) {
#pragma unroll
            for (int j = 0; j < kSkBurst; j++) load(set, s + j, j);
        } else {
#pragma unroll
            for (int j = 0; j < kSkBurst; j++) load(set, min(s + j, count - 1), j);
        }
    };
    auto consume = [&](int set, int s) {
#pragma unroll
        for (int j = 0; j < kSkBurst; j++)
            if (s + j < count) mma(set, j);
    };
    if (count > 0) {
        request(0, 0);
        for (int s = 0;; s += 2 * kSkBurst) {
            const bool more1 = s + kSkBurst < count, more2 = s + 2 * kSkBurst < count;
            if (more1) request(1, s + kSkBurst);
            consume(0, s);
            if (!more1) break;
            if (more2) request(0, s + 2 * kSkBurst);
            consume(1, s + kSkBurst);
            if (!more2) break;
        }
    }

#pragma unroll
    for (int b = 0; b < kP; b++)
#pragma unroll
        for (int v = 0; v < 4; v++) red[wave][b][v * 64 + lane] = acc[b][v];
    __syncthreads();
    constexpr int kTS = kSkCols + 8;
    __shared__ __attribute__((aligned(16))) half_t tile[kEpi == kGemmEpiRopeQkv ? 64 * kTS : 8];
    if (tid < 256) {
        float sum[kP];
#pragma unroll
        for (int b = 0; b < kP; b++) {
            sum[b] = red[0][b][tid];
#pragma unroll
            for (int w = 1; w < kSkWaves; w++) sum[b] += red[w][b][tid];
        }
        const size_t off = (size_t)o_row * p.ldc + o_col;
        if constexpr (kEpi == kGemmEpiRopeQkv) {
            tile[o_row * kTS + frow] = o_row < p.m ? (half_t)sum[0] : (half_t)0.0f; // tensor.rs:1623-1643
        } else if (o_in) {
            if constexpr (kEpi == kGemmEpiF16) reinterpret_cast<half_t *>(p.c)[off] = (half_t)sum[0]; // tensor.rs:1623-1643
            else if constexpr (kEpi == kGemmEpiSiluGateF16) reinterpret_cast<half_t *>(p.c)[off] = to_f16(silu_fast(f16r(sum[0])) * f16r(sum[kP - 1])); // tensor.rs:822-832
            else reinterpret_cast<float *>(p.c)[off] = res + f16r(sum[0]); // transformer.rs:442 / :445
        }
    }
    if constexpr (kEpi == kGemmEpiRopeQkv) {
        // the tile of 64 rows covers a whole key tile of the attention kernel: rows past m are zeros, finite padding of V^T
        for (int i = tid + 16 * kTS; i < 64 * kTS; i += 64 * kSkWaves) tile[i] = (half_t)0.0f;
        __syncthreads();
        if (wave == 0) rope_qkv_from_tile<64, kSkCols, kTS>(tile, lane, 0, n0, p.m, p.n, 64, p.rope);
    }
}

bool gemm_f16_skinny_supported(const GemmParams &p, int epilogue) {
    if (p.tune.no_skinny || p.tune.dual_plus1 != 0 || p.tune.tile_plus1 != 0 || p.tune.split_k != 0 || p.f32_operands || p.batch != 1 || p.split_k > 1 || p.k_seg != 0 || p.causal != 0) return false;
    if (p.m < 1 || p.m > 16 || p.n < 1 || p.k < 1024 || p.k % 32 != 0 || p.lda % 8 != 0 || p.ldb % 8 != 0) return false;
    // (rows shorter than 1024 are not measured: they leave sixteen wavefronts less than two K-steps each; results are right there too)
    // Fragments of 16 rows are 64 bytes per row and load instruction, which the memory path takes at about 4.7 TB/s; large products
    // are faster through LDS in whole lines in spite of their second kernel (7B shape, 8 rows: w1|w3 42 us here, 36 there)
    if ((size_t)p.n * p.k * (p.b2 != nullptr ? 4 : 2) > ((size_t)48 << 20)) return false;
    // What the tiled kernels do better (while K is whole K-tiles of theirs), us, tiled -> this:
    const int tiles = (p.n + kSkCols - 1) / kSkCols, n_cu = p.compute_units;
    if (p.k % 64 == 0 && tiles > n_cu) {
        // Two products on more workgroups than compute units (w1|w3 of 5632 x 2048, 8 / 16 rows: 18.6 -> 19.1 / 20.6; 5120 x 1408: 15.5 -> 17.4 / 19.2).
        if (p.b2 != nullptr) return false;
        // One product: eight or four wavefronts share K, and a burst that is not whole requests its last K-step again (8192 columns, 8 / 16 rows:
        // K = 2048 14.5 -> 12.9 / 13.6, 1536 13 -> 12.5 / 13.9, 1280 12.2 -> 12.9 / -, 2560 17 -> 16.7 / 18.5; 11008 x 2048 15.7 -> 14.8 / 17.1, x 1792
        // 14.2 -> 15.3 / -).  Beyond K = 3072 the tiled kernels need two launches.
        const bool whole = p.k % 1024 == 0;
        if (tiles > 2 * n_cu ? !whole || p.m > 8 : !whole && p.k <= 3072 && p.m > (p.k < 1408 ? 4 : 10)) return false;
    }
    // Long rows, where each wavefront's chain of bursts is long and the tiled kernels cut K further: sooner where their 64-wide tiles and pieces
    // make exactly one round (2048 columns, 7 / 12 / 16 rows: K = 4096 14.5 -> 12 / 12 / 12.5, 5632 15.8 -> 15.2 / 16.1 / 17.2, 8192 18 -> 18 / 19.4 / 20.8;
    // 7 rows, K = 6912 15.7 -> 17.9; but 2816 columns 26 -> 18.7 / 19.8 / 21 at K = 8192).
    if (p.b2 == nullptr && (p.k > 8192 || (n_cu % ((p.n + 63) / 64) == 0 && p.k > 4096 && (p.m * p.k > 40000 || (p.k > 6144 && p.k % 2048 != 0))))) return false;
    if ((reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.b) | reinterpret_cast<uintptr_t>(p.b2)) % 16 != 0) return false;
    switch (epilogue) {
    case kGemmEpiF16: return p.b2 == nullptr;
    case kGemmEpiResAddF32: return p.b2 == nullptr && p.residual != nullptr;
    case kGemmEpiSiluGateF16: return p.b2 != nullptr;
    case kGemmEpiRopeQkv: return p.b2 == nullptr;
    default: return false;
    }
}

template <int kEpi, bool kDual>
static hipError_t launch_skinny(const GemmParams &p, hipStream_t s) {
    // sixteen wavefronts fit a compute unit: as many per workgroup as let all workgroups run at once
    const int tiles = (p.n + kSkCols - 1) / kSkCols;
    [[maybe_unused]] const int n_cu = p.compute_units;
    if constexpr (kDual) hipLaunchKernelGGL((gemm_f16_skinny_kernel<kEpi, kDual, 16>), dim3(tiles), dim3(1024), 0, s, p);
    else if (tiles <= n_cu) hipLaunchKernelGGL((gemm_f16_skinny_kernel<kEpi, kDual, 16>), dim3(tiles), dim3(1024), 0, s, p);
    else if (tiles <= 2 * n_cu) hipLaunchKernelGGL((gemm_f16_skinny_kernel<kEpi, kDual, 8>), dim3(tiles), dim3(512), 0, s, p);
    else hipLaunchKernelGGL((gemm_f16_skinny_kernel<kEpi, kDual, 4>), dim3(tiles), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_gemm_f16_skinny(const GemmParams &p, int epilogue, hipStream_t s) {
    if (!gemm_f16_skinny_supported(p, epilogue)) return hipErrorInvalidValue;
    switch (epilogue) {
    case kGemmEpiF16: return launch_skinny<kGemmEpiF16, false>(p, s);
    case kGemmEpiResAddF32: return launch_skinny<kGemmEpiResAddF32, false>(p, s);
    case kGemmEpiSiluGateF16: return launch_skinny<kGemmEpiSiluGateF16, true>(p, s);
    case kGemmEpiRopeQkv: return launch_skinny<kGemmEpiRopeQkv, false>(p, s);
    default: return hipErrorInvalidValue;
    }
}

} // namespace rlh
