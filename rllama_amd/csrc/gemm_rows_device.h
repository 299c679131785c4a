// gemm_rows_device.h -- C = A * B^T (f16 operands, fp32 accumulate) for prompts of up to 160 rows, one row tile for all of them.
//
// With so few rows the product is one pass over the weights B, and what a compute unit can take in bounds it: from memory while the rows
// are few, from L2 (every workgroup stages all of A) when they are many.  So a workgroup owns all rows and 16 to 64 columns: few
// enough that every compute unit has work, and up to 16384 columns enough that all workgroups run in one round (more columns take more rounds, where
// gemm_rows.hip compares with the other kernels).  Its wavefronts split K (K-group g takes the g-th 32 halves of every unit of K), so that an operand
// byte is written to LDS once and read back once or twice; and the weights are swept in whole 256-byte pieces of rows.  Every workgroup starts
// at another unit of K: workgroups in step ask for the same columns of all rows, i.e. for addresses a whole row apart, and those meet in few memory
// channels.  The partial sums of the K-groups are added through LDS in the order of the groups: deterministic, whole sums in the epilogue.
//
// What bounds it: few rows, memory (inside a prompt of 8 rows, us: wq|wk|wv 12288 x 4096 24.8 -> 20.0, w1|w3 11008 x 4096 39.5 -> 33.2 = 5.4 TB/s, w2
// 4096 x 11008 20.3 + 5.6 for adding the pieces -> 17.2); many rows, what a compute unit takes from L2 into LDS, 45 to 50 GB/s here (131 rows:
// wq|wk|wv 44 -> 35.8, w1|w3 58 -> 44; spreading the requests over the MFMAs, wavefronts of their own for them and units of 64 change
// nothing there).  Time to the first token, former kernels -> this: 7B shape 8 / 131 rows 3.61 -> 3.03 / 5.83 -> 4.72 ms; dim 2304, 10 layers,
// 8 / 24 / 64 rows 754 / 908 / 1001 -> 564 / 632 / 735 us; dim 2816, 8 layers, 112 / 144 rows 1095 / 1128 -> 832 / 910; dim 5120, 4 layers,
// 8 / 64 / 144 rows 754 / 932 / 1060 -> 649 / 763 / 982.  Beyond 160 rows the operand of activations alone fills the LDS.
//
// Weights are the first operand of v_mfma_f32_16x16x32_f16, so a lane ends up with four consecutive columns of one row.
#pragma once

#include "kernels.h"
#include "device_utils.h"
#include "gemm_epilogue.h"

#include <type_traits>

namespace rlh {

constexpr int kRowsMax = 160, kRowsF32Max = 96;
constexpr int kRowsFrags128 = 13; // fragments (rows and columns) of a workgroup up to which three units of 128 halves fit the LDS

// kMF x kNF: 16 x 16 fragments of a workgroup's tile (rows x columns of one product; kGemmEpiSiluGateF16 computes two products).
// kBK: halves of K per unit; K-group g of the kBK / 32 takes K-step g of every unit.  kRH x kCH: wavefronts of one K-group, over rows
// and columns (of both products).  kStages: units in LDS.
template <int kEpi, int kMF, int kNF, int kBK, int kRH, int kCH, int kStages>
struct RowsShape {
    static constexpr bool kDual = kEpi == kGemmEpiSiluGateF16 || kEpi == kGemmEpiSiluGateF32;
    static constexpr int kP = kDual ? 2 : 1;
    static constexpr int kKG = kBK / 32, kWaves = kKG * kRH * kCH, kThreads = 64 * kWaves;
    static constexpr int kNFt = kNF * kP, kMFw = kMF / kRH, kNFw = kNFt / kCH;
    static constexpr int kRowBytes = kBK * 2, kCpr = kBK / 8, kRpl = 512 / kBK;
    static constexpr int kRowsT = 16 * (kMF + kNFt);
    static constexpr int kStageBytes = kRowsT * kRowBytes;
    static constexpr int kGroups = kStageBytes / 1024;
    static constexpr int kLMax = (kGroups + kWaves - 1) / kWaves, kLMin = kGroups / kWaves;
    static constexpr int kLds = kStages * kStageBytes;
    static_assert(kMF % kRH == 0 && kNFt % kCH == 0, "whole fragments per wavefront");
    static_assert(kLds <= 160 * 1024, "LDS of one compute unit");
    static_assert(kBK == 64 || kBK == 128 || kBK == 256, "K-steps of 32 halves");
};

// kF32: the operands are fp32 (f32 mode).  Staging moves bytes and is the same with units of kBK / 2 floats; a 16-byte fragment then holds
// four consecutive k of a row and feeds four v_mfma_f32_16x16x4_f32 (k slot of lane group l / 16 in the j-th of them: float j of the group's
// chunk, for A and B alike).
template <int kEpi, int kMF, int kNF, int kBK, int kRH, int kCH, int kStages, bool kF32 = false>
__global__ __launch_bounds__(2 * kBK * kRH * kCH) void gemm_f16_rows_kernel(GemmParams p) {
    using S = RowsShape<kEpi, kMF, kNF, kBK, kRH, kCH, kStages>;
    constexpr bool kDual = S::kDual;
    constexpr int kKG = S::kKG, kWaves = S::kWaves, kThreads = S::kThreads, kNFt = S::kNFt, kMFw = S::kMFw, kNFw = S::kNFw;
    constexpr int kRowBytes = S::kRowBytes, kCpr = S::kCpr, kRpl = S::kRpl, kStageBytes = S::kStageBytes, kLMax = S::kLMax, kLMin = S::kLMin;
    constexpr int kBM = 16 * kMF, kBN = 16 * kNF;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pos = wave % (kRH * kCH), g = wave / (kRH * kCH), rh = pos % kRH, ch = pos / kRH;
    const int bx = blockIdx.x, bn0 = bx * kBN;
    constexpr int kE = kF32 ? 2 : 1; // halves per element: k and k offsets below are in halves
    const int M = p.m, N = p.n, K = p.k * kE;
    // split_k > 1: grid.z counts ranges of units of one product, C item z (stride_c apart) gets its partial sums (kGemmEpiF32 only)
    int u0 = 0, cnt = K / kBK;
    if (p.split_k > 1) {
        const int total = cnt, q = total / p.split_k, r = total % p.split_k, z = (int)blockIdx.z;
        cnt = q + (z < r ? 1 : 0);
        u0 = z * q + min(z, r);
    }
    // Where a workgroup starts: apart from those of its XCD, which are 8 launches apart, and from the other XCDs.  Chosen by time: among bx, bx >> 3 and bx & 7
    // plus 1, 3, 5 or 7 times bx >> 3 all are within 1.2 % over 15 products of 2 to 131 rows (in step 3.5 % slower, apart by XCD only 2.8), and 5 is the
    // fastest where it matters, long rows (8 rows, us, in step / bx / 1 / 3 / 5 / 7: 4096 x 11008 21.0 / 18.9 / 18.8 / 17.7 / 17.4 / 18.2, 24576 x 8192
    // 77.6 / 72.9 / 70.4 / 68.9 / 68.5 / 70.1).  It decides the order of the fp32 sums; any order is as good.
    const int rot = (int)(((unsigned)(bx >> 3) * 5u + (unsigned)(bx & 7)) % (unsigned)cnt);

    // ---- staging: rows of B (then of B2), then of A, 16-byte chunk c of row r at chunk c ^ swz(r): conflict-free fragment reads, and free
    //      here because every lane names its own global address.  Groups of kRpl rows (1 KiB) are dealt round-robin to the wavefronts.
    auto swz = [](int row) { return kBK == 64 ? (row >> 1) & 7 : row & 15; };
    const bool short_wave = kLMax != kLMin && (kLMax - 1) * kWaves + wave >= S::kGroups; // one load fewer
    const half_t *gbase[kLMax];
    unsigned voff[kLMax];
#pragma unroll
    for (int i = 0; i < kLMax; i++) {
        const int r0 = min(i * kWaves + wave, S::kGroups - 1) * kRpl; // uniform; a group lies within one matrix
        const int row2 = r0 + lane / kCpr;
        const int lc = (lane % kCpr) ^ swz(row2);
        if (r0 >= 16 * kNFt) {
            gbase[i] = p.a;
            voff[i] = (unsigned)((min(row2 - 16 * kNFt, M - 1) * p.lda * kE + lc * 8) * 2); // rows past the edge: a valid row, never stored
        } else {
            const bool second = kDual && r0 >= kBN;
            gbase[i] = (second ? p.b2 : p.b) + (size_t)bn0 * p.ldb * kE;
            voff[i] = (unsigned)((min(second ? row2 - kBN : row2, N - 1 - bn0) * p.ldb * kE + lc * 8) * 2);
        }
    }
    const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)lds_raw;
    int iss_slot = 0;
    int iss_ko = (u0 + rot) * kBK;
    const int ko_end = (u0 + cnt) * kBK, ko_0 = u0 * kBK;
    auto issue_load = [&](int i) { // load i of the next unit, in the order rot, rot + 1, ..., cnt - 1, 0, ...; issue_done behind each unit
        if (i < kLMin || !short_wave) dma16_base(gbase[i] + iss_ko, voff[i], lds_base + (unsigned)iss_slot * kStageBytes + (unsigned)wave * 1024 + i * (kWaves * 1024));
    };
    auto issue_done = [&]() {
        iss_ko += kBK;
        if (iss_ko == ko_end) iss_ko = ko_0;
        if (++iss_slot == kStages) iss_slot = 0;
    };

    // kF32: a unit's four MFMAs per fragment start from zero and are added to acc at its end, so that not all of K follows each other in
    // one register: a block of 8 rows, 7B / 1024-dim shape, is 1.42e-6 / 4.8e-7 from float64 with one running
    // sum and 6.0e-7 / 2.5e-7 like this (on the kernels for any number of rows 1.16e-6 / 3.3e-7).
    float4_t acc[kMFw][kNFw];
    [[maybe_unused]] float4_t part[kF32 ? kMFw : 1][kF32 ? kNFw : 1] = {};
#pragma unroll
    for (int i = 0; i < kMFw; i++)
#pragma unroll
        for (int j = 0; j < kNFw; j++) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

    // fragments: lane l supplies row l % 16, chunk 4 g + l / 16 of the unit.  Weights are the first operand: accumulator register v of
    // lane l is column 4 (l / 16) + v of row l % 16.
    const int frow = lane & 15;
    const int coff = ((g * 4 + (lane >> 4)) ^ swz(frow)) << 4;
    const int xa = (16 * kNFt + rh * kMFw * 16 + frow) * kRowBytes + coff, xb = (ch * kNFw * 16 + frow) * kRowBytes + coff;
    half8_t fa[2][kMFw], fb[2][kNFw];
    constexpr int kSlots = kMFw * kNFw, kReads = kMFw + kNFw;
    auto read_frag = [&](auto set, const unsigned char *stage, int r) {
        constexpr int s = decltype(set)::value;
        if (r < kNFw) fb[s][r] = *reinterpret_cast<const half8_t *>(stage + xb + r * (16 * kRowBytes));
        else fa[s][r - kNFw] = *reinterpret_cast<const half8_t *>(stage + xa + (r - kNFw) * (16 * kRowBytes));
    };
    // waits until at most kUnits units of this wavefront are outstanding
    auto wait_units = [&](auto units) {
        constexpr int kUnits = decltype(units)::value;
        if (kLMax == kLMin || !short_wave) wait_vmcnt<kUnits * kLMax>();
        else wait_vmcnt<kUnits * kLMin>();
    };
    auto wait_left = [&](int left) { // left: units that may stay outstanding
        if (left >= kStages - 2) wait_units(std::integral_constant<int, kStages - 2>{});
        else if (kStages > 3 && left == 1) wait_units(std::integral_constant<int, 1>{});
        else if (kStages > 4 && left == 2) wait_units(std::integral_constant<int, 2>{});
        else if (kStages > 5 && left == 3) wait_units(std::integral_constant<int, 3>{});
        else wait_vmcnt<0>();
    };
    const int fill = min(kStages, cnt);
    for (int t = 0; t < fill; t++) {
#pragma unroll
        for (int i = 0; i < kLMax; i++) issue_load(i);
        issue_done();
    }
    if (fill == kStages) wait_units(std::integral_constant<int, kStages - 1>{});
    else wait_vmcnt<0>();
    int slot = 0; // of unit t
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kReads; r++) read_frag(std::integral_constant<int, 0>{}, lds_raw, r);
    constexpr int kMmas = kF32 ? 4 * kSlots : kSlots; // of a unit; fp32: the first of every fragment pair, then the second of every pair, ...
    auto mma = [&](auto set, auto index) {
        constexpr int s = decltype(set)::value, x = decltype(index)::value, i = x % kSlots / kNFw, j = x % kNFw;
        if constexpr (kF32) {
            constexpr int e = x / kSlots;
            const float4_t b4 = __builtin_bit_cast(float4_t, fb[s][j]), a4 = __builtin_bit_cast(float4_t, fa[s][i]);
            if constexpr (e == 0) part[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b4[e], a4[e], float4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
            else part[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b4[e], a4[e], part[i][j], 0, 0, 0);
        } else {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[s][j], fa[s][i], acc[i][j], 0, 0, 0);
        }
    };
    // unit t: the fragments of unit t + 1 are read (kRead) and unit t + kStages is requested (kLoad) between its MFMAs
    auto step = [&](int t, auto set, auto rd, auto ld) {
        constexpr int s = decltype(set)::value;
        constexpr bool kRead = decltype(rd)::value, kLoad = decltype(ld)::value;
        if constexpr (kRead) {
            if constexpr (kLoad) wait_units(std::integral_constant<int, kStages - 2>{});
            else wait_left(cnt - 2 - t);
            __syncthreads(); // unit t + 1 is in LDS for everybody, and nobody reads unit t any more
            if (++slot == kStages) slot = 0;
        }
        const unsigned char *next = lds_raw + slot * kStageBytes;
        static_for<kMmas>([&](auto index) {
            constexpr int x = decltype(index)::value;
            if constexpr (kRead && x < kReads) read_frag(std::integral_constant<int, s ^ 1>{}, next, x);
            if constexpr (kRead && x == 0 && kReads > kMmas) {
#pragma unroll
                for (int r = kMmas; r < kReads; r++) read_frag(std::integral_constant<int, s ^ 1>{}, next, r);
            }
            mma(set, index);
            if constexpr (kLoad) {
                constexpr int lo = x * kLMax / kMmas, hi = (x + 1) * kLMax / kMmas;
#pragma unroll
                for (int i = lo; i < hi; i++) issue_load(i);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (kF32) {
#pragma unroll
            for (int i = 0; i < kMFw; i++)
#pragma unroll
                for (int j = 0; j < kNFw; j++) acc[i][j] += part[i][j];
        }
        if constexpr (kLoad) issue_done();
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    const int steady = cnt > kStages ? (cnt - kStages) & ~1 : 0; // units during which another one is requested, in pairs (the fragment sets alternate)
    int t = 0;
    for (; t < steady; t += 2) {
        step(t, even, yes, yes);
        step(t + 1, odd, yes, yes);
    }
    for (;; t += 2) {
        if (t + kStages < cnt) step(t, even, yes, yes);
        else if (t + 1 < cnt) step(t, even, yes, no);
        else { step(t, even, no, no); break; }
        if (t + 2 < cnt) step(t + 1, odd, yes, no);
        else { step(t + 1, odd, no, no); break; }
    }

    // ---- the K-groups' partial sums: every fragment of a position goes to one K-group, which adds them in the order of the groups.  (The
    //      fragments of both products at one place go to the same group where the epilogue works on registers.)
    constexpr int kF = kMFw * kNFw;
    constexpr bool kPairs = kEpi == kGemmEpiSiluGateF32;
    static_assert(!kPairs || kCH == 1, "both products in one wavefront");
    constexpr int kOwn = kPairs ? (kF / 2 + kKG - 1) / kKG * 2 : (kF + kKG - 1) / kKG;
    constexpr auto owner = [](int f) { return (kPairs ? f / kNFw * kNF + f % kNFw % kNF : f) % kKG; };
    constexpr auto slot_of = [](int f) { return kPairs ? (f / kNFw * kNF + f % kNFw % kNF) / kKG * 2 + f % kNFw / kNF : f / kKG; };
    auto row_of = [&](int f) { return (rh * kMFw + f / kNFw) * 16 + frow; };
    auto col_of = [&](int f) { return bn0 + (ch * kNFw + f % kNFw % (kPairs ? kNF : kNFw)) * 16 + (lane >> 4) * 4; };
    float4_t out[kOwn];
    [[maybe_unused]] float4_t prev[kF32 && kEpi == kGemmEpiF32 ? kOwn : 1]; // what the sums are added to, requested ahead of the exchange
    if constexpr (kF32 && kEpi == kGemmEpiF32) {
        static_for<kF>([&](auto fc) {
            constexpr int f = decltype(fc)::value;
            if (owner(f) == g) {
                const bool in = p.accumulate && row_of(f) < M && col_of(f) < N;
                prev[slot_of(f)] = in ? *reinterpret_cast<const float4_t *>(reinterpret_cast<const float *>(p.c) + (size_t)row_of(f) * p.ldc + col_of(f)) : float4_t{0, 0, 0, 0};
            }
        });
    }
    constexpr int kRoundMax = S::kLds / 1024 / kWaves;
    static_assert(kRoundMax >= 1, "a round of partial sums fits the stages");
    constexpr int kRound = kRoundMax < kF ? kRoundMax : kF;
    float4_t *xbuf = reinterpret_cast<float4_t *>(lds_raw);
    static_for<(kF + kRound - 1) / kRound>([&](auto round) {
        constexpr int f0 = decltype(round)::value * kRound, n_f = kF - f0 < kRound ? kF - f0 : kRound;
        __syncthreads(); // the stages (or the round before) have been read
        static_for<n_f>([&](auto fc) {
            constexpr int i = decltype(fc)::value, f = f0 + i;
            if (owner(f) != g) xbuf[((pos * kKG + g) * kRound + i) * 64 + lane] = acc[f / kNFw][f % kNFw];
        });
        __syncthreads();
        static_for<n_f>([&](auto fc) {
            constexpr int i = decltype(fc)::value, f = f0 + i;
            if (owner(f) == g) {
                float4_t sum;
                static_for<kKG>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    float4_t term;
                    if constexpr (q == owner(f)) term = acc[f / kNFw][f % kNFw];
                    else term = xbuf[((pos * kKG + q) * kRound + i) * 64 + lane];
                    if constexpr (q == 0) sum = term;
                    else sum = sum + term;
                });
                out[slot_of(f)] = sum;
            }
        });
    });
    if constexpr (kEpi == kGemmEpiF32 || kEpi == kGemmEpiSiluGateF32) {
        static_for<kF>([&](auto fc) {
            constexpr int f = decltype(fc)::value;
            if constexpr (!kPairs || f % kNFw < kNF) {
                if (owner(f) == g && row_of(f) < M && col_of(f) < N) {
                    float4_t o = out[slot_of(f)];
                    if constexpr (kPairs) {
                        const float4_t u = out[slot_of(f) + 1];
#pragma unroll
                        for (int e = 0; e < 4; e++) o[e] = (o[e] / (1.0f + expf(-o[e]))) * u[e]; // transformer.rs:557-565; tensor.rs:822-832, 722-734
                    }
                    if constexpr (kF32 && kEpi == kGemmEpiF32) {
                        if (p.accumulate) o = prev[slot_of(f)] + o;
                    }
                    *reinterpret_cast<float4_t *>(reinterpret_cast<float *>(p.c) + (size_t)blockIdx.z * p.stride_c + (size_t)row_of(f) * p.ldc + col_of(f)) = o;
                }
            }
        });
        return;
    } else {
        constexpr int kTW = 16 * kNFt, kTS = kTW + 8;
        static_assert(kBM * kTS * 2 <= S::kLds, "the output tile reuses the stages");
        half_t *tile = reinterpret_cast<half_t *>(lds_raw);
        __syncthreads();
#pragma unroll
        for (int f = 0; f < kF; f++)
            if (owner(f) == g) {
                typedef __attribute__((ext_vector_type(4))) _Float16 half4_t;
                half4_t o;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = (half_t)out[slot_of(f)][e]; // tensor.rs:1623-1643
                const int rr = row_of(f);
                if (rr >= M) o = half4_t{0, 0, 0, 0}; // (the padding of V^T has to be finite)
                *reinterpret_cast<half4_t *>(tile + rr * kTS + (ch * kNFw + f % kNFw) * 16 + (lane >> 4) * 4) = o;
            }
        __syncthreads();
        if constexpr (kEpi == kGemmEpiRopeQkv) {
            rope_qkv_from_tile<kBM, kTW, kTS, kThreads>(tile, tid, 0, bn0, M, N, kBM, p.rope);
        } else {
            constexpr int kChunks = kBN / 8;
#pragma unroll
            for (int it = 0; it < (kBM * kChunks + kThreads - 1) / kThreads; it++) {
                const int idx = it * kThreads + tid;
                const int rr = idx / kChunks, cc = (idx - rr * kChunks) * 8;
                const int c = bn0 + cc;
                if (rr < M && c < N) {
                    half8_t o = *reinterpret_cast<const half8_t *>(tile + rr * kTS + cc);
                    const size_t off = (size_t)rr * p.ldc + c;
                    if constexpr (kDual) {
                        const half8_t u = *reinterpret_cast<const half8_t *>(tile + rr * kTS + kBN + cc);
#pragma unroll
                        for (int e = 0; e < 8; e++) o[e] = to_f16(silu_fast((float)o[e]) * (float)u[e]); // tensor.rs:822-832 on the f16 gate
                    }
                    if constexpr (kEpi == kGemmEpiResAddF32) { // transformer.rs:442 / :445 on the f16-rounded product
                        const float4_t *res = reinterpret_cast<const float4_t *>(p.residual + off);
                        float4_t *dst = reinterpret_cast<float4_t *>(reinterpret_cast<float *>(p.c) + off);
                        float4_t r0 = res[0], r1 = res[1];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            r0[e] += (float)o[e];
                            r1[e] += (float)o[e + 4];
                        }
                        dst[0] = r0;
                        dst[1] = r1;
                    } else {
                        *reinterpret_cast<half8_t *>(reinterpret_cast<half_t *>(p.c) + off) = o;
                    }
                }
            }
        }
    }
}

// 16-row fragments of a product's tile.  From 65 rows on an even number (fp32: 6): their wavefronts split the rows in two, and two wavefronts per
// SIMD cover for each other's waits (7B shape, 131 rows: pieces of wo and w2 25.3 us on nine fragments and four wavefronts, 23.0 on ten and eight).
inline int rows_fragments(const GemmParams &p) {
    const int needed = (p.m + 15) / 16;
    return needed <= 4 ? needed : p.f32_operands ? 6 : (needed + 1) / 2 * 2;
}

// Microseconds per 1024 values of k that the workgroups of a product of `pieces` pieces take on nf x 16 columns each: rounds of
// workgroups x what a compute unit stages at 45 GB/s, or (fp32) what its matrix cores take at 0.45 TFLOP/s, whichever is longer.
inline double rows_us_k(const GemmParams &p, int pieces, int nf) {
    const int mf = rows_fragments(p), cols = nf * (p.b2 != nullptr ? 2 : 1);
    const long blocks = (long)((p.n + 16 * nf - 1) / (16 * nf)) * pieces, rounds = (blocks + p.compute_units - 1) / p.compute_units;
    const double staged = (mf + cols) * 16 * 1024.0 * (p.f32_operands ? 4 : 2) / 45e3;
    const double mfma = p.f32_operands ? 2.0 * 256 * mf * cols * 1024 / 0.45e6 : 0.0;
    return rounds * (staged > mfma ? staged : mfma);
}

// 16-column fragments per workgroup: the number that takes least (two fp32 products of many rows: as many as the registers hold).
inline int rows_columns(const GemmParams &p, int pieces) {
    const int most = p.f32_operands && p.b2 != nullptr ? (p.m > 64 ? 2 : p.m > 48 ? 3 : 4) : 4;
    int best = 1;
    for (int nf = 2; nf <= most; nf++)
        if (rows_us_k(p, pieces, nf) < rows_us_k(p, pieces, best)) best = nf;
    return best;
}

template <int kEpi, int kMF, int kNF, bool kF32, int kBKFixed = 0>
hipError_t launch_rows(const GemmParams &p, hipStream_t s) {
    // Units of 128 halves (whole 256-byte pieces of rows) while at least three fit the LDS, else of 64.  One fragment of rows and few
    // columns: 80 KB, so that two workgroups share a compute unit, and for long rows units of 256, i.e. twice the wavefronts.  2 to 16
    // rows of 1024 to 8192 columns, K = 6144 to 22016, units of 256 against 128: 0.86 to 1.07 of the time, mean 0.98, but 5120 columns (a quarter more
    // than one workgroup per compute unit) 1.0 to 1.13 up to K = 11008.  Below 6144 it depends on the columns alike (0.87 to 1.0 up to 4096 of them, 1.0 to 1.15 at
    // 5120 and 6656); with the residual and its norm, 4096 x 4096 of 8 rows: 9.1 us with units of 128, 10.8 with 256.
    if constexpr (kMF == 1 && kNF <= 2 && kBKFixed == 0 && !kF32 && kEpi != kGemmEpiSiluGateF16) {
        if (p.k >= 6144 && p.k % 256 == 0) return launch_rows<kEpi, kMF, kNF, kF32, 256>(p, s);
    }
    constexpr int kFrags = kMF + kNF * (kEpi == kGemmEpiSiluGateF16 || kEpi == kGemmEpiSiluGateF32 ? 2 : 1);
    constexpr int kBK = kBKFixed > 0 ? kBKFixed : kFrags <= kRowsFrags128 ? 128 : 64;
    constexpr int kFit = (kMF == 1 && kFrags <= 5 ? 80 : 160) * 32 / (kFrags * kBK); // units of kFrags * 32 * kBK bytes
    constexpr int kStages = kFit > 8 ? 8 : kFit > 6 && kMF > 1 ? 6 : kFit;
    constexpr int kCH = kEpi == kGemmEpiSiluGateF16 || (kBK == 64 && kEpi != kGemmEpiSiluGateF32) ? 2 : 1;
    constexpr int kRH = kMF % 2 == 0 && (kBK == 64 || (kMF >= 4 && kCH == 1)) ? 2 : 1;
    using S = RowsShape<kEpi, kMF, kNF, kBK, kRH, kCH, kStages>;
    const auto kern = gemm_f16_rows_kernel<kEpi, kMF, kNF, kBK, kRH, kCH, kStages, kF32>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds);
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL(kern, dim3((p.n + 16 * kNF - 1) / (16 * kNF), 1, p.split_k > 1 ? p.split_k : 1), dim3(S::kThreads), S::kLds, s, p);
    return hipGetLastError();
}

template <int kEpi, int kMF, bool kF32 = false>
hipError_t launch_rows_mf(const GemmParams &p, hipStream_t s) {
    switch (rows_columns(p, p.split_k > 1 ? p.split_k : 1)) {
    case 1: return launch_rows<kEpi, kMF, 1, kF32>(p, s);
    case 2: return launch_rows<kEpi, kMF, 2, kF32>(p, s);
    case 3:
        if constexpr (kEpi != kGemmEpiSiluGateF32 || kMF <= 4) return launch_rows<kEpi, kMF, 3, kF32>(p, s);
        return hipErrorInvalidValue;
    default:
        if constexpr (kEpi != kGemmEpiSiluGateF32 || kMF <= 3) return launch_rows<kEpi, kMF, 4, kF32>(p, s);
        return hipErrorInvalidValue;
    }
}

template <int kEpi>
hipError_t launch_rows_epi(const GemmParams &p, hipStream_t s) {
    switch (rows_fragments(p)) {
    case 1: return launch_rows_mf<kEpi, 1>(p, s);
    case 2: return launch_rows_mf<kEpi, 2>(p, s);
    case 3: return launch_rows_mf<kEpi, 3>(p, s);
    case 4: return launch_rows_mf<kEpi, 4>(p, s);
    case 6: return launch_rows_mf<kEpi, 6>(p, s);
    case 8: return launch_rows_mf<kEpi, 8>(p, s);
    case 10: return launch_rows_mf<kEpi, 10>(p, s);
    default: return hipErrorInvalidValue;
    }
}

} // namespace rlh
