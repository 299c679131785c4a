// gemm_split3.hip -- C = A * B^T on fp32 operands (f32 mode, tensor.rs:1282-1475 for src.rows > 1) through the bf16 matrix
// cores, at fp32 precision.
//
// The fp32 matrix instruction (v_mfma_f32_32x32x2_f32, gemm_dma.hip) retires 64 flop per cycle and SIMD, the bf16 one 1024.
// Every fp32 value is the sum of three bf16 values exactly -- hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi - mid), 8 + 8 +
// 8 significand bits plus the signs of mid and lo against the 24 of x -- and of the nine products of two such sums the six
// largest are taken:  lo hi' + hi lo' + mid mid' + mid hi' + hi mid' + hi hi' (the splitting of Henry, Tang and Heinecke, "Leveraging the
// bfloat16 artificial intelligence datatype for higher-precision computations", 2019).  What is left out, mid lo' and lo mid' of up to
// 2^-25 of a product each and lo lo' of 2^-34, is at most 2^-24 of it, one rounding of fp32.  The sums are fp32 like before, and there are fewer of them: one
// addition to the accumulator per 16 values of k and product instead of one per 2.  Six bf16 products cost 6/16 of the fp32
// instruction's cycles.
//
// Both operands are multiplied by 2^16 first and the sums by 2^-32 at the end, all exact: the last bit of the smallest fp32 number,
// 2^-149, becomes 2^-133, the last bit of a bf16 number, so the parts hold every value however small.  (Without it values below 2^-109
// lose bits: 2-norm error 2.2e-3 at 2^-126.)
//
// Values that the decomposition cannot hold (infinities, and finite values from 2^112 on, whose bf16 part is infinite: x - hi is then not
// a remainder), and sums from 2^96 on, make every product they enter NaN or infinite.  An element of C that comes out non-finite is
// therefore computed again, with the fp32 matrix instruction on the operands themselves, so infinities and NaN are those of the plain sum.
// (A wavefront repeats every 32 x 32 tile that holds such an element.  Call of 200 x 11008 x 4096, 225 us without one: one NaN in A
// 290 us, one infinity in B 450, NaN in every row 640; the fp32 instruction throughout 340.)
//
// A (the activations, few rows) is decomposed once by a kernel of its own into three bf16 planes laid out as the LDS image of a
// K-tile, so that staging it is a linear copy.  B (the weights, read once) is staged as fp32 and decomposed by the wavefront
// that feeds it to the matrix cores: 9 vector instructions per pair of values against 12 MFMAs per fragment and row tile.
//
// Blocking.  A workgroup owns 32 kT rows x 128 columns and has eight wavefronts: 2 row groups x 2 column groups x 2 K-groups
// (K-group g takes the g-th 16 of the 32 values of k in a K-tile).  A wavefront's tile is up to 128 x 64, which needs 16 KB of
// LDS reads per 48 MFMAs (1536 cycles); with eight wavefronts and the staging that is about 62 bytes per cycle and compute unit at
// 256 rows.  The K-groups' sums are added through LDS at the end.  A's stages are as deep as LDS allows beside four or more
// stages of B, whose latency is the HBM's.  With an odd number of 32-row tiles the row groups are one tile apart; the K-groups
// swap row groups, so that every SIMD gets one wavefront of each size.
//
// What bounds it: 1024 rows x 4096 x 11008 runs its matrix pipes 65 % busy at 1.93 GHz (power); with fewer rows, 58 % on the
// compute units that have a tile.  Against the fp32 instruction, decomposition of A and sum of the pieces included, us:
// 11008 x 4096 weights, 16 / 64 / 128 / 200 / 300 / 1024 rows: 87 / 143 / 155 / 270 / 445 / 795 -> 52 / 74 / 97 / 139 / 192 / 541;
// 4096 x 11008: 68 / 105 / 125 / 205 / 394 / 705 -> 53 / 65 / 87 / 121 / 163 / 448.  7B shape, 200 prompt rows: 38.0 -> 21.0 ms.
// Error against float64 (2-norm, 200 x 12288 x 4096): 5.0e-7 where the fp32 instruction has 1.15e-6 (fewer additions).
// Products whose tiles do not fill the compute units are cut along K (partial sums in the workspace, added in order of the
// pieces by gemm_split_finish_kernel).
#include "kernels.h"
#include "device_utils.h"
#include "split3_plan.h"

#include <type_traits>

namespace rlh {

typedef __attribute__((ext_vector_type(16))) float float16_t;
typedef __attribute__((ext_vector_type(8))) float float8_t;
typedef __attribute__((ext_vector_type(8))) __bf16 bf8_t;

constexpr int kS3Waves = 8;
constexpr float kS3Scale = 65536.0f; // of every operand, exact: keeps the parts of the smallest values
constexpr float kS3Unscale = 1.0f / (kS3Scale * kS3Scale);
constexpr int kS3BStage = kS3Cols * kS3K * 4;
constexpr int s3_a_stage(int t) { return 3 * t * 32 * kS3K * 2; }
constexpr int s3_a_stages(int t) { return t >= 6 ? 2 : t >= 4 ? 3 : 4; }
constexpr int s3_b_stages(int t) {
    const int left = (160 * 1024 - s3_a_stages(t) * s3_a_stage(t)) / kS3BStage;
    return left > 8 ? 8 : left;
}

struct Split3Params {
    const float *a, *b;
    float *c;
    const unsigned char *planes; // [k / 32][3][m_pad][32] bf16, 16-byte chunk c of row r at chunk c ^ ((r / 4) % 4)
    int m, n, k, lda, ldb, ldc;
    int m_pad;                   // row tiles x 32 kT
    int accumulate;
    int split_k;
    size_t stride_c;             // elements between the pieces' partial sums
};

// x - hi and the next remainder as v_dot2_f32_bf16 of the converted pair with (-1, 0) or (0, -1): one instruction instead of taking a half
// out of the pair and subtracting it, and exact for all finite values, subnormals and pairs of any two magnitudes among them (checked
// against the subtraction).  The constants come out of registers on purpose: as literals they are not what the instruction reads.  11 vector
// instructions per pair of values without, 9 with it and the scale; call of 11008 x 4096 weights, 8 / 64 / 200 / 1024 rows, no scale and no
// dot product -> both: 49 / 75 / 171 / 538 -> 45 / 68 / 141 / 541 us (scale alone: 53 / 80 / 174 / 560, 3 % of a 7B prompt of 64 to 100 rows).
__device__ __forceinline__ void split3(const float8_t x_in, bf8_t &hi, bf8_t &mid, bf8_t &lo) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf2_t;
    unsigned c0 = 0x0000bf80u, c1 = 0xbf800000u; // (-1, 0) and (0, -1)
    asm("" : "+s"(c0), "+s"(c1));
    const bf2_t first = __builtin_bit_cast(bf2_t, c0), second = __builtin_bit_cast(bf2_t, c1);
    float8_t x = x_in * kS3Scale;
    auto rest = [&](const bf8_t part) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const bf2_t pair = {part[e], part[e + 1]};
            x[e] = __builtin_amdgcn_fdot2_f32_bf16(pair, first, x[e], false);
            x[e + 1] = __builtin_amdgcn_fdot2_f32_bf16(pair, second, x[e + 1], false);
        }
    };
    hi = __builtin_convertvector(x, bf8_t);
    rest(hi);
    mid = __builtin_convertvector(x, bf8_t);
    rest(mid);
    lo = __builtin_convertvector(x, bf8_t);
}

// A [m x k] fp32 -> planes.  Four threads per row and K-tile: a wavefront reads 16 rows x 128 bytes and writes 1 KiB per plane.
__global__ __launch_bounds__(256) void split3_rows_kernel(const float *a, unsigned char *planes, int m, int m_pad, int k, int lda) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int c = (int)(idx & 3);
    const size_t rk = idx >> 2;
    const int r = (int)(rk % (size_t)m_pad), kt = (int)(rk / (size_t)m_pad);
    if (kt >= k / kS3K) return;
    float8_t x = {0, 0, 0, 0, 0, 0, 0, 0};
    if (r < m) {
        const float4_t *src = reinterpret_cast<const float4_t *>(a + (size_t)r * lda + kt * kS3K + c * 8);
        const float4_t u = src[0], v = src[1];
        x = float8_t{u[0], u[1], u[2], u[3], v[0], v[1], v[2], v[3]};
    }
    bf8_t pl[3];
    split3(x, pl[0], pl[1], pl[2]);
#pragma unroll
    for (int p = 0; p < 3; p++)
        *reinterpret_cast<bf8_t *>(planes + (((size_t)kt * 3 + p) * m_pad + r) * (kS3K * 2) + ((c ^ ((r >> 2) & 3)) << 4)) = pl[p];
}

template <int kT>
__global__ __launch_bounds__(64 * kS3Waves) void gemm_split3_kernel(Split3Params p) {
    constexpr int kRows = 32 * kT;
    constexpr int kAStages = s3_a_stages(kT), kBStages = s3_b_stages(kT);
    constexpr int kAStage = s3_a_stage(kT), kPlane = kRows * kS3K * 2;
    constexpr int kAGroups = kAStage / 1024, kLA = (kAGroups + kS3Waves - 1) / kS3Waves;
    constexpr int kLB = kS3BStage / 1024 / kS3Waves;
    constexpr int kN0 = (kT + 1) / 2, kN1 = kT / 2; // 32-row tiles of row group 0 and 1
    static_assert(kBStages > kAStages && kAStages >= 2, "the waits below count on it");
    static_assert(kAStages * kAStage + kBStages * kS3BStage <= 160 * 1024, "LDS of one compute unit");
    static_assert(kS3Waves * kN0 * 4096 <= kAStages * kAStage + kBStages * kS3BStage, "the exchanged sums reuse the stages");
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds_raw[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wave >> 2, wn = wave & 1, wm = ((wave >> 1) & 1) ^ kg;
    int bx = blockIdx.x, by = blockIdx.y;
    if (gridDim.y > 1 && gridDim.x % 8 != 0) {
        // workgroups go to the 8 XCDs round-robin in launch order: keep the row tiles of one column tile on one XCD
        const int nx = gridDim.x, ny = gridDim.y;
        const int L = by * nx + bx, per = 8 * ny;
        const int chunk = L / per, j = L - chunk * per;
        const int w = min(8, nx - chunk * 8);
        by = j / w;
        bx = chunk * 8 + (j - by * w);
    }
    const int bm0 = by * kRows, bn0 = bx * kS3Cols;
    // piece z of a product cut along K: K-tiles [z q + min(z, r), ...) of the split_k q + r tiles
    int kt0 = 0, n_kt = p.k / kS3K;
    if (p.split_k > 1) {
        const int q = n_kt / p.split_k, r = n_kt % p.split_k, z = (int)blockIdx.z;
        kt0 = z * q + min(z, r);
        n_kt = q + (z < r ? 1 : 0);
    }

    // ---- staging: A's stages, then B's.  1 KiB per wavefront-wide load; every wavefront issues kLA + kLB loads per K-tile
    //      (a wavefront without a group of its own left repeats the last one: same bytes, same place).
    unsigned voff_a[kLA], dst_a[kLA], voff_b[kLB];
#pragma unroll
    for (int i = 0; i < kLA; i++) {
        const int g = min(i * kS3Waves + wave, kAGroups - 1);
        const int plane = g / (2 * kT), rg = g - plane * (2 * kT);
        voff_a[i] = (unsigned)((plane * p.m_pad + rg * 16) * (kS3K * 2) + lane * 16);
        dst_a[i] = (unsigned)g * 1024;
    }
#pragma unroll
    for (int i = 0; i < kLB; i++) {
        const int row = (i * kS3Waves + wave) * 8 + (lane >> 3);
        const int lc = (lane & 7) ^ ((row >> 1) & 7);
        voff_b[i] = (unsigned)((min(bn0 + row, p.n - 1) - bn0) * p.ldb * 4 + lc * 16); // columns past the edge: a valid one, never stored
    }
    const unsigned lds_base = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)lds_raw;
    const unsigned lds_b = lds_base + kAStages * kAStage;
    const unsigned char *src_a = p.planes + (size_t)bm0 * (kS3K * 2);
    const float *src_b = p.b + (size_t)bn0 * p.ldb;
    auto issue_a = [&](int t) { // past the end the last K-tile is loaded again (keeps the in-flight count constant)
        const int kt = kt0 + min(t, n_kt - 1);
        const half_t *base = reinterpret_cast<const half_t *>(src_a + (size_t)kt * 3 * p.m_pad * (kS3K * 2));
        const unsigned dst = lds_base + (unsigned)(t % kAStages) * kAStage;
#pragma unroll
        for (int i = 0; i < kLA; i++) dma16_base(base, voff_a[i], dst + dst_a[i]);
    };
    auto issue_b = [&](int t) {
        const int kt = kt0 + min(t, n_kt - 1);
        const half_t *base = reinterpret_cast<const half_t *>(src_b + (size_t)kt * kS3K);
        const unsigned dst = lds_b + (unsigned)(t % kBStages) * kS3BStage + (unsigned)wave * 1024;
#pragma unroll
        for (int i = 0; i < kLB; i++) dma16_base(base, voff_b[i], dst + i * (kS3Waves * 1024));
    };

    // ---- the loop of one wavefront over kNI 32-row tiles; both row groups pass the same barriers
    auto run = [&](auto n_tiles, int tile0) {
        constexpr int kNI = decltype(n_tiles)::value;
        constexpr int kA = kNI > 0 ? kNI : 1;
        float16_t acc[kA][2];
#pragma unroll
        for (int i = 0; i < kA; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
        const int frow = lane & 31, half = lane >> 5;
        const int a_off = (tile0 * 32 + frow) * (kS3K * 2) + (((kg * 2 + half) ^ ((frow >> 2) & 3)) << 4);
        const int b_row = (wn * 64 + frow) * (kS3K * 4), b_sw = (frow >> 1) & 7, b_c = kg * 4 + half * 2;
        bf8_t af[2][3], bs[2][2][3];
        auto read_a = [&](int set, int t, int i) {
            const unsigned char *s = lds_raw + (t % kAStages) * kAStage + a_off + i * (32 * kS3K * 2);
#pragma unroll
            for (int q = 0; q < 3; q++) af[set][q] = *reinterpret_cast<const bf8_t *>(s + q * kPlane);
        };
        auto split_b = [&](int set, int t, int j) {
            const unsigned char *s = lds_raw + kAStages * kAStage + (t % kBStages) * kS3BStage + b_row + j * (32 * kS3K * 4);
            const float4_t u = *reinterpret_cast<const float4_t *>(s + ((b_c ^ b_sw) << 4));
            const float4_t v = *reinterpret_cast<const float4_t *>(s + (((b_c + 1) ^ b_sw) << 4));
            split3(float8_t{u[0], u[1], u[2], u[3], v[0], v[1], v[2], v[3]}, bs[set][j][0], bs[set][j][1], bs[set][j][2]);
        };
        // Loads in the order the loop issues them: at the end of K-tile t, A's t + kAStages and B's t + kBStages + 1 (B runs one
        // K-tile further ahead: the fragments of K-tile t + 1 are read and decomposed under the MFMAs of K-tile t)
#pragma unroll
        for (int s = 0; s < kBStages; s++) {
            issue_b(s);
            if (s + 1 > kBStages - kAStages) issue_a(s - (kBStages - kAStages));
        }
        wait_vmcnt<kBStages * kLB + kAStages * kLA - kLB>();
        __syncthreads(); // B's K-tile 0
        if constexpr (kNI > 0) {
            split_b(0, 0, 0);
            split_b(0, 0, 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads(); // ... is read
        issue_b(kBStages);
        wait_vmcnt<kLB + (kAStages - 1) * (kLA + kLB)>();
        __syncthreads(); // A's K-tile 0 and B's K-tile 1
        if constexpr (kNI > 0) read_a(0, 0, 0);
        auto k_tile = [&](int t, auto parity) { // parity of t
            constexpr int kBCur = decltype(parity)::value, kBNxt = kBCur ^ 1;
            constexpr int kP = (kBCur * kNI) & 1; // A fragment set of row tile 0
#pragma unroll
            for (int i = 0; i < kA; i++) {
                [[maybe_unused]] const int cur = (i + kP) & 1, nxt = cur ^ 1;
                if constexpr (kNI > 0) {
                    if (i == 0) split_b(kBNxt, t + 1, 0);
                    if (i == (kNI > 1 ? 1 : 0)) split_b(kBNxt, t + 1, 1);
                }
                if (i + 1 < kA) {
                    read_a(nxt, t, i + 1);
                } else {
                    // the K-tile change, in front of the last row tile's MFMAs
                    __builtin_amdgcn_sched_barrier(0);
                    wait_vmcnt<kLB + (kAStages - 2) * (kLA + kLB)>();
                    __syncthreads(); // A's K-tile t + 1 and B's t + 2 are in LDS for everybody, and nobody reads A's t and B's t + 1 any more
                    issue_a(t + kAStages);
                    issue_b(t + kBStages + 1);
                    if constexpr (kNI > 0) read_a(nxt, t + 1, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (kNI > 0) {
                    // the six products, small ones first
                    constexpr int kPa[6] = {2, 0, 1, 1, 0, 0}, kPb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
                    for (int q = 0; q < 6; q++)
#pragma unroll
                        for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[cur][kPa[q]], bs[kBCur][j][kPb[q]], acc[i][j], 0, 0, 0);
                    if (i + 1 < kA) { // LDS reads first, then B's decomposition (about 36 vector instructions) between the MFMAs
                        if (i < 2) __builtin_amdgcn_sched_group_barrier(0x100, 5, 0);
                        else __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
                        for (int r = 0; r < 12; r++) {
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                        }
                    }
                }
            }
        };
        for (int t = 0; t < n_kt; t += 2) {
            k_tile(t, std::integral_constant<int, 0>{});
            if (t + 1 < n_kt) k_tile(t + 1, std::integral_constant<int, 1>{});
        }
        wait_vmcnt<0>(); // drain the clamped tail loads before LDS is reused
        __syncthreads();

        // ---- the K-groups' sums: K-group g keeps column tile g and receives the other group's
        float *xbuf = reinterpret_cast<float *>(lds_raw) + lane;
        if constexpr (kNI > 0) {
            float *mine = xbuf + wave * (kN0 * 1024);
#pragma unroll
            for (int i = 0; i < kNI; i++)
#pragma unroll
                for (int v = 0; v < 16; v++) mine[(i * 16 + v) * 64] = kg ? acc[i][0][v] : acc[i][1][v];
        }
        __syncthreads();
        if constexpr (kNI > 0) {
            const int partner = (kg ^ 1) * 4 + ((wm ^ kg ^ 1) << 1) + wn;
            const float *theirs = xbuf + partner * (kN0 * 1024);
            const int c = bn0 + wn * 64 + kg * 32 + frow;
            float *out = p.c + (size_t)blockIdx.z * p.stride_c;
#pragma unroll
            for (int i = 0; i < kNI; i++) {
                float16_t o;
                [[maybe_unused]] float16_t prev;
                const int r0 = bm0 + (tile0 + i) * 32 + half * 4;
                bool bad = false;
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    o[v] = ((kg ? acc[i][1][v] : acc[i][0][v]) + theirs[(i * 16 + v) * 64]) * kS3Unscale;
                    bad |= !__builtin_isfinite(o[v]);
                    const int r = r0 + (v >> 2) * 8 + (v & 3);
                    prev[v] = p.accumulate && r < p.m && c < p.n ? out[(size_t)r * p.ldc + c] : 0.0f;
                }
                if (__any(bad)) { // (the whole wavefront: the matrix instruction needs every lane)
                    const float *ar = p.a + (size_t)min(bm0 + (tile0 + i) * 32 + frow, p.m - 1) * p.lda + kt0 * kS3K + half * 16;
                    const float *br = p.b + (size_t)min(c, p.n - 1) * p.ldb + kt0 * kS3K + half * 16;
                    float16_t s;
#pragma unroll
                    for (int v = 0; v < 16; v++) s[v] = 0.0f;
#pragma unroll 1
                    for (int t = 0; t < n_kt; t++, ar += kS3K, br += kS3K) { // lane half h takes k values 16 h .. 16 h + 15 of a K-tile
                        float4_t u[4], w[4];
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            u[q] = reinterpret_cast<const float4_t *>(ar)[q];
                            w[q] = reinterpret_cast<const float4_t *>(br)[q];
                        }
#pragma unroll
                        for (int q = 0; q < 4; q++)
#pragma unroll
                            for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(u[q][e], w[q][e], s, 0, 0, 0);
                    }
#pragma unroll
                    for (int v = 0; v < 16; v++) o[v] = __builtin_isfinite(o[v]) ? o[v] : s[v];
                }
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int r = r0 + (v >> 2) * 8 + (v & 3);
                    if (r < p.m && c < p.n) out[(size_t)r * p.ldc + c] = p.accumulate ? prev[v] + o[v] : o[v];
                }
            }
        }
    };
    if (wm == 0) run(std::integral_constant<int, kN0>{}, 0);
    else run(std::integral_constant<int, kN1>{}, kN0);
}

template <int kT>
static hipError_t launch_split3(const Split3Params &p, hipStream_t s) {
    constexpr size_t lds = (size_t)s3_a_stages(kT) * s3_a_stage(kT) + (size_t)s3_b_stages(kT) * kS3BStage;
    static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(gemm_split3_kernel<kT>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (attr != hipSuccess) return attr;
    const dim3 grid((p.n + kS3Cols - 1) / kS3Cols, p.m_pad / (32 * kT), p.split_k);
    hipLaunchKernelGGL(gemm_split3_kernel<kT>, grid, dim3(64 * kS3Waves), lds, s, p);
    return hipGetLastError();
}

bool gemm_split3_supported(const GemmParams &p, int epilogue) {
    if (p.tune.split3_plus1 == 1 || !p.f32_operands || epilogue != kGemmEpiF32 || p.batch != 1 || p.k_seg != 0 || p.causal != 0 || p.split_k > 1) return false;
    if (p.m < 1 || p.n < 1 || p.k < kS3K || p.k % kS3K != 0 || p.lda % 4 != 0 || p.ldb % 4 != 0) return false;
    if ((reinterpret_cast<uintptr_t>(p.a) | reinterpret_cast<uintptr_t>(p.b)) % 16 != 0) return false;
    if (p.workspace == nullptr || reinterpret_cast<uintptr_t>(p.workspace) % 16 != 0) return false;
    if ((size_t)kS3Cols * p.ldb * 4 >= ((size_t)1 << 31)) return false; // 32-bit byte offsets within a column tile
    if (p.tune.split3_plus1 == 2) return plan_split3(p.m, p.n, p.k, p.ldc, p.workspace_bytes, p.compute_units).rows > 0; // the first pass, and with it every one
    if (p.tune.tile_plus1 != 0 || p.tune.split_k != 0) return false; // those name tiles and pieces of the fp32 instruction's kernel
    // Short rows, and columns whose tiles and pieces on the fp32 instruction make whole rounds, are faster there: one or two launches
    // instead of two or three, and no decomposition.  No single size separates the two, so their times are estimated and compared: over
    // 2688 sizes that loses more than 4 % against the better kernel at 28 (at most 12 %).  us, fp32 instruction against this: 704 x 256
    // weights, 2 / 128 / 512 rows 10 / 17 / 26 against 13 / 22 / 34; 1408 x 1408, 24 / 128 / 512 rows 17 / 24 / 55 against 20 / 28 / 41;
    // 64 x 2048, 1024 rows 30 against 39; 3072 x 1024, 2 / 200 rows 20 / 49 against 18 / 37.
    const double us = split3_us(p.m, p.n, p.k, p.ldc, p.workspace_bytes, p.compute_units);
    return us >= 0.0 && us < gemm_f32_instruction_us(p);
}

hipError_t launch_gemm_split3(const GemmParams &p, hipStream_t s) {
    for (int r0 = 0; r0 < p.m;) {
        GemmParams part = p;
        part.m = p.m - r0;
        part.a = reinterpret_cast<const half_t *>(reinterpret_cast<const float *>(p.a) + (size_t)r0 * p.lda);
        part.c = reinterpret_cast<float *>(p.c) + (size_t)r0 * p.ldc;
        const Split3Plan plan = plan_split3(part.m, p.n, p.k, p.ldc, p.workspace_bytes, p.compute_units);
        if (plan.rows <= 0) return hipErrorInvalidValue;
        part.m = plan.rows;
        unsigned char *planes = reinterpret_cast<unsigned char *>(p.workspace);
        float *partial = reinterpret_cast<float *>(planes + plan.planes_bytes);
        const size_t threads = (size_t)(p.k / kS3K) * plan.m_pad * 4;
        hipLaunchKernelGGL(split3_rows_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, reinterpret_cast<const float *>(part.a), planes,
                           part.m, plan.m_pad, p.k, p.lda);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        Split3Params q{};
        q.a = reinterpret_cast<const float *>(part.a);
        q.b = reinterpret_cast<const float *>(p.b);
        q.planes = planes;
        q.m = part.m;
        q.n = p.n;
        q.k = p.k;
        q.lda = p.lda;
        q.ldb = p.ldb;
        q.m_pad = plan.m_pad;
        q.split_k = plan.pieces;
        q.c = plan.pieces > 1 ? partial : reinterpret_cast<float *>(part.c);
        q.ldc = plan.pieces > 1 ? p.n : p.ldc;
        q.stride_c = plan.pieces > 1 ? (size_t)part.m * p.n : 0;
        q.accumulate = plan.pieces > 1 ? 0 : p.accumulate;
        switch (plan.tiles) {
        case 1: e = launch_split3<1>(q, s); break;
        case 2: e = launch_split3<2>(q, s); break;
        case 3: e = launch_split3<3>(q, s); break;
        case 4: e = launch_split3<4>(q, s); break;
        case 5: e = launch_split3<5>(q, s); break;
        case 6: e = launch_split3<6>(q, s); break;
        case 7: e = launch_split3<7>(q, s); break;
        case 8: e = launch_split3<8>(q, s); break;
        default: return hipErrorInvalidValue;
        }
        if (e == hipSuccess && plan.pieces > 1) e = launch_gemm_split_finish_f32(part, partial, plan.pieces, s);
        if (e != hipSuccess) return e;
        r0 += plan.rows;
    }
    return hipSuccess;
}

} // namespace rlh
