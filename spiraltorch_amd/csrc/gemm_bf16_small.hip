// bf16 products of few rows (f32 sums, the fused epilogue of gemm_bf16.hip): a decoder's projections on one prompt, a mid-size
// batch against a narrow weight.  The 128- and 256-row tiles leave most of the chip without work there (117×2048×512 is 16
// tiles) and walk k in a chain of load latencies, or cut it over workgroups and need a second launch to add the pieces.
//
// Here a workgroup takes a small tile of C (32×16, 32×32 or 64×64) and its wavefronts split k: each streams its own range of A
// and B through a two-stage ring of its own in LDS with direct loads, so up to 1024 of k (512 for the 64×64 tile) is requested
// at once, there is no barrier in the loop, and one launch does.  The wavefronts' sums are added through LDS in wavefront order:
// results do not depend on scheduling, and are the same for both layouts of B.
//
// What bounds it is latency: a launch (2.0 µs for an empty kernel), one trip to memory, the sums' trip through LDS.  Of a
// launch among others, before -> here: 117×1536×512 10.4 -> 3.6 µs, 117×512×512 10.1 -> 3.1, 117×2048×512 10.0 -> 3.6,
// 117×512×2048 11.4 -> 4.5, 512×1536×512 8.3 -> 7.0, 1024×512×2048 14.4 -> 9.6, 256×1000×512 11.0 -> 4.3.  Larger launches are
// bound by LDS and L2 traffic (16 to 32 flops a byte) and belong to the large tiles.  Layer normalisation of the rows on their
// way in was tried: 3.2 µs more a launch, where the kernel of its own takes 2.4.
#include <algorithm>
#include <cmath>

#include "device_math.h"
#include "kernels.h"

namespace sthip {

namespace {

typedef float f32x4_acc __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void *lds_void_ptr;
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

#define ST_SMALL_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (7 << 4) | (15 << 8) | ((((n) >> 4) & 3) << 14))

struct SmallArgs {
    const uint16_t *A;
    const uint16_t *B;
    float *C32;
    uint16_t *C16;
    const float *bias, *residual;
    int M, N, K, tiles_m;
    int ring_bytes;  // LDS of a wavefront: its one or two stages, later its sums
    float scale;
    int activation;
};

// Where 16-byte chunk q of row r stands in a 128-byte LDS row: the sixteen rows of a fragment read spread over all banks.
__device__ __forceinline__ int small_swizzle(int row) { return (row ^ (row >> 3)) & 7; }

constexpr int kSmallStages = 2;

// C(16·MT × 16·NT) by one workgroup, k split over its wavefronts.
template <int MT, int NT, int WAVES, bool ROWMAJOR_B>
__device__ __forceinline__ void gemm_bf16_small_body(const SmallArgs &p)
{
    constexpr int BM = 16 * MT, BN = 16 * NT;
    constexpr int A_LOADS = 2 * MT, B_LOADS = 2 * NT, LOADS = A_LOADS + B_LOADS;  // requests of 1 KB a stage
    constexpr int STAGE = LOADS * 1024;
    constexpr int C_STRIDE = BN + 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_bytes[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lj = lane & 15, lg = lane >> 4;
    const int M = p.M, N = p.N, K = p.K;
    // Workgroup ids go round-robin over the 8 XCDs: each takes a contiguous run of tiles, down the rows of up to eight row tiles
    // first, so that the tiles that share columns of B or rows of A find them in its L2.  Before / after: 117×512×2048 4.7 / 4.3 µs,
    // 64×4096×4096 12.3 / 9.0, 6272×256×2304 25.6 / 20.7.  (Without the groups of eight, 4096×512×2048 went from 18.7 to 26.6.)
    const int grid = static_cast<int>(gridDim.x), xcd = static_cast<int>(blockIdx.x) & 7;
    int run = xcd * (grid >> 3) + min(xcd, grid & 7) + (static_cast<int>(blockIdx.x) >> 3), first_m = 0, rows = p.tiles_m;
    if (p.tiles_m > 8) {
        const int group_tiles = 8 * (grid / p.tiles_m), group = run / group_tiles;
        run -= group * group_tiles;
        first_m = group * 8;
        rows = min(p.tiles_m - first_m, 8);
    }
    const int tile_n = run / rows, tile_m = first_m + run - tile_n * rows;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int k_tiles = K / 64, per_wave = (k_tiles + WAVES - 1) / WAVES;
    const int first = wave * per_wave, count = max(0, min(k_tiles, first + per_wave) - first);
    const int ring_bytes = p.ring_bytes;
    unsigned char *const ring = lds_bytes + wave * ring_bytes;

    const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(p.B), 0, static_cast<int>(static_cast<unsigned>(N) * static_cast<unsigned>(K) * 2u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(p.A), 0, static_cast<int>(static_cast<unsigned>(M) * static_cast<unsigned>(K) * 2u), 0x00020000);
    unsigned a_off[A_LOADS], b_off[B_LOADS];
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
        const int row = i * 8 + (lane >> 3);
        a_off[i] = (static_cast<unsigned>(m0 + row) * K + static_cast<unsigned>(first) * 64 + ((lane & 7) ^ small_swizzle(row)) * 8) * 2u;
    }
#pragma unroll
    for (int i = 0; i < B_LOADS; ++i) {
        if constexpr (ROWMAJOR_B) {
            constexpr int LPR = 2 * NT;  // lanes a k-row of the stage takes
            const int row = i * (64 / LPR) + lane / LPR;
            const int chunk = (lane % LPR) ^ (NT == 4 ? ((row >> 1) & 3) * 2 : 0);
            b_off[i] = (static_cast<unsigned>(first * 64 + row) * N + n0 + chunk * 8) * 2u;
        } else {
            const int row = i * 8 + (lane >> 3);
            b_off[i] = (static_cast<unsigned>(n0 + row) * K + static_cast<unsigned>(first) * 64 + ((lane & 7) ^ small_swizzle(row)) * 8) * 2u;
        }
    }
    const unsigned b_step = ROWMAJOR_B ? static_cast<unsigned>(N) * 128u : 128u;
    auto load_stage = [&](int t) {
        unsigned char *const base = ring + (t & (kSmallStages - 1)) * STAGE;
        const unsigned tile = static_cast<unsigned>(t);
#pragma unroll
        for (int i = 0; i < B_LOADS; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_void_ptr)(base + i * 1024), 16, b_off[i], tile * b_step, 0, 0);
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_void_ptr)(base + (B_LOADS + i) * 1024), 16, a_off[i], tile * 128u, 0, 0);
    };

    if (count > 0) load_stage(0);
    if (count > 1) load_stage(1);

    f32x4_acc acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4_acc{0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t < count; ++t) {
        if (t + 1 < count) ST_SMALL_WAIT_VMCNT(LOADS);
        else ST_SMALL_WAIT_VMCNT(0);
        asm volatile("" ::: "memory");
        const unsigned char *const stage = ring + (t & (kSmallStages - 1)) * STAGE;
        [[maybe_unused]] const unsigned stage_address = static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_void_ptr)ring)) + (t & (kSmallStages - 1)) * STAGE;
        bf16x8 fa[2][MT], fb[2][NT];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int chunk = s * 4 + lg;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if constexpr (ROWMAJOR_B) {
                    // Lane 4i + j of a group of sixteen gives the address of four columns of k-row i, and receives column 4i + j.
                    const int row = s * 32 + lg * 8 + (lj >> 2);
                    const int piece = nt * 4 + (lj & 3);  // 8-byte piece of the k-row
                    auto at = [&](int r) {
                        const int q = (piece >> 1) ^ (NT == 4 ? ((r >> 1) & 3) * 2 : 0);
                        return stage_address + r * (32 * NT) + q * 16 + (piece & 1) * 8;
                    };
                    // (Reads and wait as one assembly block: before a transposing read of its own the compiler waits for all loads.)
                    u32x2_t lo, hi;
                    asm volatile("ds_read_b64_tr_b16 %0, %2\n"
                                 "ds_read_b64_tr_b16 %1, %3\n"
                                 "s_waitcnt lgkmcnt(0)"
                                 : "=&v"(lo), "=&v"(hi)
                                 : "v"(at(row)), "v"(at(row + 4))
                                 : "memory");
                    const u32x4_t both = {lo[0], lo[1], hi[0], hi[1]};
                    fb[s][nt] = __builtin_bit_cast(bf16x8, both);
                } else {
                    const int row = nt * 16 + lj;
                    fb[s][nt] = *reinterpret_cast<const bf16x8 *>(stage + row * 128 + ((chunk ^ small_swizzle(row)) << 4));
                }
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const int row = mt * 16 + lj;
                fa[s][mt] = *reinterpret_cast<const bf16x8 *>(stage + B_LOADS * 1024 + row * 128 + ((chunk ^ small_swizzle(row)) << 4));
            }
        }
        // The fragments are in registers before the stage is filled again.
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        asm volatile("" ::: "memory");
        if (t + 2 < count) load_stage(t + 2);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[s][nt], fa[s][mt], acc[mt][nt], 0, 0, 0);
    }

    // Register i of lane (lj, lg) is C[16·mt + lj][16·nt + 4·lg + i] of the wavefront's share of the sum.
    float *const mine = reinterpret_cast<float *>(ring);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            *reinterpret_cast<float4 *>(&mine[(mt * 16 + lj) * C_STRIDE + nt * 16 + lg * 4]) =
                make_float4(acc[mt][nt][0], acc[mt][nt][1], acc[mt][nt][2], acc[mt][nt][3]);
    __syncthreads();
    with_epilogue_ops(p.activation, p.residual != nullptr, [&](auto &&act, auto has_residual) {
#pragma unroll
        for (int e = tid; e < BM * BN / 4; e += WAVES * 64) {
            const int local_row = e / (BN / 4), local_col = e % (BN / 4) * 4;
            const int row = m0 + local_row, col = n0 + local_col;
            if (row >= M || col >= N) continue;
            const size_t idx = static_cast<size_t>(row) * N + col;
            float4 v = *reinterpret_cast<const float4 *>(lds_bytes + (local_row * C_STRIDE + local_col) * 4);
#pragma unroll
            for (int w = 1; w < WAVES; ++w) {
                const float4 q = *reinterpret_cast<const float4 *>(lds_bytes + w * ring_bytes + (local_row * C_STRIDE + local_col) * 4);
                v.x += q.x; v.y += q.y; v.z += q.z; v.w += q.w;
            }
            float value[4] = {v.x * p.scale, v.y * p.scale, v.z * p.scale, v.w * p.scale};
            if (col + 4 <= N) {  // (16-byte accesses at whatever boundary the rows have)
                if (p.bias) {
                    const f32x4_a4 b = *reinterpret_cast<const f32x4_a4 *>(p.bias + col);
#pragma unroll
                    for (int i = 0; i < 4; ++i) value[i] += b[i];
                }
                if constexpr (decltype(has_residual)::value) {
                    const f32x4_a4 r = *reinterpret_cast<const f32x4_a4 *>(p.residual + idx);
#pragma unroll
                    for (int i = 0; i < 4; ++i) value[i] += r[i];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) value[i] = act(value[i]);
                if (p.C32) *reinterpret_cast<f32x4_a4 *>(p.C32 + idx) = f32x4_a4{value[0], value[1], value[2], value[3]};
                if (p.C16) *reinterpret_cast<u32x2_a2 *>(p.C16 + idx) = u32x2_a2{pack_bf16x2_rne(value[0], value[1]), pack_bf16x2_rne(value[2], value[3])};
            } else {
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    if (col + i >= N) continue;
                    if (p.bias) value[i] += p.bias[col + i];
                    if constexpr (decltype(has_residual)::value) value[i] += p.residual[idx + i];
                    value[i] = act(value[i]);
                    if (p.C32) p.C32[idx + i] = value[i];
                    if (p.C16) p.C16[idx + i] = f32_to_bf16_rne(value[i]);
                }
            }
        }
    });
}

__global__ __launch_bounds__(512) void gemm_bf16_small_32x16_kernel(SmallArgs p) { gemm_bf16_small_body<2, 1, 8, false>(p); }
__global__ __launch_bounds__(512) void gemm_bf16_small_32x32_kernel(SmallArgs p) { gemm_bf16_small_body<2, 2, 8, false>(p); }
__global__ __launch_bounds__(256) void gemm_bf16_small_64x64_kernel(SmallArgs p) { gemm_bf16_small_body<4, 4, 4, false>(p); }
__global__ __launch_bounds__(512) void gemm_bf16_small_32x16_rm_kernel(SmallArgs p) { gemm_bf16_small_body<2, 1, 8, true>(p); }
__global__ __launch_bounds__(512) void gemm_bf16_small_32x32_rm_kernel(SmallArgs p) { gemm_bf16_small_body<2, 2, 8, true>(p); }
__global__ __launch_bounds__(256) void gemm_bf16_small_64x64_rm_kernel(SmallArgs p) { gemm_bf16_small_body<4, 4, 4, true>(p); }

// Estimated time (µs; of a pair the first is constant, the second per 64 of k): a launch alone, what 256 workgroups add, what having more
// than 256 adds, and each further round, a round being what the compute units hold at a time.  Fitted to some 200 products a tile of 33 to 4096 rows, 14 shapes of n and
// k from 256 to 4096, the small ones timed without the host between them, operands that the L2 does not hold from the launch before:
// within 15 % of each, 5 % in the rms.
struct SmallTimes {
    double alone, alone_k, units, units_k, second, round, round_k;
};
struct SmallConfig {
    void (*packed)(SmallArgs);
    void (*rowmajor)(SmallArgs);
    int bm, bn, waves;  // powers of two
    SmallTimes packed_us, rowmajor_us;

    size_t tiles(size_t m, size_t n) const { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); }
    // A wavefront's stages (one is enough where it has one k-tile), and its sums in the same place.
    size_t ring_bytes(size_t k) const
    {
        const size_t stages = k / 64 > static_cast<size_t>(waves) ? kSmallStages : 1;
        return std::max<size_t>(stages * (bm + bn) * 128, static_cast<size_t>(bm) * (bn + 4) * sizeof(float));
    }
};
const SmallConfig kSmallConfigs[] = {
    {gemm_bf16_small_32x16_kernel, gemm_bf16_small_32x16_rm_kernel, 32, 16, 8,
     {2.42, 0.051, 0.22, 0.034, 0.40, 1.03, 0.028}, {2.42, 0.094, 0.39, 0.025, 0.40, 0.77, 0.090}},
    {gemm_bf16_small_32x32_kernel, gemm_bf16_small_32x32_rm_kernel, 32, 32, 8,
     {2.44, 0.089, 0.57, 0.005, 0.00, 1.09, 0.069}, {2.44, 0.124, 0.47, 0.008, 0.00, 1.30, 0.097}},
    {gemm_bf16_small_64x64_kernel, gemm_bf16_small_64x64_rm_kernel, 64, 64, 4,
     {3.89, 0.174, 1.03, 0.000, 0.00, 2.33, 0.159}, {3.89, 0.227, 1.08, 0.000, 0.00, 3.62, 0.135}},
};

}  // namespace

// The same tile for both layouts of B, so that they give the same bits.  (Asked for every launch, of which a short decoder makes forty: no
// 64-bit divisions.)
GemmSmallChoice gemm_bf16_small_choice(size_t m, size_t n, size_t k)
{
    GemmSmallChoice best;
    // 32-bit byte offsets up to a tile past the operands' ends
    if (m == 0 || n == 0 || k < 64 || k % 64 != 0 || k > 65536 || (m + 64) * k * 2 >= (1ull << 31) || (n + 64) * k * 2 >= (1ull << 31)) return best;
    const double k_tiles = static_cast<double>(k / 64);
    double best_us = 0.0;
    for (int i = 0; i < 3; ++i) {
        const SmallConfig &c = kSmallConfigs[i];
        const unsigned bm = static_cast<unsigned>(c.bm), bn = static_cast<unsigned>(c.bn);
        const double units = static_cast<double>((static_cast<unsigned>(m) + bm - 1) >> __builtin_ctz(bm)) *
                             static_cast<double>((static_cast<unsigned>(n) + bn - 1) >> __builtin_ctz(bn)) / 256;
        const unsigned resident = std::min(160u * 1024 / (static_cast<unsigned>(c.ring_bytes(k)) * c.waves), 32u / c.waves);
        const double rounds = units > resident ? std::ceil(units / resident) - 1 : 0.0;
        auto us = [&](const SmallTimes &t) {
            return t.alone + t.alone_k * k_tiles + units * (t.units + t.units_k * k_tiles) + (units > 1.0 ? t.second : 0.0) + rounds * (t.round + t.round_k * k_tiles);
        };
        const double packed = us(c.packed_us), rowmajor = us(c.rowmajor_us);
        if (best.tile < 0 || packed + 0.3 * rowmajor < best_us) {
            best = GemmSmallChoice{i, packed, rowmajor};
            best_us = packed + 0.3 * rowmajor;
        }
    }
    return best;
}

hipError_t launch_gemm_bf16_small(int tile, size_t m, size_t n, size_t k, const uint16_t *lhs, const uint16_t *rhs, bool rhs_packed, float *out_f32,
                                  uint16_t *out_bf16, const GemmEpilogue &epilogue, hipStream_t stream)
{
    const SmallConfig &config = kSmallConfigs[tile];
    SmallArgs args;
    args.A = lhs;
    args.B = rhs;
    args.C32 = out_f32;
    args.C16 = out_bf16;
    args.bias = epilogue.bias;
    args.residual = epilogue.residual;
    args.M = static_cast<int>(m);
    args.N = static_cast<int>(n);
    args.K = static_cast<int>(k);
    args.tiles_m = static_cast<int>((m + config.bm - 1) / config.bm);
    args.scale = epilogue.scale;
    args.activation = epilogue.activation;
    args.ring_bytes = static_cast<int>(config.ring_bytes(k));
    const size_t lds = config.waves * config.ring_bytes(k), tiles = config.tiles(m, n);
    if (tiles > 0x7fffffffu || lds > 160 * 1024) return hipErrorInvalidConfiguration;
    auto kernel = rhs_packed ? config.packed : config.rowmajor;
    if (lds > 64 * 1024) {  // more than a launch may take unasked; the most any k needs, whatever other threads ask for meanwhile
        const hipError_t rc = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (rc != hipSuccess) return rc;
    }
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(tiles)), dim3(static_cast<unsigned>(config.waves) * 64), lds, stream, args);
    return hipGetLastError();
}

}  // namespace sthip
