// f32 products of few rows or columns, or of odd sizes, on the f32 matrix instruction: a small batch against a layer's weights, the
// weight gradients of a narrow layer, in all three layouts (A and B row-major, B packed n×k, A stored k×m) and at any alignment.
// The 64×64 tiles that ran them left most of the chip idle and walked k one 16-wide tile after another at 0.3 to 0.75 µs each, with
// a second launch where k was sliced, or a first where a packed B was unpacked.
//
// As in gemm_bf16_small.hip a workgroup takes 32×16 or 32×32 of C and its eight wavefronts split k, each with a two-stage ring of
// its own in LDS filled by direct loads: no barrier in the loop, up to 512 of k requested at once, one launch, the wavefronts' sums
// added in wavefront order.  Rows off 16-byte boundaries are requested value by value (four times the requests, a fifth to a third
// more time); values past the end of k read as zero in the operand whose rows run along k, so that nothing foreign is multiplied.
//
// What bounds it is latency: a launch, one trip to memory, 0.1 to 0.2 µs a 32-wide k-tile.  Before -> here (µs): 64×512×784
// 6.9 -> 5.5, packed 64×384×1152 11.6 -> 6.1, transposed 108×216×256 9.0 -> 3.3, 504×252×1311 18.9 -> 7.7; odd sizes 16×690×230
// 12.2 -> 4.0, packed 16×2487×829 50 -> 7.1, transposed 171×342×704 22.6 -> 5.7.  Over 119 products of the range it takes, 0.55
// of the time before.  64×64 tiles of this form are slower than either everywhere.
#include <algorithm>

#include "device_math.h"
#include "kernels.h"

namespace sthip {

namespace {

typedef __attribute__((address_space(3))) void *lds_void_ptr;

#define ST_SMALL32_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt((((n) < 63 ? (n) : 63) & 15) | (7 << 4) | (15 << 8) | (((((n) < 63 ? (n) : 63) >> 4) & 3) << 14))

constexpr unsigned kOutside = 0x80000000u;  // past the end of either operand: such loads give zeros
constexpr int kSmallStages = 2, kSmallK = 32;

struct SmallF32Args {
    const float *A, *B;
    float *C;
    const float *bias, *residual;
    int M, N, K, tiles_m;
    int ring_bytes;  // LDS of a wavefront: its one or two stages, later its sums
    float scale;
    int activation;
    int vector_stores;  // rows of C and of the residual start on 16-byte boundaries, and so does the bias
};

// One operand of a tile: ROWS rows (of A, or columns of B) by the 32 values of k of a stage, which a wavefront requests for
// itself.  K_MAJOR: memory holds k rows of `count` values (a row-major B, a transposed A), otherwise `count` rows of k values.
// VEC: 16 bytes a lane (rows on 16-byte boundaries), otherwise single values, and the image of a request in LDS is followed by
// padding that spreads a fragment's rows over the banks; under VEC the chunks of a row are permuted instead.
template <int ROWS, bool K_MAJOR, bool VEC>
struct SmallOperand {
    static constexpr int LOADS = VEC ? ROWS / 8 : ROWS / 2;
    static constexpr int PAD = VEC ? 0 : !K_MAJOR ? 16 : ROWS == 16 ? 64 : ROWS == 32 ? 32 : 16;
    static constexpr int BYTES = LOADS * ((VEC ? 1024 : 256) + PAD);
    static constexpr int OFFSETS = VEC ? LOADS : 1;

    __amdgpu_buffer_rsrc_t rsrc;
    unsigned offset[OFFSETS];
    int first_k[OFFSETS];  // of the lane's values, within a stage
    unsigned stage_step, load_step;
    int lane;

    static __device__ __forceinline__ int chunk_of(int row) { return K_MAJOR ? (ROWS >= 32 ? ((row >> 2) & 1) * 4 : 0) : (row ^ (row >> 3)) & 7; }

    __device__ __forceinline__ SmallOperand(const float *data, int count, int k, int row0, int stage0, int lane_) : lane(lane_)
    {
        const unsigned ld = static_cast<unsigned>(K_MAJOR ? count : k);
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(data), 0, static_cast<int>(static_cast<unsigned>(count) * static_cast<unsigned>(k) * 4u), 0x00020000);
        stage_step = K_MAJOR ? ld * (kSmallK * 4u) : kSmallK * 4u;
        load_step = VEC ? 0u : ld * 4u * (K_MAJOR ? 64 / ROWS : 2);
#pragma unroll
        for (int i = 0; i < OFFSETS; ++i) {
            if constexpr (K_MAJOR) {
                const int value = (i * 64 + lane) * (VEC ? 4 : 1), kl = value / ROWS, row = value % ROWS;
                first_k[i] = kl;
                offset[i] = ((static_cast<unsigned>(stage0) * kSmallK + kl) * ld + row0 + (VEC ? (row / 4 ^ chunk_of(kl)) * 4 : row)) * 4u;
            } else {
                const int row = VEC ? i * 8 + (lane >> 3) : lane >> 5;
                first_k[i] = VEC ? ((lane & 7) ^ chunk_of(row)) * 4 : lane & 31;
                offset[i] = (static_cast<unsigned>(row0 + row) * ld + static_cast<unsigned>(stage0) * kSmallK + first_k[i]) * 4u;
            }
        }
    }
    // Request i of stage t (of this wavefront's), of which `left` values of k exist: the rest reads as zero.  (A k-major
    // operand's rows past the last lie past its end.)
    __device__ __forceinline__ void load(unsigned char *base, int i, int t, int left) const
    {
        const int o = VEC ? i : 0;
        const unsigned v = K_MAJOR || first_k[o] < left ? offset[o] : kOutside;
        const unsigned s = static_cast<unsigned>(t) * stage_step + i * load_step;
        if constexpr (VEC) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_ptr)(base + i * 1024), 16, v, s, 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_ptr)(base + i * (256 + PAD)), 4, v, s, 0, 0);
    }
    // k-values 4·chunk .. + 3 of row `row`
    __device__ __forceinline__ f32x4 fragment(const unsigned char *base, int row, int chunk) const
    {
        if constexpr (!K_MAJOR) {
            if constexpr (VEC) return *reinterpret_cast<const f32x4 *>(base + row * 128 + ((chunk ^ chunk_of(row)) << 4));
            else return *reinterpret_cast<const f32x4 *>(base + (row >> 1) * (256 + PAD) + (row & 1) * 128 + chunk * 16);
        } else {
            f32x4 v;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int kl = chunk * 4 + t;
                if constexpr (VEC) {
                    v[t] = *reinterpret_cast<const float *>(base + kl * (ROWS * 4) + ((row >> 2) ^ chunk_of(kl)) * 16 + (row & 3) * 4);
                } else {
                    const int value = kl * ROWS + row;
                    v[t] = *reinterpret_cast<const float *>(base + (value >> 6) * (256 + PAD) + (value & 63) * 4);
                }
            }
            return v;
        }
    }
};

// C(16·MT × 16·NT) by one workgroup, k split over its wavefronts.
template <int MT, int NT, int WAVES, bool A_K_MAJOR, bool B_K_MAJOR, bool VEC>
__device__ __forceinline__ void gemm_f32_small_body(const SmallF32Args &p)
{
    using OperandA = SmallOperand<16 * MT, A_K_MAJOR, VEC>;
    using OperandB = SmallOperand<16 * NT, B_K_MAJOR, VEC>;
    constexpr int BM = 16 * MT, BN = 16 * NT, LOADS = OperandA::LOADS + OperandB::LOADS;
    constexpr int STAGE = OperandA::BYTES + OperandB::BYTES, C_STRIDE = BN + 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_bytes[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lj = lane & 15, lg = lane >> 4;
    const int M = p.M, N = p.N, K = p.K;
    const int tile_n = static_cast<int>(blockIdx.x) / p.tiles_m, tile_m = static_cast<int>(blockIdx.x) - tile_n * p.tiles_m;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int k_tiles = (K + kSmallK - 1) / kSmallK, per_wave = (k_tiles + WAVES - 1) / WAVES;
    const int first = wave * per_wave, count = max(0, min(k_tiles, first + per_wave) - first);
    const int ring_bytes = p.ring_bytes;
    unsigned char *const ring = lds_bytes + wave * ring_bytes;
    const OperandA a(p.A, M, K, m0, first, lane);
    const OperandB b(p.B, N, K, n0, first, lane);
    auto load_stage = [&](int t) {
        unsigned char *const base = ring + (t & (kSmallStages - 1)) * STAGE;
        const int left = K - (first + t) * kSmallK;
#pragma unroll
        for (int i = 0; i < OperandB::LOADS; ++i) b.load(base, i, t, left);
#pragma unroll
        for (int i = 0; i < OperandA::LOADS; ++i) a.load(base + OperandB::BYTES, i, t, left);
    };
    if (count > 0) load_stage(0);
    if (count > 1) load_stage(1);

    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t < count; ++t) {
        if (t + 1 < count) ST_SMALL32_WAIT_VMCNT(LOADS);
        else ST_SMALL32_WAIT_VMCNT(0);
        asm volatile("" ::: "memory");
        const unsigned char *const stage = ring + (t & (kSmallStages - 1)) * STAGE;
        f32x4 fa[2][MT], fb[2][NT];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) fb[s][nt] = b.fragment(stage, nt * 16 + lj, s * 4 + lg);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) fa[s][mt] = a.fragment(stage + OperandB::BYTES, mt * 16 + lj, s * 4 + lg);
        }
        // The fragments are in registers before the stage is filled again.
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        asm volatile("" ::: "memory");
        if (t + 2 < count) load_stage(t + 2);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[s][nt][e], fa[s][mt][e], acc[mt][nt], 0, 0, 0);
    }

    // Register i of lane (lj, lg) is C[16·mt + lj][16·nt + 4·lg + i] of the wavefront's share of the sum.
    float *const mine = reinterpret_cast<float *>(ring);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            *reinterpret_cast<f32x4 *>(&mine[(mt * 16 + lj) * C_STRIDE + nt * 16 + lg * 4]) = acc[mt][nt];
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
            if (p.vector_stores) {
                if (p.bias) {
                    const float4 add = *reinterpret_cast<const float4 *>(p.bias + col);
                    value[0] += add.x; value[1] += add.y; value[2] += add.z; value[3] += add.w;
                }
                if constexpr (decltype(has_residual)::value) {
                    const float4 r = *reinterpret_cast<const float4 *>(p.residual + idx);
                    value[0] += r.x; value[1] += r.y; value[2] += r.z; value[3] += r.w;
                }
                *reinterpret_cast<float4 *>(p.C + idx) = make_float4(act(value[0]), act(value[1]), act(value[2]), act(value[3]));
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (col + i >= N) continue;
                    if (p.bias) value[i] += p.bias[col + i];
                    if constexpr (decltype(has_residual)::value) value[i] += p.residual[idx + i];
                    p.C[idx + i] = act(value[i]);
                }
            }
        }
    });
}

#define ST_SMALL_F32_KERNELS(NAME, MT, NT, WAVES)                                                                                              \
    __global__ __launch_bounds__(WAVES * 64) void gemm_f32_small_##NAME##_nn_kernel(SmallF32Args p) { gemm_f32_small_body<MT, NT, WAVES, false, true, true>(p); }      \
    __global__ __launch_bounds__(WAVES * 64) void gemm_f32_small_##NAME##_nt_kernel(SmallF32Args p) { gemm_f32_small_body<MT, NT, WAVES, false, false, true>(p); }     \
    __global__ __launch_bounds__(WAVES * 64) void gemm_f32_small_##NAME##_tn_kernel(SmallF32Args p) { gemm_f32_small_body<MT, NT, WAVES, true, true, true>(p); }       \
    __global__ __launch_bounds__(WAVES * 64) void gemm_f32_small_##NAME##_nn_any_kernel(SmallF32Args p) { gemm_f32_small_body<MT, NT, WAVES, false, true, false>(p); } \
    __global__ __launch_bounds__(WAVES * 64) void gemm_f32_small_##NAME##_nt_any_kernel(SmallF32Args p) { gemm_f32_small_body<MT, NT, WAVES, false, false, false>(p); }\
    __global__ __launch_bounds__(WAVES * 64) void gemm_f32_small_##NAME##_tn_any_kernel(SmallF32Args p) { gemm_f32_small_body<MT, NT, WAVES, true, true, false>(p); }
ST_SMALL_F32_KERNELS(32x16, 2, 1, 8)
ST_SMALL_F32_KERNELS(32x32, 2, 2, 8)
#undef ST_SMALL_F32_KERNELS

// Estimated time (µs): a tile alone, and what each further round of 256 adds, constant and per 32 of k; fitted to 150 products of
// 8 to 4096 rows and columns, 12 to 3840 terms (90 % within a fifth).
struct SmallF32Times {
    double alone, alone_k, round, round_k;
};
struct SmallF32Config {
    int bm, bn, waves;
    void (*kernels[2][3])(SmallF32Args);  // [any alignment][A and B row-major, B packed, A transposed]
    SmallF32Times times[2][3];

    size_t tiles(size_t m, size_t n) const { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); }
    double us(size_t m, size_t n, size_t k, int layout, bool any) const
    {
        const SmallF32Times &t = times[any ? 1 : 0][layout];
        const double k_tiles = static_cast<double>((k + kSmallK - 1) / kSmallK), rounds = static_cast<double>(tiles(m, n)) / 256;
        return t.alone + t.alone_k * k_tiles + std::max(rounds - 0.5, 0.0) * (t.round + t.round_k * k_tiles);
    }
    // A wavefront's stages (one is enough where it has one k-tile) with the padding of any layout, and its sums in the same place.
    size_t ring_bytes(size_t k, bool any) const
    {
        const size_t stages = ((k + kSmallK - 1) / kSmallK + waves - 1) / waves > 1 ? kSmallStages : 1;
        const size_t stage = any ? static_cast<size_t>(bm + bn) / 2 * (256 + 32) + 1024 : static_cast<size_t>(bm + bn) * 128;
        return std::max(stages * stage, static_cast<size_t>(bm) * (bn + 4) * sizeof(float));
    }
};
#define ST_SMALL_F32_FAMILY(NAME)                                                                                                \
    {{gemm_f32_small_##NAME##_nn_kernel, gemm_f32_small_##NAME##_nt_kernel, gemm_f32_small_##NAME##_tn_kernel},                  \
     {gemm_f32_small_##NAME##_nn_any_kernel, gemm_f32_small_##NAME##_nt_any_kernel, gemm_f32_small_##NAME##_tn_any_kernel}}
const SmallF32Config kSmallF32Configs[] = {
    {32, 16, 8, ST_SMALL_F32_FAMILY(32x16),
     {{{2.73, 0.092, 0.14, 0.174}, {2.55, 0.096, 1.68, 0.098}, {2.65, 0.080, 0.32, 0.157}},
      {{3.01, 0.135, 0.05, 0.206}, {2.94, 0.127, 0.03, 0.236}, {2.62, 0.133, 0.58, 0.161}}}},
    {32, 32, 8, ST_SMALL_F32_FAMILY(32x32),
     {{{2.80, 0.157, 0.45, 0.253}, {2.74, 0.155, 2.98, 0.121}, {2.81, 0.143, 0.73, 0.206}},
      {{3.22, 0.207, 0.20, 0.294}, {3.13, 0.206, 0.00, 0.335}, {3.04, 0.181, 0.68, 0.247}}}},
};
#undef ST_SMALL_F32_FAMILY

const SmallF32Config &choose_small(size_t m, size_t n, size_t k, int layout, bool any)
{
    const SmallF32Config &narrow = kSmallF32Configs[0], &wide = kSmallF32Configs[1];
    return narrow.us(m, n, k, layout, any) <= wide.us(m, n, k, layout, any) ? narrow : wide;
}

bool aligned16(const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

// Whether the operands' rows in memory are not all on 16-byte boundaries.
bool any_alignment(size_t m, size_t n, size_t k, int layout, const float *lhs, const float *rhs)
{
    return !aligned16(lhs) || !aligned16(rhs) || (layout == 2 ? m : k) % 4 != 0 || (layout == 1 ? k : n) % 4 != 0;
}

}  // namespace

bool gemm_f32_small_applies(size_t m, size_t n, size_t k, bool lhs_transposed, bool rhs_packed, const float *lhs, const float *rhs, double other_us)
{
    // 32-bit byte offsets up to a tile past the operands' ends
    if (m == 0 || n == 0 || k == 0 || k > 65536 || (m + 64) * (k + 64) * 4 >= (1ull << 31) || (n + 64) * (k + 64) * 4 >= (1ull << 31)) return false;
    const int layout = lhs_transposed ? 2 : rhs_packed ? 1 : 0;
    const bool any = any_alignment(m, n, k, layout, lhs, rhs);
    const SmallF32Config &c = choose_small(m, n, k, layout, any);
    // Beyond two rounds, and as A·Bᵀ beyond one, the estimates of both sides are a fifth off and the gain is small where there is one:
    // as A·Bᵀ 635×832×2496 took 43.7 µs against 34.7, 468×640×1920 25.6 against 23.0.
    // The A stored k×m is read in rows of 128 bytes whatever the tile: 208×3584×384 in 784 tiles 17.2 µs against 11.8.
    // Beyond 1024 tiles of one or two k-tiles each, where a tile is little but its turn on a unit and its stores, the estimate is up to half
    // too low: as A·Bᵀ 3520×513×13 11.4 µs against 8.5, 2493×1002×27 13.6 against 10.5; 192×3129×29 7.0 against 5.4.
    const size_t tiles = c.tiles(m, n);
    const double margin = tiles > 1024 && k <= 64 ? 0.6 : tiles > (layout == 1 ? 256 : 512) ? (layout == 2 && !any ? 0.7 : 0.75) : 0.95;
    return c.us(m, n, k, layout, any) < margin * other_us;
}

hipError_t launch_gemm_f32_small(size_t m, size_t n, size_t k, bool lhs_transposed, const float *lhs, bool rhs_packed, const float *rhs,
                                 float *out, const GemmEpilogue &epilogue, hipStream_t stream)
{
    const int layout = lhs_transposed ? 2 : rhs_packed ? 1 : 0;
    const bool any = any_alignment(m, n, k, layout, lhs, rhs);
    const SmallF32Config &config = choose_small(m, n, k, layout, any);
    SmallF32Args args;
    args.A = lhs;
    args.B = rhs;
    args.C = out;
    args.bias = epilogue.bias;
    args.residual = epilogue.residual;
    args.M = static_cast<int>(m);
    args.N = static_cast<int>(n);
    args.K = static_cast<int>(k);
    args.tiles_m = static_cast<int>((m + config.bm - 1) / config.bm);
    args.ring_bytes = static_cast<int>(config.ring_bytes(k, any));
    args.scale = epilogue.scale;
    args.activation = epilogue.activation;
    args.vector_stores = n % 4 == 0 && aligned16(out) && aligned16(epilogue.bias) && aligned16(epilogue.residual);
    const size_t lds = config.waves * config.ring_bytes(k, any), tiles = config.tiles(m, n);
    if (tiles > 0x7fffffffu || lds > 160 * 1024) return hipErrorInvalidConfiguration;
    auto kernel = config.kernels[any ? 1 : 0][layout];
    if (lds > 64 * 1024) {  // more than a launch may take unasked; the most any k needs, whatever other threads ask for meanwhile
        const hipError_t rc = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (rc != hipSuccess) return rc;
    }
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(tiles)), dim3(static_cast<unsigned>(config.waves) * 64), lds, stream, args);
    return hipGetLastError();
}

}  // namespace sthip
