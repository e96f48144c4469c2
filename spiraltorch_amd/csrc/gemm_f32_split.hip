// Large f32 products on the bf16 matrix cores: every f32 operand value is written as the sum of three bf16 values,
// x = hi + mid + lo (hi = bf16(x), mid = bf16(x - hi), lo = x - hi - mid, each difference exact: 3 × 8 mantissa bits hold
// all 24 of an f32), and a product a·b is accumulated in f32 from six of the nine piece products,
//     lo·hi, mid·hi, mid·mid, hi·mid, hi·lo, hi·hi.
// What is left out (mid·lo, lo·mid, lo·lo) is at most 2^-24 of |a·b|, as much as rounding one f32 product can cost, and 2^-27.4 in
// the rms over N(0,1) operands (|mid| <= 2^-8 |x|, |lo| <= 2^-17 |x|).
// v_mfma_f32_32x32x16_bf16 multiplies exactly and adds into f32 accumulators, and the result carries one rounding of the
// large sum per sixteen terms where the f32 instruction rounds after every term, so it is closer to the exact sum than the
// f32 matrix cores' (rms error against float64, N(0,1) operands, of the result's rms: k = 768 1.6e-7 against 5.0e-7,
// k = 3072 1.6e-7 to 2.3e-7 against 5.0e-7 to 7.0e-7, k = 4096 4.0e-7 against 1.1e-6).
//
// Six bf16 products take 6/16 of the f32 instruction's time at their nominal rates.  What bounds the product kernel is the
// power the matrix cores draw on random operands: a 32×32×16 instruction takes 21 ns of a SIMD here, 19 in a loop of
// nothing else, 13 on zeros; then come the splitting pass (memory: 4 bytes read and 6 written a value, ~6 TB/s), and 11 µs
// of launches, first loads and stores.  Measured with the pass, f32 matrix cores -> here: 4096³ 1014 -> 615 µs
// (223 TFLOP/s), 1576×3072×768 70 -> 48, A stored k×m 3072×768×1576 100 -> 62, B prepacked 2384×1120×3708 243 -> 133,
// and where rows are unaligned or k is no multiple of 16 853×1399×1747 114 -> 43, 182×425×2895 161 -> 20 µs.
//
// Both operands are scaled by a power of two first, so that the pieces are exact down to the smallest f32 value.  Values too
// large for that or not finite, and pairs of magnitudes whose scaled sums could overflow (about 1e10 against 1e10), are
// found by the splitting pass; the tiles they touch are summed on the f32 matrix cores from the original operands.
#include <algorithm>
#include <type_traits>

#include "device_math.h"
#include "kernels.h"
#include "split_product.h"

namespace sthip {

namespace {

typedef __attribute__((address_space(3))) void *lds_void_ptr;
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// ---- the splitting pass ------------------------------------------------------------------------------------------
// An operand of `rows` rows along a reduction of `k` terms becomes blocks of 32 rows × 16 terms.  A block is three
// fragments (hi, mid, lo) of 1 KB, each in the order the matrix instruction wants its operand: lane l holds row l % 32,
// terms 8·(l / 32) .. + 7.  Block (rb, ks) starts at (rb·ksteps + ks)·3 KB; rows and terms past the end are zeros, so the
// product kernel needs no edge cases, and any m, n, k and alignment of the operands is served alike.
//
// Beside every pair of blocks along k, a status word: the largest magnitude in it (split_top).
struct SplitJob {
    const float *src;
    unsigned char *blocks;
    unsigned *status;
    int rows, k, ld;
    int transposed;  // 0: src[row·ld + term], 1: src[term·ld + row]
    int ksteps;  // ceil(k / 16), rounded up to even
    unsigned groups_k;  // workgroups along k: 128 terms each (32 when transposed)
};

__device__ __forceinline__ float4 load4_guarded(const float *row, int first, int limit)
{
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (first + 4 <= limit) {
        const f32x4_a4 w = *reinterpret_cast<const f32x4_a4 *>(row + first);
        v = make_float4(w[0], w[1], w[2], w[3]);
    } else {
        if (first + 0 < limit) v.x = row[first + 0];
        if (first + 1 < limit) v.y = row[first + 1];
        if (first + 2 < limit) v.z = row[first + 2];
    }
    return v;
}

// A workgroup splits 32 rows × 128 terms (128 rows × 32 terms when the source runs along the rows): 512-byte pieces of the
// source go through LDS, a wavefront then owns two neighbouring blocks and writes their 6 KB contiguously.
__global__ __launch_bounds__(256) void split_operands_kernel(SplitJob first, SplitJob second, unsigned first_groups)
{
    constexpr int STRIDE = 132;
    __shared__ __attribute__((aligned(16))) float tile[32 * STRIDE];
    const bool is_first = blockIdx.x < first_groups;
    const SplitJob &job = is_first ? first : second;
    const unsigned group = blockIdx.x - (is_first ? 0u : first_groups);
    const int gk = static_cast<int>(group % job.groups_k), gr = static_cast<int>(group / job.groups_k);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 31, lh = lane >> 5;
    const int r0 = gr * (job.transposed ? 128 : 32), k0 = gk * (job.transposed ? 32 : 128);
    {
        const int line0 = job.transposed ? k0 : r0, lines = job.transposed ? job.k : job.rows;
        const int along0 = (job.transposed ? r0 : k0) + (tid & 31) * 4, along = job.transposed ? job.rows : job.k;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int line = i * 8 + (tid >> 5);
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (line0 + line < lines) v = load4_guarded(job.src + static_cast<size_t>(line0 + line) * job.ld, along0, along);
            *reinterpret_cast<float4 *>(&tile[line * STRIDE + (tid & 31) * 4]) = v;
        }
    }
    __syncthreads();
    const int rb = job.transposed ? gr * 4 + wave : gr;
    const int pair = job.transposed ? gk : gk * 4 + wave;
    if (rb * 32 >= job.rows || pair * 2 >= job.ksteps) return;
    unsigned top = 0;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        const int ks = pair * 2 + half;
        float x[8];
        if (job.transposed) {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = tile[(half * 16 + lh * 8 + e) * STRIDE + wave * 32 + li];
        } else {
            const float *src = &tile[li * STRIDE + (wave * 2 + half) * 16 + lh * 8];
            const float4 v0 = *reinterpret_cast<const float4 *>(src), v1 = *reinterpret_cast<const float4 *>(src + 4);
            x[0] = v0.x; x[1] = v0.y; x[2] = v0.z; x[3] = v0.w; x[4] = v1.x; x[5] = v1.y; x[6] = v1.z; x[7] = v1.w;
        }
        uint32_t piece[3][4];
        split_pieces(x, piece);
        top = split_top(x, top);
        unsigned char *dst = job.blocks + (static_cast<size_t>(rb) * job.ksteps + ks) * 3072 + lane * 16;
#pragma unroll
        for (int plane = 0; plane < 3; ++plane)
            *reinterpret_cast<uint4 *>(dst + plane * 1024) = make_uint4(piece[plane][0], piece[plane][1], piece[plane][2], piece[plane][3]);
    }
    top = wave_top(top);
    if (lane == 0) job.status[static_cast<size_t>(rb) * (job.ksteps / 2) + pair] = top;
}

// ---- the product -------------------------------------------------------------------------------------------------
// Where the row block `block` of a tile that starts at row `first` lies for reduction step `step`, in bytes from the start
// of its operand's blocks.  Tiles reach past the last row block; they read the last one again (what that gives is not
// stored).  These offsets go into a load's scalar offset, which its bounds check does not see: every one of them has to lie
// inside the buffer.
__host__ __device__ inline unsigned split_block_offset(int first, int block, int rows, int ksteps, int step)
{
    const int row_block = first / 32 + block, last = (rows - 1) / 32;
    return static_cast<unsigned>((row_block < last ? row_block : last) * ksteps + step) * 3072u;
}

struct SplitGemmArgs {
    const unsigned char *blocks;  // A's blocks, then B's at b_base
    unsigned b_base, bytes;
    const unsigned *status_a, *status_b;
    float *C;  // the result, or plane `split` of the partial sums
    const float *bias, *residual;
    const float *A, *B;  // the original operands, for the tiles the splitting pass marked
    int a_row, a_k, b_col, b_k;  // their strides
    int M, N, K, ksteps;  // ksteps: even
    int tiles_m, tiles_n, steps_per_split;
    float scale;
    int activation;
};

// Whether A's 32-row blocks [ra, ra + TM) against B's [rb, rb + TN) hold anything the three pieces cannot carry, over block
// pairs [pair0, pair1): wavefront-uniform.
template <int TM, int TN>
__device__ __forceinline__ bool split_status_bad(const SplitGemmArgs &p, int ra, int rb, int pair0, int pair1, int lane)
{
    const int pairs = p.ksteps / 2, blocks_a = (p.M + 31) / 32, blocks_b = (p.N + 31) / 32;
    unsigned top_a = 0, top_b = 0;
    for (int i = pair0 + lane; i < pair1; i += 64) {
#pragma unroll
        for (int b = 0; b < TM; ++b)  // (blocks past the end repeat the last one)
            top_a = max(top_a, p.status_a[static_cast<size_t>(min(ra + b, blocks_a - 1)) * pairs + i]);
#pragma unroll
        for (int b = 0; b < TN; ++b) top_b = max(top_b, p.status_b[static_cast<size_t>(min(rb + b, blocks_b - 1)) * pairs + i]);
    }
    return !split_in_range(wave_top(top_a), wave_top(top_b), p.K);
}

// acc = a marked tile's sums over terms [k_begin, k_end), from the original operands on the f32 matrix cores: f32 arithmetic,
// infinities and NaN included.  Eight terms at a time straight from memory, four in each half of the wavefront; rows past
// the end repeat the last one.  Bound by those loads.  2048³ with one NaN in every tile row, and with NaN throughout, 380 µs (97 without; a
// chain of multiply-adds per value took 30000), 1576×3072×768 200 (52; 7000 to 13000).
template <int TM, int TN>
__device__ __forceinline__ void split_f32_sums(const SplitGemmArgs &p, int row_first, int col_first, int k_begin, int k_end, int lane,
                                               f32x16 (&acc)[TM][TN])
{
    const int li = lane & 31, lh = lane >> 5;
    const float *a_row[TM], *b_row[TN];
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) a_row[tm] = p.A + static_cast<size_t>(min(row_first + tm * 32 + li, p.M - 1)) * p.a_row;
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) b_row[tn] = p.B + static_cast<size_t>(min(col_first + tn * 32 + li, p.N - 1)) * p.b_col;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
            acc[tm][tn] = f32x16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto load4 = [&](const float *row, int stride, int k, f32x4 &v) {
        if (k + 4 <= k_end && stride == 1) {
            v = *reinterpret_cast<const f32x4_a4 *>(row + k);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = k + e < k_end ? row[static_cast<size_t>(k + e) * stride] : 0.0f;
        }
    };
    for (int k = k_begin + lh * 4; k - lh * 4 < k_end; k += 8) {
        f32x4 a[TM], b[TN];
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) load4(a_row[tm], p.a_k, k, a[tm]);
#pragma unroll
        for (int tn = 0; tn < TN; ++tn) load4(b_row[tn], p.b_k, k, b[tn]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[tn][e], a[tm][e], acc[tm][tn], 0, 0, 0);
    }
}

template <int BM, int BN, int WM, int WN, int STAGES>
__device__ __forceinline__ void gemm_f32_split_body(const SplitGemmArgs &p)
{
    using Tile = SplitTile<BM, BN, WM, WN, STAGES>;
    constexpr int WTM = Tile::WTM, WTN = Tile::WTN, TM = Tile::TM, TN = Tile::TN;
    constexpr int PIECES = Tile::PIECES, LOADS = Tile::LOADS, STAGE = Tile::STAGE;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_bytes[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int li = lane & 31, lh = lane >> 5;

    // Every XCD takes one contiguous run of tiles, walked in groups of 4 tile rows, so that what is resident on an XCD at
    // a time shares its A and B panels through that L2.
    const int grid = static_cast<int>(gridDim.x), xcd = static_cast<int>(blockIdx.x) & 7;
    int logical = xcd * (grid >> 3) + min(xcd, grid & 7) + (static_cast<int>(blockIdx.x) >> 3);
    const int tiles = p.tiles_m * p.tiles_n;
    const int split = logical / tiles;
    logical -= split * tiles;
    constexpr int GROUP_M = 4;
    const int width = GROUP_M * p.tiles_n;
    const int group = logical / width;
    const int first_m = group * GROUP_M;
    const int group_size = min(p.tiles_m - first_m, GROUP_M);
    const int m0 = (first_m + (logical % width) % group_size) * BM, n0 = (logical % width) / group_size * BN;
    const int step0 = split * p.steps_per_split;
    const int steps = min(p.steps_per_split, p.ksteps - step0);

    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char *>(p.blocks), 0, static_cast<int>(p.bytes), 0x00020000);
    // Piece q of a stage: fragment q % 3 of row block q / 3 of the tile (A's blocks first).
    unsigned piece_off[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int q = min(wave * LOADS + i, PIECES - 1);
        const int block = q / 3, plane = q % 3;
        piece_off[i] = plane * 1024u + (block < BM / 32 ? split_block_offset(m0, block, p.M, p.ksteps, step0)
                                                        : p.b_base + split_block_offset(n0, block - BM / 32, p.N, p.ksteps, step0));
    }
    const unsigned lane_off = lane * 16;
    struct Where {
        unsigned step_off, lane_off;  // past the last step: outside the buffer (zeros, no memory access)
    };
    auto load = [&](int stage, int i, const Where &where) {
        const int q = min(wave * LOADS + i, PIECES - 1);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_ptr)(lds_bytes + stage * STAGE + q * 1024), 16, where.lane_off,
                                                 piece_off[i] + where.step_off, 0, 0);
    };

    f32x16 acc[TM][TN];
    const bool bad = split_product_loop<BM, BN, WM, WN, STAGES>(
        lds_bytes, wave, lane, steps, acc, [&](int t) { return Where{t * 3072u, t < steps ? lane_off : 0x80000000u}; }, load,
        [&] { return split_status_bad<TM, TN>(p, m0 / 32 + wm * TM, n0 / 32 + wn * TN, step0 / 2, (step0 + steps) / 2, lane); });

    // Epilogue through a strip of LDS per wavefront, so that stores and residual loads cover whole row segments.
    __syncthreads();
    constexpr int C_STRIDE = WTN + 4;
    constexpr int LPR = WTN / 4, ROWS_PER_PASS = 64 / LPR, PASSES = 32 / ROWS_PER_PASS;
    float *strip = reinterpret_cast<float *>(lds_bytes) + wave * (32 * C_STRIDE);
    const int row_first = m0 + wm * WTM, col_first = n0 + wn * WTN;
    const int col0 = col_first + (lane & (LPR - 1)) * 4;
    if (bad) split_f32_sums<TM, TN>(p, row_first, col_first, step0 * 16, min(p.K, (step0 + steps) * 16), lane, acc);
    const float unscale = bad ? 1.0f : kSplitUnscale;
    float *const C = p.C + static_cast<size_t>(split) * p.M * p.N;
    float bias[4] = {-0.0f, -0.0f, -0.0f, -0.0f};  // x + -0.0f == x for every x
    if (p.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (col0 + e < p.N) bias[e] = p.bias[col0 + e];
    }
    with_epilogue_ops(p.activation, p.residual != nullptr, [&](auto &&act, auto has_residual) {
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const int row_base = row_first + tm * 32;
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<float4 *>(&strip[li * C_STRIDE + tn * 32 + g * 8 + lh * 4]) =
                        make_float4(acc[tm][tn][4 * g] * unscale, acc[tm][tn][4 * g + 1] * unscale,
                                    acc[tm][tn][4 * g + 2] * unscale, acc[tm][tn][4 * g + 3] * unscale);
#pragma unroll
            for (int j = 0; j < PASSES; ++j) {
                const int local_row = j * ROWS_PER_PASS + lane / LPR;
                const int row = row_base + local_row;
                const float4 s4 = *reinterpret_cast<const float4 *>(&strip[local_row * C_STRIDE + (lane & (LPR - 1)) * 4]);
                if (row >= p.M || col0 >= p.N) continue;
                const size_t idx = static_cast<size_t>(row) * p.N + col0;
                const float v[4] = {s4.x * p.scale + bias[0], s4.y * p.scale + bias[1], s4.z * p.scale + bias[2], s4.w * p.scale + bias[3]};
                if (col0 + 4 <= p.N) {
                    f32x4_a4 out = {v[0], v[1], v[2], v[3]};
                    if constexpr (decltype(has_residual)::value) out += *reinterpret_cast<const f32x4_a4 *>(p.residual + idx);
                    *reinterpret_cast<f32x4_a4 *>(C + idx) = f32x4_a4{act(out[0]), act(out[1]), act(out[2]), act(out[3])};
                } else {
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                        if (col0 + e >= p.N) continue;
                        float value = v[e];
                        if constexpr (decltype(has_residual)::value) value += p.residual[idx + e];
                        C[idx + e] = act(value);
                    }
                }
            }
        }
    });
}

// (Plain kernels around the templated body: a kernel template whose body uses the LDS-load builtins loses its host-side
// launch stub with this compiler.)
__global__ __launch_bounds__(512) void gemm_f32_split_256x128_kernel(SplitGemmArgs p) { gemm_f32_split_body<256, 128, 4, 2, 3>(p); }
__global__ __launch_bounds__(256) void gemm_f32_split_160x128_kernel(SplitGemmArgs p) { gemm_f32_split_body<160, 128, 1, 4, 5>(p); }
__global__ __launch_bounds__(256, 2) void gemm_f32_split_128x128_kernel(SplitGemmArgs p) { gemm_f32_split_body<128, 128, 2, 2, 3>(p); }
__global__ __launch_bounds__(256) void gemm_f32_split_96x128_kernel(SplitGemmArgs p) { gemm_f32_split_body<96, 128, 1, 4, 3>(p); }
__global__ __launch_bounds__(256, 2) void gemm_f32_split_64x128_kernel(SplitGemmArgs p) { gemm_f32_split_body<64, 128, 2, 2, 4>(p); }
__global__ __launch_bounds__(256, 2) void gemm_f32_split_64x64_kernel(SplitGemmArgs p) { gemm_f32_split_body<64, 64, 2, 2, 6>(p); }

// The tile shapes, and what one 32×32 block of a tile costs per 16-term step (measured on N(0,1) operands with the chip
// full; the matrix pipe alone needs 19 ns of the four it shares between SIMDs at the clock that data allows).
struct SplitConfig {
    void (*kernel)(SplitGemmArgs);
    int bm, bn, threads, stages;
    double block_ns;
};
const SplitConfig kSplitConfigs[] = {
    {gemm_f32_split_256x128_kernel, 256, 128, 512, 3, 32.5}, {gemm_f32_split_160x128_kernel, 160, 128, 256, 5, 32.0},
    {gemm_f32_split_128x128_kernel, 128, 128, 256, 3, 33.5}, {gemm_f32_split_96x128_kernel, 96, 128, 256, 3, 35.0},
    {gemm_f32_split_64x128_kernel, 64, 128, 256, 4, 38.0},   {gemm_f32_split_64x64_kernel, 64, 64, 256, 6, 42.0},
};

struct SplitPlan {
    const SplitConfig *config = nullptr;
    int splits = 1, steps_per_split = 0;
    double us = 0.0;  // estimate, the splitting pass included
};

constexpr double kCopyBytesPerUs = 5.0e6;  // what streaming kernels reach here

// Tile shape and k-split with the least estimated time.  Work is handed out by whole tiles, so what counts is the
// fullest of the 256 compute units: 1576×3072×768 is 240 tiles of 160×128 (one round, 41 µs) but 312 of 128×128 (two,
// 50 µs).  A k-split costs its partial planes (written and read once) and a launch.
SplitPlan plan_split(size_t m, size_t n, size_t k, bool may_split_k)
{
    const size_t ksteps = (k + 31) / 32 * 2;
    SplitPlan best;
    for (const SplitConfig &c : kSplitConfigs) {
        const size_t tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn);
        const double blocks = c.bm / 32 * (c.bn / 32);
        for (size_t splits = 1; splits <= 8; ++splits) {
            if (splits > 1 && (!may_split_k || ksteps / splits < 16 || tiles * splits > 1024)) break;
            const size_t steps = (ksteps / 2 + splits - 1) / splits * 2;
            if (splits > 1 && (splits - 1) * steps >= ksteps) continue;
            const double rounds = static_cast<double>((tiles * splits + 255) / 256);
            double us = 4.5 + rounds * (steps * std::max(blocks * c.block_ns * 1e-3, 0.16) + 1.0) + 4.0 * m * n * splits / kCopyBytesPerUs;
            if (splits > 1) us += 3.0 + 4.0 * m * n * (splits + 1) / kCopyBytesPerUs;
            if (best.config == nullptr || us < best.us) {
                best.config = &c;
                best.splits = static_cast<int>(splits);
                best.steps_per_split = static_cast<int>(steps);
                best.us = us;
            }
        }
    }
    best.us += 4.5 + 10.0 * (static_cast<double>(m) + n) * k / 7.0e6;  // the splitting pass: 4 bytes read, 6 written a value
    return best;
}

unsigned split_groups(SplitJob &job)
{
    job.groups_k = static_cast<unsigned>(job.transposed ? (job.k + 31) / 32 : (job.k + 127) / 128);
    return job.groups_k * static_cast<unsigned>(job.transposed ? (job.rows + 127) / 128 : (job.rows + 31) / 32);
}

}  // namespace

bool gemm_f32_split_applies(size_t m, size_t n, size_t k, double other_us, bool may_split_k)
{
    if (k < 64 || m < 32 || n < 32) return false;
    // all block offsets below 2^31, so that the ones past the end can be marked by bit 31
    const double bytes = (static_cast<double>(m) + n + 64) * (static_cast<double>(k) + 32) * 6.0;
    if (bytes >= static_cast<double>(1ull << 31)) return false;
    return plan_split(m, n, k, may_split_k).us < 0.9 * other_us;  // a tenth for the error of both estimates
}

GemmSplitPlanReport gemm_f32_split_plan_report(size_t m, size_t n, size_t k)
{
    const SplitPlan plan = plan_split(m, n, k, true);
    const SplitConfig &config = *plan.config;
    const int ksteps = static_cast<int>((k + 31) / 32 * 2);
    const int rows[2] = {static_cast<int>(m), static_cast<int>(n)}, tile[2] = {config.bm, config.bn};
    GemmSplitPlanReport report{};
    report.tile_rows = config.bm;
    report.tile_cols = config.bn;
    report.k_splits = plan.splits;
    report.steps_per_split = plan.steps_per_split;
    for (int side = 0; side < 2; ++side) {
        const int tiles = (rows[side] + tile[side] - 1) / tile[side];
        (side == 0 ? report.tiles_m : report.tiles_n) = tiles;
        report.bytes[side] = static_cast<uint64_t>((rows[side] + 31) / 32) * ksteps * 3072;
        for (int t = 0; t < tiles; ++t)
            for (int block = 0; block < tile[side] / 32; ++block)  // the last fragment of the last step
                report.reach[side] = std::max<uint64_t>(report.reach[side], split_block_offset(t * tile[side], block, rows[side], ksteps, ksteps - 1) + 3072ull);
    }
    return report;
}

hipError_t launch_gemm_f32_split(size_t m, size_t n, size_t k, bool lhs_transposed, const float *lhs, bool rhs_packed, const float *rhs,
                                 float *out, const GemmEpilogue &epilogue, hipStream_t stream, bool may_split_k)
{
    const SplitPlan plan = plan_split(m, n, k, may_split_k);
    const SplitConfig &config = *plan.config;
    const size_t ksteps = (k + 31) / 32 * 2, rows_a = (m + 31) / 32, rows_b = (n + 31) / 32;
    const size_t bytes_a = rows_a * ksteps * 3072, bytes_b = rows_b * ksteps * 3072;
    void *blocks = nullptr, *planes = nullptr;
    hipError_t rc = stream_workspace_slot(stream, 1, bytes_a + bytes_b + (rows_a + rows_b) * (ksteps / 2) * sizeof(unsigned), &blocks);
    if (rc == hipSuccess && plan.splits > 1) rc = stream_workspace(stream, plan.splits * m * n * sizeof(float), &planes);
    if (rc != hipSuccess) return rc;
    unsigned char *const base = static_cast<unsigned char *>(blocks);
    unsigned *const status = reinterpret_cast<unsigned *>(base + bytes_a + bytes_b);

    SplitJob job_a{lhs, base, status, static_cast<int>(m), static_cast<int>(k), static_cast<int>(lhs_transposed ? m : k),
                   lhs_transposed ? 1 : 0, static_cast<int>(ksteps), 0};
    SplitJob job_b{rhs, base + bytes_a, status + rows_a * (ksteps / 2), static_cast<int>(n), static_cast<int>(k),
                   static_cast<int>(rhs_packed ? k : n), rhs_packed ? 0 : 1, static_cast<int>(ksteps), 0};
    const unsigned groups_a = split_groups(job_a), groups_b = split_groups(job_b);
    hipLaunchKernelGGL(split_operands_kernel, dim3(groups_a + groups_b), dim3(256), 0, stream, job_a, job_b, groups_a);
    rc = hipGetLastError();
    if (rc != hipSuccess) return rc;

    SplitGemmArgs args;
    args.blocks = base;
    args.b_base = static_cast<unsigned>(bytes_a);
    args.bytes = static_cast<unsigned>(bytes_a + bytes_b);
    args.status_a = job_a.status;
    args.status_b = job_b.status;
    args.A = lhs;
    args.B = rhs;
    args.a_row = static_cast<int>(lhs_transposed ? 1 : k);
    args.a_k = static_cast<int>(lhs_transposed ? m : 1);
    args.b_col = static_cast<int>(rhs_packed ? k : 1);
    args.b_k = static_cast<int>(rhs_packed ? 1 : n);
    args.M = static_cast<int>(m);
    args.N = static_cast<int>(n);
    args.K = static_cast<int>(k);
    args.ksteps = static_cast<int>(ksteps);
    args.tiles_m = static_cast<int>((m + config.bm - 1) / config.bm);
    args.tiles_n = static_cast<int>((n + config.bn - 1) / config.bn);
    args.steps_per_split = plan.steps_per_split;
    const bool split = plan.splits > 1;
    args.C = split ? static_cast<float *>(planes) : out;
    args.bias = split ? nullptr : epilogue.bias;
    args.residual = split ? nullptr : epilogue.residual;
    args.scale = split ? 1.0f : epilogue.scale;
    args.activation = split ? ST_HIP_ACT_NONE : epilogue.activation;
    const size_t lds = static_cast<size_t>(config.bm + config.bn) / 32 * 3072 * config.stages;
    rc = hipFuncSetAttribute(reinterpret_cast<const void *>(config.kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (rc != hipSuccess) return rc;
    const size_t groups = static_cast<size_t>(args.tiles_m) * args.tiles_n * plan.splits;
    hipLaunchKernelGGL(config.kernel, dim3(static_cast<unsigned>(groups)), dim3(config.threads), lds, stream, args);
    rc = hipGetLastError();
    if (rc != hipSuccess || !split) return rc;
    return launch_f32_slice_reduce(m, n, static_cast<size_t>(plan.splits), args.C, out, epilogue, stream);
}

}  // namespace sthip
