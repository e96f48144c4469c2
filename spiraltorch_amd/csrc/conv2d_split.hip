// Large f32 convolutions on the bf16 matrix cores: the implicit GEMM out(pixels × C_out) = patches · weightᵀ with both
// operands as three exact bf16 pieces (the arithmetic of gemm_f32_split.hip, and its error).  The forward pass and, with
// the taps flipped and the channel roles swapped, grad_input of layers with stride 1 (crates/st-nn/src/layers/conv.rs:803-809).
//
// One pass re-lays the operands.  The images become channels-last strips of 16 channels, zero-padded, piece by piece:
// [image][16-channel block][piece][half][padded pixel][8], so that a step of the reduction (one tap, 16 channels) of 32
// pixels is one load of two 512-byte runs per piece in the matrix instruction's operand order, wherever the pixels lie: each
// lane keeps the offset of its own pixel, and the tap and channel block are one scalar offset.  No patch matrix, no
// bounds checks along x and y.  The weights become blocks of 32 rows × 16 terms in the same step order.
//
// What bounds it is the matrix cores on random operands, as in the GEMM (21 ns per 32×32×16 instruction and SIMD).
// Of the whole call, f32 kernels -> here, batch 32 unless given, 3×3: 64 -> 128 on 56×56 146 -> 115 µs (of which 15 are the
// pass), 128 -> 128 on 28×28 93 -> 65, 256 -> 256 on 14×14 99 -> 64, 512 -> 512 on 7×7 119 -> 72,
// 250 -> 250 on 14×15, batch 31, 189 -> 64, 24 -> 96 5×5 on 112×112, batch 4, 105 -> 67, 256 -> 256 on 28×28, batch 2, 41 -> 30.
// 64 -> 64 on 56×56 and one-tap layers stay on the f32 kernels (70 against 69 µs, 46 against 51): the pass costs what the
// matrix cores save.  Errors against float64 are 0.34 to 0.62 of those of the kernels that ran before (rms, six layers with
// rectified N(0,1) images).
//
// Values the scaled pieces cannot carry or whose sums could overflow (gemm_f32_split.hip) are found by the pass, by the image
// and by the weight block; tiles that see such magnitudes are summed on the f32 matrix cores from the original operands.  Small
// values, subnormal ones included, cost nothing.
#include <algorithm>

#include "kernels.h"
#include "split_product.h"

namespace sthip {

namespace {

typedef __attribute__((address_space(3))) void *lds_void_ptr;

constexpr unsigned kOutside = 0x80000000u;

struct ConvSplitArgs {
    const float *input, *weight, *bias;
    float *out;  // the result, or the planes of the partial sums
    unsigned char *pieces;  // the images' strips, then the weights' blocks at weight_base
    unsigned *status;  // the largest magnitude (split_top): a word per workgroup of the image pass, then per weight block and step
    ConvShape s;
    int weight_row, weight_channel, flip;  // element strides of the weights; flip: taps from last to first
    int padded_w, padded_pixels, channel_blocks, taps, groups_px;
    unsigned plane_bytes, block_bytes, image_bytes, weight_base, weight_status, bytes, image_groups;
    int ksteps, real_steps;  // channel_blocks · taps, and that rounded up to even
    int M, spatial, tiles_m, tiles_n, steps_per_split;
    int activation;
};

// Images: a workgroup takes 128 padded pixels of one 16-channel block, two lanes a pixel, eight channels each: reads are
// 128-byte runs of eight planes in flight, writes 1 KB a wavefront and piece.  Weights: a wavefront a block and step.
__global__ __launch_bounds__(256) void conv_split_pieces_kernel(ConvSplitArgs p)
{
    __shared__ unsigned tops[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const ConvShape &s = p.s;
    float x[8];
    uint32_t piece[3][4];
    if (blockIdx.x < p.image_groups) {
        const int group = static_cast<int>(blockIdx.x % p.groups_px);
        const int block = static_cast<int>(blockIdx.x / p.groups_px);  // image · channel_blocks + channel block
        const int half = lane >> 5;
        const int image = block / p.channel_blocks, c0 = (block - image * p.channel_blocks) * 16 + half * 8;
        const int pixel = group * 128 + wave * 32 + (lane & 31);
        const int yy = pixel / p.padded_w, y = yy - s.pad_h, col = pixel - yy * p.padded_w - s.pad_w;
        const bool inside = pixel < p.padded_pixels && y >= 0 && y < s.h && col >= 0 && col < s.w;
        const size_t plane = static_cast<size_t>(s.h) * s.w;
        const float *src = p.input + (static_cast<size_t>(image) * s.c_in + c0) * plane + (inside ? static_cast<size_t>(y) * s.w + col : 0);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = inside && c0 + e < s.c_in ? src[e * plane] : 0.0f;
        split_pieces(x, piece);
        if (pixel < p.padded_pixels) {
            unsigned char *dst = p.pieces + static_cast<size_t>(block) * p.block_bytes + (static_cast<size_t>(half) * p.padded_pixels + pixel) * 16;
#pragma unroll
            for (int i = 0; i < 3; ++i)
                *reinterpret_cast<uint4 *>(dst + static_cast<size_t>(i) * p.plane_bytes) = make_uint4(piece[i][0], piece[i][1], piece[i][2], piece[i][3]);
        }
        const unsigned top = wave_top(split_top(x, 0u));
        if (lane == 0) tops[wave] = top;
        __syncthreads();
        if (tid == 0) p.status[blockIdx.x] = max(max(tops[0], tops[1]), max(tops[2], tops[3]));
        return;
    }
    const int unit = static_cast<int>(blockIdx.x - p.image_groups) * 4 + wave;  // row block · ksteps + step
    const int row_block = unit / p.ksteps, step = unit - row_block * p.ksteps;
    if (row_block * 32 >= s.c_out) return;
    const int row = row_block * 32 + (lane & 31), channel_block = step / p.taps, tap = step - channel_block * p.taps;
    const int c0 = channel_block * 16 + (lane >> 5) * 8;
    const float *src = p.weight + static_cast<size_t>(row) * p.weight_row + (p.flip ? p.taps - 1 - tap : tap);
#pragma unroll
    for (int e = 0; e < 8; ++e)  // (the step that makes their number even lies past the last channel)
        x[e] = row < s.c_out && c0 + e < s.c_in ? src[static_cast<size_t>(c0 + e) * p.weight_channel] : 0.0f;
    split_pieces(x, piece);
    unsigned char *dst = p.pieces + p.weight_base + static_cast<size_t>(unit) * 3072 + lane * 16;
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4 *>(dst + i * 1024) = make_uint4(piece[i][0], piece[i][1], piece[i][2], piece[i][3]);
    const unsigned top = wave_top(split_top(x, 0u));
    if (lane == 0) p.status[p.weight_status + unit] = top;
}

// Whether pixel rows [row0, row0 + rows) against output channels [oc0, oc0 + cols) hold anything the pieces cannot carry, by
// the status words of the images and weight blocks they lie in.
__device__ __forceinline__ bool conv_split_bad(const ConvSplitArgs &p, int row0, int rows, int oc0, int cols, int lane)
{
    const ConvShape &s = p.s;
    if (row0 >= p.M || oc0 >= s.c_out) return false;
    const int row_end = min(row0 + rows, p.M), oc_end = min(oc0 + cols, s.c_out);
    const unsigned per_image = static_cast<unsigned>(p.channel_blocks) * p.groups_px;
    unsigned top_image = 0, top_weight = 0;
    const unsigned end = (static_cast<unsigned>((row_end - 1) / p.spatial) + 1) * per_image;
    for (unsigned i = static_cast<unsigned>(row0 / p.spatial) * per_image + lane; i < end; i += 64) top_image = max(top_image, p.status[i]);
    const int unit_end = ((oc_end - 1) / 32 + 1) * p.ksteps;
    for (int i = oc0 / 32 * p.ksteps + lane; i < unit_end; i += 64) top_weight = max(top_weight, p.status[p.weight_status + i]);
    return !split_in_range(wave_top(top_image), wave_top(top_weight), s.c_in * p.taps);
}

// acc = a marked tile's sums over `steps` steps, from the original operands on the f32 matrix cores: f32 arithmetic,
// infinities and NaN included.  A step's sixteen channels straight from memory, eight in each half of the wavefront; rows
// past the end repeat the last one.  64 -> 128 channels on 56×56, batch 32, with NaN throughout 460 µs, with one 188 (115 without; a chain
// of multiply-adds per value took 7600 and 2100), 256 -> 256 on 14×14 310 (67; 7000).
template <int TM, int TN>
__device__ __forceinline__ void conv_split_f32_sums(const ConvSplitArgs &p, int row_first, int col_first, int step0, int steps, int lane,
                                                    f32x16 (&acc)[TM][TN])
{
    const ConvShape &s = p.s;
    const int li = lane & 31, lh = lane >> 5;
    const size_t plane = static_cast<size_t>(s.h) * s.w;
    const float *image[TM], *weight[TN];
    int y0[TM], x0[TM];
#pragma unroll
    for (int tm = 0; tm < TM; ++tm) {
        const int row = min(row_first + tm * 32 + li, p.M - 1);
        const int n = row / p.spatial, px = row - n * p.spatial, oy = px / s.ow;
        image[tm] = p.input + static_cast<size_t>(n) * s.c_in * plane;
        y0[tm] = oy * s.stride_h - s.pad_h;
        x0[tm] = (px - oy * s.ow) * s.stride_w - s.pad_w;
    }
#pragma unroll
    for (int tn = 0; tn < TN; ++tn) weight[tn] = p.weight + static_cast<size_t>(min(col_first + tn * 32 + li, s.c_out - 1)) * p.weight_row;
#pragma unroll
    for (int tm = 0; tm < TM; ++tm)
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
            acc[tm][tn] = f32x16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int t = step0; t < min(step0 + steps, p.real_steps); ++t) {
        const int channel_block = t / p.taps, tap = t - channel_block * p.taps, ky = tap / s.kw, kx = tap - ky * s.kw;
        const int c0 = channel_block * 16 + lh * 8, weight_tap = p.flip ? p.taps - 1 - tap : tap;
        float x[TM][8], w[TN][8];
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const int y = y0[tm] + ky * s.dil_h, col = x0[tm] + kx * s.dil_w;
            const bool inside = y >= 0 && y < s.h && col >= 0 && col < s.w;
            const float *src = image[tm] + (inside ? static_cast<size_t>(y) * s.w + col : 0);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[tm][e] = inside && c0 + e < s.c_in ? src[(c0 + e) * plane] : 0.0f;
        }
#pragma unroll
        for (int tn = 0; tn < TN; ++tn)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                w[tn][e] = c0 + e < s.c_in ? weight[tn][static_cast<size_t>(c0 + e) * p.weight_channel + weight_tap] : 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int tm = 0; tm < TM; ++tm)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn) acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[tn][e], x[tm][e], acc[tm][tn], 0, 0, 0);
    }
}

// Where the first tap of output pixel px lies among an image's padded pixels, and how far behind it tap `tap`.
__host__ __device__ inline int conv_split_pixel(const ConvShape &s, int padded_w, int px)
{
    const int oy = px / s.ow, ox = px - oy * s.ow;
    return oy * s.stride_h * padded_w + ox * s.stride_w;
}
__host__ __device__ inline int conv_split_tap(const ConvShape &s, int padded_w, int tap)
{
    const int ky = tap / s.kw, kx = tap - ky * s.kw;
    return ky * s.dil_h * padded_w + kx * s.dil_w;
}

template <int BM, int BN, int WM, int WN, int STAGES>
__device__ __forceinline__ void conv_split_body(const ConvSplitArgs &p)
{
    using Tile = SplitTile<BM, BN, WM, WN, STAGES>;
    constexpr int TM = Tile::TM, TN = Tile::TN, LOADS = Tile::LOADS;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_bytes[];
    const ConvShape &s = p.s;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int wm = wave / WN, wn = wave % WN;
    const int li = lane & 31, lh = lane >> 5;

    // Every XCD takes one contiguous run of tiles, those of the same pixels next to each other: neighbouring tiles share
    // image rows through that L2.
    const int grid = static_cast<int>(gridDim.x), xcd = static_cast<int>(blockIdx.x) & 7;
    int logical = xcd * (grid >> 3) + min(xcd, grid & 7) + (static_cast<int>(blockIdx.x) >> 3);
    const int tiles = p.tiles_m * p.tiles_n;
    const int split = logical / tiles;
    logical -= split * tiles;
    const int m0 = logical / p.tiles_n * BM, n0 = logical % p.tiles_n * BN;
    const int step0 = split * p.steps_per_split;
    const int steps = min(p.steps_per_split, p.ksteps - step0);

    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(p.pieces, 0, static_cast<int>(p.bytes), 0x00020000);
    // A piece of the image side: the lane's own pixel (pixels past the last read zeros); of the weight side: a block in
    // operand order (blocks past the last channel repeat the last, what they give is not stored).
    unsigned vector_off[LOADS], scalar_off[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int q = min(wave * LOADS + i, Tile::PIECES - 1);
        const int block = q / 3, plane = q % 3;
        if (block < BM / 32) {
            const int row = m0 + block * 32 + li;
            const int image = row / p.spatial, px = row - image * p.spatial;
            vector_off[i] = row < p.M ? static_cast<unsigned>(image) * p.image_bytes +
                                            static_cast<unsigned>(lh * p.padded_pixels + conv_split_pixel(s, p.padded_w, px)) * 16u
                                      : kOutside;
            scalar_off[i] = plane * p.plane_bytes;
        } else {
            const unsigned row_block = min(n0 / 32 + block - BM / 32, (s.c_out - 1) / 32);
            vector_off[i] = lane * 16;
            scalar_off[i] = p.weight_base + row_block * p.ksteps * 3072u + plane * 1024u;
        }
    }
    struct Where {
        unsigned image_off, weight_off;
        bool live;
    };
    // Steps walk the taps of a channel block, then the next block.  The step that makes their number even repeats the
    // last one's pixels (its weights are zeros).
    int ky = 0, kx = 0;
    unsigned image_off = 0;
    {
        const int first = min(step0, p.real_steps - 1), channel_block = first / p.taps, tap = first - channel_block * p.taps;
        ky = tap / s.kw;
        kx = tap - ky * s.kw;
        image_off = channel_block * p.block_bytes + static_cast<unsigned>(conv_split_tap(s, p.padded_w, tap)) * 16u;
    }
    const unsigned next_row = static_cast<unsigned>(s.dil_h * p.padded_w - (s.kw - 1) * s.dil_w) * 16u;
    const unsigned next_block = p.block_bytes - static_cast<unsigned>((s.kh - 1) * s.dil_h * p.padded_w + (s.kw - 1) * s.dil_w) * 16u;
    auto locate = [&](int t) {
        const Where where{image_off, static_cast<unsigned>(step0 + t) * 3072u, t < steps};
        if (step0 + t + 1 < p.real_steps) {
            const bool row_done = kx + 1 == s.kw, block_done = row_done && ky + 1 == s.kh;
            image_off += block_done ? next_block : row_done ? next_row : static_cast<unsigned>(s.dil_w) * 16u;
            kx = row_done ? 0 : kx + 1;
            ky = block_done ? 0 : row_done ? ky + 1 : ky;
        }
        return where;
    };
    auto load = [&](int stage, int i, const Where &where) {
        const int q = min(wave * LOADS + i, Tile::PIECES - 1);
        const unsigned step_off = q < BM / 32 * 3 ? where.image_off : where.weight_off;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_ptr)(lds_bytes + stage * Tile::STAGE + q * 1024), 16,
                                                 where.live ? vector_off[i] : kOutside, scalar_off[i] + step_off, 0, 0);
    };
    const int row_first = m0 + wm * Tile::WTM, col_first = n0 + wn * Tile::WTN;
    f32x16 acc[TM][TN];
    const bool bad = split_product_loop<BM, BN, WM, WN, STAGES>(lds_bytes, wave, lane, steps, acc, locate, load, [&] {
        return conv_split_bad(p, row_first, Tile::WTM, col_first, Tile::WTN, lane);
    });

    if (bad) conv_split_f32_sums<TM, TN>(p, row_first, col_first, step0, steps, lane, acc);
    const float unscale = bad ? 1.0f : kSplitUnscale;

    // Register 4g + j of lane (li, lh) is pixel li, channel 8g + 4·lh + j: a store covers 128 bytes of two planes.
    float *const out = p.out + static_cast<size_t>(split) * p.M * s.c_out;
    with_epilogue_ops(p.activation, false, [&](auto &&act, auto) {
#pragma unroll
        for (int tm = 0; tm < TM; ++tm) {
            const int row = row_first + tm * 32 + li;
            const int image = row / p.spatial, px = row - image * p.spatial;
            float *const dst = out + static_cast<size_t>(image) * s.c_out * p.spatial + px;
#pragma unroll
            for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int oc = col_first + tn * 32 + (r >> 2) * 8 + lh * 4 + (r & 3);
                    if (row >= p.M || oc >= s.c_out) continue;
                    dst[static_cast<size_t>(oc) * p.spatial] = act(acc[tm][tn][r] * unscale + (p.bias ? p.bias[oc] : -0.0f));
                }
        }
    });
}

__global__ __launch_bounds__(256, 2) void conv_split_128x128_kernel(ConvSplitArgs p) { conv_split_body<128, 128, 2, 2, 3>(p); }
__global__ __launch_bounds__(256, 2) void conv_split_256x64_kernel(ConvSplitArgs p) { conv_split_body<256, 64, 4, 1, 2>(p); }
__global__ __launch_bounds__(256, 2) void conv_split_128x64_kernel(ConvSplitArgs p) { conv_split_body<128, 64, 2, 2, 4>(p); }
__global__ __launch_bounds__(256, 2) void conv_split_128x32_kernel(ConvSplitArgs p) { conv_split_body<128, 32, 4, 1, 5>(p); }
__global__ __launch_bounds__(256, 2) void conv_split_64x64_kernel(ConvSplitArgs p) { conv_split_body<64, 64, 2, 2, 6>(p); }

// Tiles of which two workgroups share a compute unit, so that one's first loads and stores run under the other's products
// (64 -> 128 channels, 56×56, batch 32, the whole call: 128×128 108 µs; 256×128 and 160×128, one workgroup a unit, 17 and 47
// more).  Over nineteen layers, every tile forced in turn, the plan below takes the fastest or one within 5 % of it, but for
// that layer: it takes 128×64 tiles, 112 to 118 µs.  Counting a last round that is not full as less than a round would choose
// right there and wrong elsewhere (of 24 other layers it recuts, 18 come out 3 to 20 % slower).
struct ConvSplitConfig {
    void (*kernel)(ConvSplitArgs);
    int bm, bn, threads, stages;
    double block_ns, tile_us;  // of a 32×32 block per step and of a tile besides, with the chip full
};
const ConvSplitConfig kConvSplitConfigs[] = {
    {conv_split_128x128_kernel, 128, 128, 256, 3, 37.0, 4.0}, {conv_split_256x64_kernel, 256, 64, 256, 2, 37.0, 5.0},
    {conv_split_128x64_kernel, 128, 64, 256, 4, 38.0, 3.0},   {conv_split_128x32_kernel, 128, 32, 256, 5, 46.0, 2.0},
    {conv_split_64x64_kernel, 64, 64, 256, 6, 43.0, 2.0},
};

constexpr double kStreamBytesPerUs = 5.0e6;

struct ConvSplitPlan {
    const ConvSplitConfig *config = nullptr;
    int splits = 1, steps_per_split = 0;
    double us = 0.0;
    size_t padded_h = 0, padded_w = 0, channel_blocks = 0, ksteps = 0, image_piece_bytes = 0, weight_bytes = 0;
};

// Tile shape and split of the reduction with the least estimated time: the fullest compute unit counts.
ConvSplitPlan plan_conv_split(const ConvShape &s)
{
    ConvSplitPlan best;
    best.padded_h = static_cast<size_t>(s.oh - 1) * s.stride_h + static_cast<size_t>(s.kh - 1) * s.dil_h + 1;
    best.padded_w = static_cast<size_t>(s.ow - 1) * s.stride_w + static_cast<size_t>(s.kw - 1) * s.dil_w + 1;
    best.channel_blocks = (static_cast<size_t>(s.c_in) + 15) / 16;
    const size_t ksteps = best.ksteps = (best.channel_blocks * s.kh * s.kw + 1) / 2 * 2;
    const size_t m = static_cast<size_t>(s.batch) * s.oh * s.ow, n = s.c_out;
    for (const ConvSplitConfig &c : kConvSplitConfigs) {
        const size_t tiles = ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn);
        const double blocks = c.bm / 32 * (c.bn / 32);
        for (size_t splits = 1; splits <= 8; ++splits) {
            if (splits > 1 && (ksteps / splits < 16 || tiles * splits > 1024)) break;
            const size_t steps = (ksteps / 2 + splits - 1) / splits * 2;
            if (splits > 1 && (splits - 1) * steps >= ksteps) continue;
            const double rounds = static_cast<double>((tiles * splits + 255) / 256);
            const double alone = rounds > 1.0 ? 1.0 : 1.12;  // nothing to run under a lone workgroup's loads
            double us = 4.0 + alone * rounds * (steps * blocks * c.block_ns * 1e-3 + c.tile_us) + 2.0 * m * n * splits / kStreamBytesPerUs;
            if (splits > 1) us += 3.0 + 4.0 * m * n * (splits + 1) / kStreamBytesPerUs;
            if (best.config == nullptr || us < best.us) {
                best.config = &c;
                best.splits = static_cast<int>(splits);
                best.steps_per_split = static_cast<int>(steps);
                best.us = us;
            }
        }
    }
    const double values = static_cast<double>(s.batch) * best.channel_blocks * 16 * best.padded_h * best.padded_w;
    best.us += 1.5 + (10.0 * values + 10.0 * n * ksteps * 16) / 5.6e6;  // the splitting pass: 4 bytes read, 6 written a value
    return best;
}

__global__ __launch_bounds__(256) void conv_split_reduce_kernel(size_t count, int splits, int c_out, int spatial, int activation,
                                                                const float *partial, const float *bias, float *out)
{
    const size_t idx = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= count) return;
    float part[8], value = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) part[j] = j < splits ? partial[j * count + idx] : 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) value += part[j];
    if (bias) value += bias[(idx / spatial) % c_out];
    out[idx] = apply_activation(value, activation);
}

}  // namespace

bool conv2d_f32_split_applies(const ConvShape &s, double other_us)
{
    if (s.batch == 0 || s.oh == 0 || s.ow == 0 || s.c_out < 16 || s.c_in < 16) return false;
    const double m = static_cast<double>(s.batch) * s.oh * s.ow, k = static_cast<double>(s.c_in) * s.kh * s.kw;
    const double flops = 2.0 * m * s.c_out * k;
    if (k < 64 || flops < 5e8) return false;  // (below, launches decide)

    const ConvSplitPlan plan = plan_conv_split(s);
    // every byte offset below 2^31, so that what lies outside can be marked by bit 31; pixel and group counts as 32-bit integers
    const double image_bytes = static_cast<double>(s.batch) * plan.channel_blocks * 96.0 * plan.padded_h * plan.padded_w;
    const double weight_bytes = (s.c_out + 31) / 32 * 3072.0 * plan.ksteps;
    if (image_bytes + weight_bytes >= static_cast<double>(1ull << 31) - 65536.0) return false;
    if (static_cast<double>(s.c_in) * s.c_out * s.kh * s.kw >= static_cast<double>(1ull << 31) || m * s.c_out >= 4e9) return false;
    return plan.us < 0.95 * other_us;  // a margin for the error of both estimates
}

ConvSplitPlanReport conv2d_f32_split_plan_report(const ConvShape &s)
{
    const ConvSplitPlan plan = plan_conv_split(s);
    const int taps = s.kh * s.kw, padded_w = static_cast<int>(plan.padded_w), padded_pixels = static_cast<int>(plan.padded_h * plan.padded_w);
    ConvSplitPlanReport report{};
    report.tile_pixels = plan.config->bm;
    report.tile_channels = plan.config->bn;
    report.k_splits = plan.splits;
    report.steps_per_split = plan.steps_per_split;
    const uint64_t block_bytes = static_cast<uint64_t>(padded_pixels) * 96;
    report.image_bytes = static_cast<uint64_t>(s.batch) * plan.channel_blocks * block_bytes;
    report.weight_bytes = (static_cast<uint64_t>(s.c_out) + 31) / 32 * plan.ksteps * 3072;
    // the last lane, piece, tap and channel block of the last pixel's loads
    report.image_reach = (static_cast<uint64_t>(s.batch) * plan.channel_blocks - 1) * block_bytes + static_cast<uint64_t>(padded_pixels) * 64 +
                         (static_cast<uint64_t>(padded_pixels) + conv_split_pixel(s, padded_w, s.oh * s.ow - 1) + conv_split_tap(s, padded_w, taps - 1)) * 16 + 16;
    report.weight_reach = ((static_cast<uint64_t>(s.c_out) - 1) / 32 * plan.ksteps + plan.ksteps - 1) * 3072 + 3072;
    return report;
}

hipError_t launch_conv2d_f32_split(const ConvShape &shape, int activation, const float *input, const float *weight, bool adjoint_weight,
                                   const float *bias, float *out, hipStream_t stream)
{
    const ConvSplitPlan plan = plan_conv_split(shape);
    const ConvSplitConfig &config = *plan.config;
    ConvSplitArgs args;
    args.input = input;
    args.weight = weight;
    args.s = shape;
    args.taps = shape.kh * shape.kw;
    // weight[row][channel][tap], or the forward layer's weight[channel][row][flipped tap]
    args.weight_row = adjoint_weight ? args.taps : shape.c_in * args.taps;
    args.weight_channel = adjoint_weight ? shape.c_out * args.taps : args.taps;
    args.flip = adjoint_weight ? 1 : 0;
    args.padded_w = static_cast<int>(plan.padded_w);
    args.padded_pixels = static_cast<int>(plan.padded_h * plan.padded_w);
    args.channel_blocks = static_cast<int>(plan.channel_blocks);
    args.groups_px = (args.padded_pixels + 127) / 128;
    args.plane_bytes = static_cast<unsigned>(args.padded_pixels) * 32u;
    args.block_bytes = args.plane_bytes * 3u;
    args.image_bytes = args.block_bytes * static_cast<unsigned>(args.channel_blocks);
    args.ksteps = static_cast<int>(plan.ksteps);
    args.real_steps = args.channel_blocks * args.taps;
    const size_t image_bytes = static_cast<size_t>(shape.batch) * args.image_bytes;
    const size_t row_blocks = (static_cast<size_t>(shape.c_out) + 31) / 32, weight_units = row_blocks * plan.ksteps;
    const size_t bytes = image_bytes + weight_units * 3072;
    args.weight_base = static_cast<unsigned>(image_bytes);
    args.bytes = static_cast<unsigned>(bytes);
    args.image_groups = static_cast<unsigned>(static_cast<size_t>(shape.batch) * args.channel_blocks * args.groups_px);
    args.weight_status = args.image_groups;
    args.spatial = shape.oh * shape.ow;
    args.M = shape.batch * args.spatial;
    args.tiles_m = (args.M + config.bm - 1) / config.bm;
    args.tiles_n = (shape.c_out + config.bn - 1) / config.bn;
    args.steps_per_split = plan.steps_per_split;

    const bool split = plan.splits > 1;
    const size_t count = static_cast<size_t>(args.M) * shape.c_out;
    void *scratch = nullptr, *planes = nullptr;
    hipError_t rc = stream_workspace_slot(stream, 1, bytes + (args.image_groups + weight_units) * sizeof(unsigned), &scratch);
    if (rc == hipSuccess && split) rc = stream_workspace(stream, plan.splits * count * sizeof(float), &planes);
    if (rc != hipSuccess) return rc;
    args.pieces = static_cast<unsigned char *>(scratch);
    args.status = reinterpret_cast<unsigned *>(args.pieces + bytes);
    args.out = split ? static_cast<float *>(planes) : out;
    args.bias = split ? nullptr : bias;
    args.activation = split ? ST_HIP_ACT_NONE : activation;

    hipLaunchKernelGGL(conv_split_pieces_kernel, dim3(args.image_groups + static_cast<unsigned>((weight_units + 3) / 4)), dim3(256), 0,
                       stream, args);
    rc = hipGetLastError();
    if (rc != hipSuccess) return rc;
    const size_t lds = static_cast<size_t>(config.bm + config.bn) / 32 * 3072 * config.stages;
    rc = hipFuncSetAttribute(reinterpret_cast<const void *>(config.kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (rc != hipSuccess) return rc;
    hipLaunchKernelGGL(config.kernel, dim3(static_cast<unsigned>(args.tiles_m * args.tiles_n * plan.splits)), dim3(config.threads), lds,
                       stream, args);
    rc = hipGetLastError();
    if (rc != hipSuccess || !split) return rc;
    hipLaunchKernelGGL(conv_split_reduce_kernel, dim3(static_cast<unsigned>((count + 255) / 256)), dim3(256), 0, stream, count,
                       plan.splits, shape.c_out, args.spatial, activation, args.out, bias, out);
    return hipGetLastError();
}

}  // namespace sthip
