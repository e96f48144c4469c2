// bf16 convolution with f32 sums (crates/st-nn/src/layers/conv.rs:685-748, 2559-2599 on bf16 operands): the implicit GEMM
// channels × pixels on the matrix cores, out(C_out × pixels) = weight · patchesᵀ, no patch matrix.
//
// One pass re-lays the operands in chunks of eight channels of one tap, 16 bytes a row: the images zero-padded as
// [image][8 channels][position][8], the weights as [8 channels][tap][C_out][8].  A request of a wavefront then takes one chunk of
// 64 pixels (or 64 output channels) as 1 KB of neighbouring addresses straight into LDS, in the matrix instruction's operand
// order: each lane keeps its own pixel's offset, and chunk and tap are one scalar, read from a table.  LDS rows are read as they
// were written, 512 contiguous bytes a half wavefront, so nothing is swizzled.  k is padded to eight channels (three channels and
// 49 taps are seven k-tiles of 64, not 49) and, at its end, to 64 with requests that lie outside.
//
// What bounds it: small layers two launches and the chain of k-tiles (0.12 µs each, 64×64 tiles), middling ones LDS traffic and the
// last round of tiles, large ones the matrix cores (0.53 µs a k-tile of 256×128, of which 0.43 µs are products at 2.4 GHz).
// Of a whole call, channels-last copies of 64 channels and 128- and 256-row tiles before -> here, batch × channels, side:
// 32×256 -> 256, 14: 42.9 -> 18.3 µs (of which 4.2 are the pass; 12.9 before); 32×64 -> 128, 56: 41 -> 38; 32×256 -> 256, 28:
// 50 -> 42; 1×256 -> 256, 14: 32 -> 12; 32×3 -> 64, 112, 7×7 stride 2: 96 -> 25; 13×512 -> 192, 8, 5×5: 121 -> 21; 16×16 -> 32,
// 56: 18.5 -> 10.  Over 130 layers drawn from 1 to 32 images, 3 to 512 channels, 7 to 112 pixels a side: 0.49 of the time before,
// none slower.  More stages in flight (six and eight, one workgroup a unit) gain nothing, and 128×128 with four wavefronts
// of one 64×64 each is slower than with eight that halve k (20.8 against 17.9 µs on the first).
#include <algorithm>
#include <vector>

#include "device_math.h"
#include "kernels.h"

namespace sthip {

namespace {

typedef __attribute__((address_space(3))) void *lds_void_ptr;

#define ST_CONV16_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (7 << 4) | (15 << 8) | ((((n) >> 4) & 3) << 14))

constexpr unsigned kOutside = 0x80000000u;  // past the end of either operand: such loads give zeros

struct ConvBf16Args {
    const uint16_t *input, *weight;
    uint16_t *images, *weights;
    unsigned *image_offsets;  // by chunk: where its channels and tap lie from a pixel's first
    const float *bias;
    float *C32, *partial;
    uint16_t *C16;
    ConvShape s;
    int padded_w, padded_pixels;             // of an image's copy
    int step_h, step_w, stride_h, stride_w;  // image rows and columns between two of the copy, and its positions between two output pixels
    int channel_chunks, taps, chunks, k_tiles, offsets;
    unsigned image_bytes, weight_bytes;  // of all images, all weights
    int pixels, spatial, tiles_m;
    int activation, whole_chunks;
    int k_splits, tiles_per_split;
    unsigned image_groups, weight_groups, groups_px;
};

constexpr int kTapsPerPass = 64;  // of the weights' pass through LDS
constexpr int kMostStages = 5;

// One launch re-lays both operands and writes the table of the chunks' offsets.  Images: a thread a position of the copy and
// eight channels (reads are runs of eight planes, writes 1 KB a wavefront).  Weights: a workgroup sixteen output channels and
// eight channels, all taps, through LDS.
__global__ __launch_bounds__(256) void conv_bf16_chunks_kernel(ConvBf16Args p)
{
    __shared__ __attribute__((aligned(16))) uint16_t tile[16 * (8 * kTapsPerPass + 8)];
    const int tid = threadIdx.x;
    const ConvShape &s = p.s;
    if (blockIdx.x < p.image_groups) {
        const unsigned block = blockIdx.x / p.groups_px;  // image · channel_chunks + chunk
        const int pixel = static_cast<int>(blockIdx.x - block * p.groups_px) * 256 + tid;
        if (pixel >= p.padded_pixels) return;
        const int image = static_cast<int>(block) / p.channel_chunks, c0 = (static_cast<int>(block) - image * p.channel_chunks) * 8;
        const int yy = pixel / p.padded_w, y = yy * p.step_h - s.pad_h, x = (pixel - yy * p.padded_w) * p.step_w - s.pad_w;
        const bool inside = y >= 0 && y < s.h && x >= 0 && x < s.w;
        const size_t plane = static_cast<size_t>(s.h) * s.w;
        const uint16_t *src = p.input + (static_cast<size_t>(image) * s.c_in + c0) * plane + (inside ? static_cast<size_t>(y) * s.w + x : 0);
        uint32_t v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = inside && c0 + e < s.c_in ? src[e * plane] : 0u;
        *reinterpret_cast<uint4 *>(p.images + (static_cast<size_t>(block) * p.padded_pixels + pixel) * 8) =
            make_uint4(v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16);
        return;
    }
    const unsigned unit = blockIdx.x - p.image_groups;
    if (unit < p.weight_groups) {
        const int row_groups = (s.c_out + 15) / 16;
        const int chunk = static_cast<int>(unit) / row_groups, row0 = (static_cast<int>(unit) - chunk * row_groups) * 16;
        for (int tap0 = 0; tap0 < p.taps; tap0 += kTapsPerPass) {
            const int span = min(kTapsPerPass, p.taps - tap0), stride = 8 * span + 8;  // LDS: [row][channel][tap]
            __syncthreads();
            if (p.whole_chunks) {  // a row's values are one run of `taps` 16-byte pieces
                for (int i = tid; i < 16 * span; i += 256) {
                    const int row = i / span, piece = i - row * span;
                    if (row0 + row < s.c_out)
                        *reinterpret_cast<uint4 *>(&tile[row * stride + piece * 8]) =
                            *reinterpret_cast<const uint4 *>(p.weight + (static_cast<size_t>(row0 + row) * s.c_in + chunk * 8) * p.taps + piece * 8);
                }
            } else {
                for (int i0 = tid; i0 < 128 * span; i0 += 8 * 256) {
                    uint16_t value[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const int i = i0 + j * 256, rc = i / span, row = rc >> 3, c = rc & 7;
                        value[j] = 0;
                        if (i < 128 * span && row0 + row < s.c_out && chunk * 8 + c < s.c_in)
                            value[j] = p.weight[(static_cast<size_t>(row0 + row) * s.c_in + chunk * 8 + c) * p.taps + tap0 + (i - rc * span)];
                    }
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        const int i = i0 + j * 256, rc = i / span;
                        if (i < 128 * span) tile[(rc >> 3) * stride + (rc & 7) * span + (i - rc * span)] = value[j];
                    }
                }
            }
            __syncthreads();
            for (int i = tid; i < 16 * span; i += 256) {
                const int tap = i >> 4, row = i & 15;
                if (row0 + row >= s.c_out) continue;
                uint32_t v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = tile[row * stride + e * span + tap];
                *reinterpret_cast<uint4 *>(p.weights + ((static_cast<size_t>(chunk) * p.taps + tap0 + tap) * s.c_out + row0 + row) * 8) =
                    make_uint4(v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16);
            }
        }
        return;
    }
    for (int q = tid; q < p.offsets; q += 256) {
        const int chunk = q / p.taps, tap = q - chunk * p.taps, ky = tap / s.kw, kx = tap - ky * s.kw;
        p.image_offsets[q] = q < p.chunks ? (static_cast<unsigned>(chunk) * p.padded_pixels + ky * s.dil_h * p.padded_w + kx * s.dil_w) * 16u : 0u;
    }
}

struct ConvBf16Item {
    int split, tile_m, tile_n;
};
// Workgroup -> (run of k-tiles, tile): every XCD takes one contiguous run of tiles, those of the same pixels next to each other: they
// share an L2.
__host__ __device__ inline ConvBf16Item decode_conv_bf16_block(int grid, int k_splits, int tiles_m, int block)
{
    const int xcd = block & 7, more = grid & 7;
    const int logical = xcd * (grid >> 3) + (xcd < more ? xcd : more) + (block >> 3), tile = logical / k_splits;
    return ConvBf16Item{logical - tile * k_splits, tile % tiles_m, tile / tiles_m};
}

// Output channels 64·WM × pixels 64·WN by a workgroup of WM·WN·KS wavefronts, each 64×64 of it over a KS-th of every 64-wide
// k-tile (a wavefront tile of 64×64 reads four fragments for four products, the least LDS traffic its accumulators allow).
template <int WM, int WN, int KS, int STAGES>
__device__ __forceinline__ void conv_bf16_body(const ConvBf16Args &p)
{
    constexpr int WAVES = WM * WN * KS, BM = 64 * WM, BN = 64 * WN, STAGE = (BM + BN) * 128;
    constexpr int BLOCKS = WM + WN, LOADS = 8 * BLOCKS / WAVES, OWN = 8 / WAVES > 0 ? 8 / WAVES : 1;  // OWN: chunks of a k-tile a wavefront requests
    static_assert(LOADS == OWN * BLOCKS, "every wavefront requests whole chunks");
    static_assert(STAGES >= 3 && STAGES <= kMostStages, "requests in flight; the offset table's reserve");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_bytes[];
    const ConvShape &s = p.s;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN;
    const int li = lane & 31, lh = lane >> 5;
    const ConvBf16Item item = decode_conv_bf16_block(static_cast<int>(gridDim.x), p.k_splits, p.tiles_m, static_cast<int>(blockIdx.x));
    const int split = item.split;
    const int tile0 = split * p.tiles_per_split, tiles = min(p.tiles_per_split, p.k_tiles - tile0);
    const int m0 = item.tile_m * BM, n0 = item.tile_n * BN;

    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(p.weights, 0, static_cast<int>(p.weight_bytes), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(p.images, 0, static_cast<int>(p.image_bytes), 0x00020000);
    unsigned row_off[BLOCKS];
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) {
        if (b < WM) {
            const int row = m0 + b * 64 + lane;
            row_off[b] = row < s.c_out ? row * 16u : kOutside;
        } else {
            const int pixel = n0 + (b - WM) * 64 + lane;
            const int image = pixel / p.spatial, rest = pixel - image * p.spatial, oy = rest / s.ow, ox = rest - oy * s.ow;
            row_off[b] = pixel < p.pixels ? (static_cast<unsigned>(image) * p.channel_chunks * p.padded_pixels +
                                             static_cast<unsigned>(oy * p.stride_h * p.padded_w + ox * p.stride_w)) * 16u
                                          : kOutside;
        }
    }
    const unsigned weight_step = static_cast<unsigned>(s.c_out) * 16u;
    // (through the scalar cache: a vector load would wait behind the requests in flight)
    const auto *const offsets = (const __attribute__((address_space(4))) unsigned *)p.image_offsets;
    struct Where {
        unsigned image[OWN], weight[OWN];
        bool live[OWN];
    };
    auto locate = [&](int t) {
        Where where;
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
            const int q = (tile0 + t) * 8 + wave + o * WAVES;
            where.image[o] = offsets[q];
            where.live[o] = q < p.chunks;
            where.weight[o] = static_cast<unsigned>(min(q, p.chunks - 1)) * weight_step;
        }
        return where;
    };
    // request i of a k-tile: row block i % BLOCKS of this wavefront's chunk i / BLOCKS
    auto load = [&](int stage, int i, const Where &where) {
        const int o = i / BLOCKS, b = i % BLOCKS, chunk = wave + o * WAVES;
        unsigned char *const base = lds_bytes + stage * STAGE;
        const unsigned v = where.live[o] ? row_off[b] : kOutside;
        if (b < WM)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (lds_void_ptr)(base + chunk * (BM * 16) + b * 1024), 16, v, where.weight[o], 0, 0);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, (lds_void_ptr)(base + BM * 128 + chunk * (BN * 16) + (b - WM) * 1024), 16, v,
                                                     where.image[o], 0, 0);
    };

    f32x16 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
            acc[a][b] = f32x16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int t = 0; t < STAGES; ++t) {
        const Where where = locate(t);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) load(t, i, where);
    }
    Where ahead = locate(STAGES);
    constexpr int STEPS = 4 / KS, SLOTS = 4 * STEPS;
    const unsigned a_frag = (wm * 64 + li) * 16 + (ks * STEPS * 2 + lh) * (BM * 16);
    const unsigned b_frag = BM * 128 + (wn * 64 + li) * 16 + (ks * STEPS * 2 + lh) * (BN * 16);
    static_assert(LOADS <= SLOTS, "a slot for each request");
    // fragment 4·step + (0: A0, 1: B0, 2: B1, 3: A1) of a k-tile
    bf16x8 frag[2][SLOTS];
    auto read = [&](int buf, int stage, int slot) {
        const int step = slot / 4, which = slot % 4;
        const unsigned char *const base = lds_bytes + stage * STAGE;
        frag[buf][slot] = *reinterpret_cast<const bf16x8 *>(which == 0 || which == 3 ? base + a_frag + step * (BM * 32) + (which == 3 ? 512 : 0)
                                                                                     : base + b_frag + step * (BN * 32) + (which == 2 ? 512 : 0));
    };
    ST_CONV16_WAIT_VMCNT((STAGES - 1) * LOADS);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int slot = 0; slot < SLOTS; ++slot) read(0, 0, slot);
    int stage = 0;
    // k-tile t, whose fragments are in registers.  Behind the barrier its stage takes the requests of tile t + STAGES, and the
    // next tile's fragments are read: one memory instruction behind an MFMA, never a burst.
    auto iteration = [&](auto buf_tag, int t) {
        constexpr int BUF = decltype(buf_tag)::value;
        const int next = stage + 1 == STAGES ? 0 : stage + 1;
        ST_CONV16_WAIT_VMCNT((STAGES - 2) * LOADS);
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const Where now = ahead;
        ahead = locate(t + STAGES + 1);
#pragma unroll
        for (int slot = 0; slot < SLOTS; ++slot) {
            const int step = slot / 4, tm = slot % 4 / 2, tn = slot % 2;
            acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag[BUF][step * 4 + 1 + tn], frag[BUF][step * 4 + tm * 3], acc[tm][tn], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            read(BUF ^ 1, next, slot);
            if (slot < LOADS) load(stage, slot, now);
            __builtin_amdgcn_sched_barrier(0);
        }
        stage = next;
    };
    int t = 0;
    for (; t + 1 < tiles; t += 2) {
        iteration(std::integral_constant<int, 0>{}, t);
        iteration(std::integral_constant<int, 1>{}, t + 1);
    }
    if (t < tiles) iteration(std::integral_constant<int, 0>{}, t);
    ST_CONV16_WAIT_VMCNT(0);
    __syncthreads();

    // Register 4g + j of lane (li, lh) is channel li, pixel 8g + 4·lh + j of a 32×32 block.
    constexpr int C_STRIDE = BN + 4;
    float *const sums = reinterpret_cast<float *>(lds_bytes) + ks * (BM * C_STRIDE);
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int tn = 0; tn < 2; ++tn)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<float4 *>(&sums[(wm * 64 + tm * 32 + li) * C_STRIDE + wn * 64 + tn * 32 + g * 8 + lh * 4]) =
                    make_float4(acc[tm][tn][4 * g], acc[tm][tn][4 * g + 1], acc[tm][tn][4 * g + 2], acc[tm][tn][4 * g + 3]);
    __syncthreads();
    constexpr int QUADS = BN / 4, ROWS = WAVES * 64 / QUADS;
    const int quad = tid % QUADS, pixel0 = n0 + quad * 4;
    const int image0 = pixel0 / p.spatial;
    const bool together = (p.spatial & 3) == 0;  // four pixels share an image, on aligned addresses
    const size_t off0 = static_cast<size_t>(image0) * s.c_out * p.spatial + (pixel0 - image0 * p.spatial);
    if (pixel0 >= p.pixels) return;
    float *const out32 = p.k_splits > 1 ? p.partial + static_cast<size_t>(split) * s.c_out * p.pixels : p.C32;
    with_epilogue_ops(p.activation, false, [&](auto &&act, auto) {
#pragma unroll 4
        for (int row = tid / QUADS; row < BM; row += ROWS) {
            const int channel = m0 + row;
            if (channel >= s.c_out) break;
            const float *const src = reinterpret_cast<const float *>(lds_bytes) + row * C_STRIDE + quad * 4;
            float4 v = *reinterpret_cast<const float4 *>(src);
#pragma unroll
            for (int k = 1; k < KS; ++k) {
                const float4 q = *reinterpret_cast<const float4 *>(src + k * (BM * C_STRIDE));
                v.x += q.x; v.y += q.y; v.z += q.z; v.w += q.w;
            }
            const float bias = p.bias ? p.bias[channel] : -0.0f;
            const float value[4] = {act(v.x + bias), act(v.y + bias), act(v.z + bias), act(v.w + bias)};
            const size_t channel_off = static_cast<size_t>(channel) * p.spatial;
            if (together) {
                const size_t idx = off0 + channel_off;
                if (out32) *reinterpret_cast<float4 *>(out32 + idx) = make_float4(value[0], value[1], value[2], value[3]);
                if (p.C16) *reinterpret_cast<uint2 *>(p.C16 + idx) = make_uint2(pack_bf16x2_rne(value[0], value[1]), pack_bf16x2_rne(value[2], value[3]));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int pixel = pixel0 + e;
                    if (pixel >= p.pixels) break;
                    const int image = pixel / p.spatial;
                    const size_t idx = static_cast<size_t>(image) * s.c_out * p.spatial + channel_off + (pixel - image * p.spatial);
                    if (out32) out32[idx] = value[e];
                    if (p.C16) p.C16[idx] = f32_to_bf16_rne(value[e]);
                }
            }
        }
    });
}

// out = act(the splits' sums added in order + bias), four values a thread where four share a channel.
template <int VALUES>
__device__ __forceinline__ void conv_bf16_reduce_body(const ConvBf16Args &p, const float *bias, int activation, float *out32, uint16_t *out16)
{
    const size_t count = static_cast<size_t>(p.s.c_out) * p.pixels;
    const size_t idx = (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * VALUES;
    if (idx >= count) return;
    float sum[VALUES] = {};
    for (int k0 = 0; k0 < p.k_splits; k0 += 4) {
        float part[4][VALUES] = {};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (k0 + k >= p.k_splits) continue;
            const float *const src = p.partial + (k0 + k) * count + idx;
            if constexpr (VALUES == 4) {
                const float4 v = *reinterpret_cast<const float4 *>(src);
                part[k][0] = v.x; part[k][1] = v.y; part[k][2] = v.z; part[k][3] = v.w;
            } else {
                part[k][0] = *src;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int e = 0; e < VALUES; ++e) sum[e] += part[k][e];
    }
    const float b = bias ? bias[(idx / p.spatial) % p.s.c_out] : -0.0f;
#pragma unroll
    for (int e = 0; e < VALUES; ++e) sum[e] = apply_activation(sum[e] + b, activation);
    if constexpr (VALUES == 4) {
        if (out32) *reinterpret_cast<float4 *>(out32 + idx) = make_float4(sum[0], sum[1], sum[2], sum[3]);
        if (out16) *reinterpret_cast<uint2 *>(out16 + idx) = make_uint2(pack_bf16x2_rne(sum[0], sum[1]), pack_bf16x2_rne(sum[2], sum[3]));
    } else {
        if (out32) out32[idx] = sum[0];
        if (out16) out16[idx] = f32_to_bf16_rne(sum[0]);
    }
}
__global__ __launch_bounds__(256) void conv_bf16_reduce_kernel(ConvBf16Args p, const float *bias, int activation, float *out32, uint16_t *out16)
{
    conv_bf16_reduce_body<1>(p, bias, activation, out32, out16);
}
__global__ __launch_bounds__(256) void conv_bf16_reduce_vec_kernel(ConvBf16Args p, const float *bias, int activation, float *out32, uint16_t *out16)
{
    conv_bf16_reduce_body<4>(p, bias, activation, out32, out16);
}

__global__ __launch_bounds__(256, 2) void conv_bf16_64x64_kernel(ConvBf16Args p) { conv_bf16_body<1, 1, 4, 5>(p); }
__global__ __launch_bounds__(256, 2) void conv_bf16_128x64_kernel(ConvBf16Args p) { conv_bf16_body<2, 1, 2, 3>(p); }
__global__ __launch_bounds__(256, 2) void conv_bf16_64x128_kernel(ConvBf16Args p) { conv_bf16_body<1, 2, 2, 3>(p); }
__global__ __launch_bounds__(512) void conv_bf16_128x128_kernel(ConvBf16Args p) { conv_bf16_body<2, 2, 2, 4>(p); }
__global__ __launch_bounds__(512) void conv_bf16_256x128_kernel(ConvBf16Args p) { conv_bf16_body<4, 2, 1, 3>(p); }
__global__ __launch_bounds__(512) void conv_bf16_128x256_kernel(ConvBf16Args p) { conv_bf16_body<2, 4, 1, 3>(p); }

// Tiles, and what a launch takes (µs, fitted to 130 layers, every tile timed: half of the estimates within a tenth, the choice
// 1.8 % above the best tile on average): a workgroup alone on its unit, and each workgroup of a unit with the chip full, constant
// and per 64 of k.  The first three leave room for two workgroups on a unit, the others run in rounds of 256.
struct ConvBf16Config {
    void (*kernel)(ConvBf16Args);
    int bm, bn, waves, ks, stages;
    bool two_a_unit;
    double overlap, alone_us, alone_k_us, full_us, full_k_us;

    size_t tiles(const ConvShape &c) const
    {
        const size_t pixels = static_cast<size_t>(c.batch) * c.oh * c.ow;
        return (c.c_out + bm - 1) / bm * ((pixels + bn - 1) / bn);
    }
    size_t lds_bytes() const
    {
        return std::max<size_t>(static_cast<size_t>(stages) * (bm + bn) * 128, static_cast<size_t>(ks) * bm * (bn + 4) * sizeof(float));
    }
    double us(size_t workgroups, size_t k_tiles) const
    {
        const double k = static_cast<double>(k_tiles);
        if (!two_a_unit) return 2.0 + static_cast<double>((workgroups + 255) / 256) * (full_us + k * full_k_us);
        const double alone = alone_us + k * alone_k_us, full = static_cast<double>(workgroups) / 256 * (full_us + k * full_k_us);
        return 2.0 + std::max(alone, full) + overlap * alone * std::min(alone, full) / std::max(alone, full);
    }
};
const ConvBf16Config kConvBf16Configs[] = {
    {conv_bf16_64x64_kernel, 64, 64, 4, 4, 5, true, 0.30, 2.5, 0.120, 2.3, 0.136},
    {conv_bf16_128x64_kernel, 128, 64, 4, 2, 3, true, 0.23, 3.4, 0.178, 3.1, 0.231},
    {conv_bf16_64x128_kernel, 64, 128, 4, 2, 3, true, 0.26, 3.8, 0.178, 3.2, 0.238},
    {conv_bf16_128x128_kernel, 128, 128, 8, 2, 4, false, 0.0, 0.0, 0.0, 5.2, 0.291},
    {conv_bf16_256x128_kernel, 256, 128, 8, 1, 3, false, 0.0, 0.0, 0.0, 6.0, 0.532},
    {conv_bf16_128x256_kernel, 128, 256, 8, 1, 3, false, 0.0, 0.0, 0.0, 7.6, 0.531},
};

struct ConvBf16Plan {
    const ConvBf16Config *config;
    size_t k_splits;
};

// The tile with the least estimated time, and k cut over workgroups where a layer of few pixels has a long k (1 × 512 -> 512 on
// 7×7, 7×7 taps, is 8 tiles of 392 k-tiles): against that stands the pass that adds the pieces.
ConvBf16Plan plan_conv_bf16(const ConvShape &c, size_t k_tiles, bool may_split)
{
    const double outputs = static_cast<double>(c.batch) * c.oh * c.ow * c.c_out;
    ConvBf16Plan best{nullptr, 1};
    double best_us = 0.0;
    for (const ConvBf16Config &config : kConvBf16Configs) {
        const size_t tiles = config.tiles(c);
        for (size_t splits = 1; splits <= 16; splits *= 2) {
            if (splits > 1 && (!may_split || k_tiles / splits < 2 || tiles * splits > 512)) break;
            double us = config.us(tiles * splits, (k_tiles + splits - 1) / splits);
            if (splits > 1) us += 2.0 + 6e-7 * outputs * static_cast<double>(splits + 1);
            if (best.config == nullptr || us < best_us) best = {&config, splits}, best_us = us;
        }
    }
    return best;
}

size_t round_256(size_t bytes) { return (bytes + 255) & ~static_cast<size_t>(255); }

// What the shape alone decides.
void set_geometry(ConvBf16Args &args, const ConvShape &c)
{
    args.s = c;
    // The copy holds the rows and columns the taps reach; of a kernel one row high (or one column wide) only those it is put on.
    args.step_h = c.kh == 1 ? c.stride_h : 1;
    args.step_w = c.kw == 1 ? c.stride_w : 1;
    args.stride_h = c.kh == 1 ? 1 : c.stride_h;
    args.stride_w = c.kw == 1 ? 1 : c.stride_w;
    const size_t hp = static_cast<size_t>(c.oh - 1) * args.stride_h + static_cast<size_t>(c.kh - 1) * c.dil_h + 1;
    const size_t wp = static_cast<size_t>(c.ow - 1) * args.stride_w + static_cast<size_t>(c.kw - 1) * c.dil_w + 1;
    args.padded_w = static_cast<int>(wp);
    args.padded_pixels = static_cast<int>(hp * wp);
    args.channel_chunks = (c.c_in + 7) / 8;
    args.taps = c.kh * c.kw;
    args.chunks = args.channel_chunks * args.taps;
    args.k_tiles = (args.chunks + 7) / 8;
    args.spatial = c.oh * c.ow;
    args.pixels = c.batch * args.spatial;
    args.image_bytes = static_cast<unsigned>(static_cast<size_t>(c.batch) * args.channel_chunks * args.padded_pixels * 16);
    args.weight_bytes = static_cast<unsigned>(static_cast<size_t>(args.chunks) * c.c_out * 16);
}

// How the plan cuts it; the number of workgroups.
size_t set_tiles(ConvBf16Args &args, const ConvBf16Plan &plan)
{
    args.tiles_per_split = static_cast<int>((args.k_tiles + plan.k_splits - 1) / plan.k_splits);
    args.k_splits = (args.k_tiles + args.tiles_per_split - 1) / args.tiles_per_split;
    args.tiles_m = (args.s.c_out + plan.config->bm - 1) / plan.config->bm;
    return plan.config->tiles(args.s) * args.k_splits;
}

bool conv_bf16_block_in_range(const ConvBf16Args &a, const ConvBf16Config &config, size_t grid, size_t block)
{
    const ConvBf16Item item = decode_conv_bf16_block(static_cast<int>(grid), a.k_splits, a.tiles_m, static_cast<int>(block));
    return item.split >= 0 && item.split * static_cast<long long>(a.tiles_per_split) < a.k_tiles && item.split < a.k_splits && item.tile_m >= 0 &&
           item.tile_m < a.tiles_m && item.tile_n >= 0 && item.tile_n * static_cast<long long>(config.bn) < a.pixels;
}

// The check before a launch: the grid is tiles × runs of k-tiles, tiles and runs cover the layer and none of them is empty.
bool conv_bf16_consistent(const ConvBf16Args &a, const ConvBf16Config &config, size_t grid)
{
    if (a.k_splits < 1 || a.tiles_per_split < 1 || a.tiles_m < 1 || grid == 0 || grid > 0x7fffffffu) return false;
    const size_t tiles_n = (static_cast<size_t>(a.pixels) + config.bn - 1) / config.bn;
    if (grid != static_cast<size_t>(a.tiles_m) * tiles_n * a.k_splits) return false;
    const long long rows = static_cast<long long>(a.tiles_m) * config.bm, k = static_cast<long long>(a.k_splits) * a.tiles_per_split;
    if (rows < a.s.c_out || rows - config.bm >= a.s.c_out || k < a.k_tiles || k - a.tiles_per_split >= a.k_tiles) return false;
    return conv_bf16_block_in_range(a, config, grid, 0) && conv_bf16_block_in_range(a, config, grid, grid - 1);
}

}  // namespace

bool conv2d_bf16_supported(const ConvShape &c)
{
    if (c.batch <= 0 || c.c_out <= 0 || c.oh <= 0 || c.ow <= 0) return true;  // nothing to compute
    // 32-bit byte offsets into both copies (counted with the channels in blocks of 64), 32-bit pixel and tile counts
    const size_t c_pad = (static_cast<size_t>(c.c_in) + 63) / 64 * 64;
    const size_t hp = static_cast<size_t>(c.h) + 2 * c.pad_h, wp = static_cast<size_t>(c.w) + 2 * c.pad_w;
    const size_t image_bytes = static_cast<size_t>(c.batch) * hp * wp * c_pad * 2;
    const size_t k = static_cast<size_t>(c.kh) * c.kw * c_pad;
    const size_t pixels = static_cast<size_t>(c.batch) * c.oh * c.ow;
    return image_bytes < (1ull << 31) && static_cast<size_t>(c.c_out) * k * 2 < (1ull << 31) && pixels < (1ull << 31) &&
           k < (1ull << 31);
}

hipError_t launch_conv2d_bf16(const ConvShape &c, int activation, const uint16_t *input, const uint16_t *weight, const float *bias,
                              float *out_f32, uint16_t *out_bf16, hipStream_t stream)
{
    if (c.batch <= 0 || c.c_out <= 0 || c.oh <= 0 || c.ow <= 0) return hipSuccess;
    if (!conv2d_bf16_supported(c)) return hipErrorInvalidValue;
    ConvBf16Args args{};
    set_geometry(args, c);
    args.input = input;
    args.weight = weight;
    args.whole_chunks = c.c_in % 8 == 0 && args.taps <= kTapsPerPass && (reinterpret_cast<uintptr_t>(weight) & 15u) == 0;
    const size_t outputs = static_cast<size_t>(args.pixels) * c.c_out;

    ConvBf16Plan plan = plan_conv_bf16(c, static_cast<size_t>(args.k_tiles), true);
    args.offsets = (args.k_tiles + kMostStages + 1) * 8;
    const size_t weights_at = round_256(args.image_bytes), offsets_at = weights_at + round_256(args.weight_bytes);
    const size_t partial_at = offsets_at + round_256(args.offsets * sizeof(unsigned));
    void *scratch = nullptr;
    hipError_t rc = stream_workspace(stream, partial_at + (plan.k_splits > 1 ? plan.k_splits * outputs * sizeof(float) : 0), &scratch);
    if (plan.k_splits > 1 && scratch_unavailable(rc)) {
        plan = plan_conv_bf16(c, static_cast<size_t>(args.k_tiles), false);
        rc = stream_workspace(stream, partial_at, &scratch);
    }
    if (rc != hipSuccess) return rc;
    const ConvBf16Config &config = *plan.config;
    unsigned char *const base = static_cast<unsigned char *>(scratch);
    args.images = reinterpret_cast<uint16_t *>(base);
    args.weights = reinterpret_cast<uint16_t *>(base + weights_at);
    args.image_offsets = reinterpret_cast<unsigned *>(base + offsets_at);
    args.partial = reinterpret_cast<float *>(base + partial_at);
    const size_t workgroups = set_tiles(args, plan);
    if (!conv_bf16_consistent(args, config, workgroups)) return hipErrorInvalidConfiguration;
    const bool split = args.k_splits > 1;
    args.bias = split ? nullptr : bias;
    args.C32 = split ? nullptr : out_f32;
    args.C16 = split ? nullptr : out_bf16;
    args.activation = split ? ST_HIP_ACT_NONE : activation;
    const size_t groups_px = (static_cast<size_t>(args.padded_pixels) + 255) / 256, image_groups = static_cast<size_t>(c.batch) * args.channel_chunks * groups_px;
    const size_t weight_groups = static_cast<size_t>(args.channel_chunks) * ((c.c_out + 15) / 16);
    if (image_groups + weight_groups + 1 > 0x7fffffffu) return hipErrorInvalidConfiguration;
    args.groups_px = static_cast<unsigned>(groups_px);
    args.image_groups = static_cast<unsigned>(image_groups);
    args.weight_groups = static_cast<unsigned>(weight_groups);

    hipLaunchKernelGGL(conv_bf16_chunks_kernel, dim3(static_cast<unsigned>(image_groups + weight_groups + 1)), dim3(256), 0, stream, args);
    rc = hipGetLastError();
    if (rc != hipSuccess) return rc;
    if (config.lds_bytes() > 64 * 1024) {  // more than a launch may take unasked
        rc = hipFuncSetAttribute(reinterpret_cast<const void *>(config.kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 static_cast<int>(config.lds_bytes()));
        if (rc != hipSuccess) return rc;
    }
    hipLaunchKernelGGL(config.kernel, dim3(static_cast<unsigned>(workgroups)), dim3(static_cast<unsigned>(config.waves) * 64),
                       config.lds_bytes(), stream, args);
    rc = hipGetLastError();
    if (rc != hipSuccess || !split) return rc;
    const bool quads = args.spatial % 4 == 0;
    hipLaunchKernelGGL(quads ? conv_bf16_reduce_vec_kernel : conv_bf16_reduce_kernel,
                       dim3(static_cast<unsigned>((outputs / (quads ? 4 : 1) + 255) / 256)), dim3(256), 0, stream, args, bias, activation, out_f32,
                       out_bf16);
    return hipGetLastError();
}

ConvBf16PlanReport conv2d_bf16_plan_report(const ConvShape &c)
{
    ConvBf16PlanReport report{};
    if (c.batch <= 0 || c.c_out <= 0 || c.oh <= 0 || c.ow <= 0 || !conv2d_bf16_supported(c)) return report;
    ConvBf16Args args{};
    set_geometry(args, c);
    const ConvBf16Plan plan = plan_conv_bf16(c, static_cast<size_t>(args.k_tiles), true);
    const size_t grid = set_tiles(args, plan);
    report.tile_channels = plan.config->bm;
    report.tile_pixels = plan.config->bn;
    report.k_splits = args.k_splits;
    report.k_tiles_per_split = args.tiles_per_split;
    report.consistent = conv_bf16_consistent(args, *plan.config, grid) ? 1 : 0;
    report.workgroups = grid;
    if (grid > (1u << 24)) return report;  // the walk is for tests
    std::vector<unsigned char> seen(grid, 0);
    for (size_t block = 0; block < grid; ++block) {
        if (!conv_bf16_block_in_range(args, *plan.config, grid, block)) {
            ++report.out_of_range;
            continue;
        }
        const ConvBf16Item item = decode_conv_bf16_block(static_cast<int>(grid), args.k_splits, args.tiles_m, static_cast<int>(block));
        unsigned char &cell = seen[(static_cast<size_t>(item.tile_n) * args.tiles_m + item.tile_m) * args.k_splits + item.split];
        if (cell) ++report.duplicates; else ++report.items;
        cell = 1;
    }
    return report;
}

}  // namespace sthip
