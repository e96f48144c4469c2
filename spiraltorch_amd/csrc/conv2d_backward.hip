// Conv2d backward on gfx950: gradients with respect to the input, the weight and the bias.
//
// Reference: Conv2d::backward → accumulate_from_grad_matrix, crates/st-nn/src/layers/conv.rs:780-813, with
// G = grad_output re-laid as (batch·OH·OW, C_out) (:750-778):
//   grad_weight = (Gᵀ · patches) · scale        (matmul_lhs_transpose_scaled, :791-795; scale = 1/batch)
//   grad_bias   = column sums of G · scale       (:796-799)
//   grad_input  = col2im(G · W)                  (:803-809, col2im :860-916)
// Neither the patch matrix, nor G, nor the (pixels × C_in·KH·KW) product is materialised here:
//   * grad_input is the adjoint convolution.  For stride 1 it IS a forward convolution of grad_output with the
//     taps flipped and the channel roles swapped (padding dil·(k−1) − pad), so it runs on the forward kernels;
//     other strides take the same implicit GEMM with the adjoint gather.
//   * grad_weight is an implicit GEMM  G_b(C_out × pixels) · patches_b(pixels × C_in·KH·KW)  summed over images:
//     C_out × C_in·KH·KW is small and the reduction long, so the images are split over workgroups, partial tiles
//     go to the stream's workspace and a second kernel adds them in a fixed order (reproducible) and scales.
//   * grad_bias is a per-channel sum over NCHW planes.
#include "device_math.h"
#include "kernels.h"
#include "split_product.h"

#include <algorithm>
#include <cmath>
#include <mutex>

namespace sthip {

// Scratch of the allocation-free grad_input entry point: the flipped, channel-swapped weights live here instead of
// in memory from hipMalloc.  Each GPU the library runs on holds its own copy of the array until the process ends.
// In host code the array's name is only a stand-in for the symbol: its device address on the current GPU comes from
// hipGetSymbolAddress (noalloc_scratch below), and only that pointer is ever passed to a kernel.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
void *scratch_ptr[kMaxDevices] = {};

}  // namespace

// Device address of `scratch` on the current GPU, resolved once per device.
hipError_t noalloc_scratch(void **out)
{
    int device = 0;
    hipError_t rc = hipGetDevice(&device);
    if (rc != hipSuccess) return rc;
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (scratch_ptr[device] == nullptr) {
        void *ptr = nullptr;
        rc = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (rc != hipSuccess) return rc;
        scratch_ptr[device] = ptr;
    }
    *out = scratch_ptr[device];
    return hipSuccess;
}

namespace {

// dst[ic][oc][ky][kx] = src[oc][ic][flip ? KH-1-ky : ky][flip ? KW-1-kx : kx]
__global__ __launch_bounds__(256) void conv_weight_to_adjoint_kernel(int c_out, int c_in, int kh, int kw, int flip,
                                                                     const float *src, float *dst)
{
    const size_t total = static_cast<size_t>(c_out) * c_in * kh * kw;  // (may exceed 2^31 values)
    const size_t i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= total) return;
    const int kx = static_cast<int>(i % kw);
    size_t rest = i / kw;
    const int ky = static_cast<int>(rest % kh);
    rest /= kh;
    const int oc = static_cast<int>(rest % c_out);
    const int ic = static_cast<int>(rest / c_out);
    const int sy = flip ? kh - 1 - ky : ky, sx = flip ? kw - 1 - kx : kx;
    dst[i] = src[((static_cast<size_t>(oc) * c_in + ic) * kh + sy) * kw + sx];
}

// col2im as a gather (crates/st-nn/src/layers/conv.rs:860-916 adds patch gradients into the input gradient patch by
// patch; here every input position collects the entries that land on it, in the same order: output rows ascending,
// then output columns ascending).  cols: [images][OH·OW][C_in·KH·KW], the product grad_outputᵀ · W of each image.
// One thread per input value.
__global__ __launch_bounds__(256) void conv_col2im_gather_kernel(ConvShape s, int images, const float *cols, float *grad_input)
{
    const size_t total = static_cast<size_t>(images) * s.c_in * s.h * s.w;
    const size_t idx = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= total) return;
    const int x = static_cast<int>(idx % s.w);
    size_t rest = idx / s.w;
    const int y = static_cast<int>(rest % s.h);
    rest /= s.h;
    const int ic = static_cast<int>(rest % s.c_in);
    const int image = static_cast<int>(rest / s.c_in);
    const int S = s.c_in * s.kh * s.kw;
    const float *image_cols = cols + static_cast<size_t>(image) * s.oh * s.ow * S + static_cast<size_t>(ic) * s.kh * s.kw;
    // Taps that can reach this position: (y + pad − ky·dil) a non-negative multiple of the stride below OH·stride.
    // Without dilation they are every stride-th ky, so the loop steps over the others (a 16×16 kernel at stride 16 has
    // one candidate per axis, not sixteen).
    const int step_y = s.dil_h == 1 ? s.stride_h : 1, step_x = s.dil_w == 1 ? s.stride_w : 1;
    int ky_last = s.kh - 1, kx_last = s.kw - 1;
    if (s.dil_h == 1) ky_last -= ((ky_last - (y + s.pad_h)) % step_y + step_y) % step_y;
    if (s.dil_w == 1) kx_last -= ((kx_last - (x + s.pad_w)) % step_x + step_x) % step_x;
    float sum = 0.0f;
    for (int ky = ky_last; ky >= 0; ky -= step_y) {  // descending ky = ascending output row
        const int ty = y + s.pad_h - ky * s.dil_h;
        if (ty < 0 || ty % s.stride_h != 0) continue;
        const int oy = ty / s.stride_h;
        if (oy >= s.oh) continue;
        for (int kx = kx_last; kx >= 0; kx -= step_x) {
            const int tx = x + s.pad_w - kx * s.dil_w;
            if (tx < 0 || tx % s.stride_w != 0) continue;
            const int ox = tx / s.stride_w;
            if (ox >= s.ow) continue;
            sum += image_cols[(static_cast<size_t>(oy) * s.ow + ox) * S + ky * s.kw + kx];
        }
    }
    grad_input[idx] = sum;
}

__device__ __forceinline__ float wave_sum64(float v)
{
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) v += __shfl_xor(v, offset);
    return v;
}

// partial[b][oc] = Σ_pixels grad_output[b][oc][pixel]; one wavefront per (b, oc) plane.  A stream over grad_output, bound by
// how much of it is in flight: four loads of 16 bytes a lane, at any 4-byte alignment (32 × 128 planes of 56×56: 17.7 -> 8.9 µs).
__global__ __launch_bounds__(256) void conv_grad_bias_partial_kernel(int planes, int spatial, const float *grad_output,
                                                                     float *partial)
{
    const int lane = threadIdx.x & 63;
    const int plane = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (plane >= planes) return;
    const float *src = grad_output + static_cast<size_t>(plane) * spatial;
    typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    f32x4_a4 sums[4] = {};
    int i = lane * 4;
    for (; i + 772 <= spatial; i += 1024) {
        f32x4_a4 t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) t[u] = *reinterpret_cast<const f32x4_a4 *>(src + i + 256 * u);
#pragma unroll
        for (int u = 0; u < 4; ++u) sums[u] += t[u];
    }
    for (; i + 4 <= spatial; i += 256) sums[0] += *reinterpret_cast<const f32x4_a4 *>(src + i);
    const f32x4_a4 all = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    float sum = (all[0] + all[1]) + (all[2] + all[3]);
    for (int e = i; e < min(i + 4, spatial); ++e) sum += src[e];  // (one lane's, the last quad's)
    sum = wave_sum64(sum);
    if (lane == 0) partial[plane] = sum;
}

// The whole sum of a channel by one workgroup, in one launch: its sixteen wavefronts take the images' planes (planes cut in `parts`
// where the images are fewer than they), and their sums are added in a fixed order.  Bound by what a compute unit reads, and by the
// launch: two launches / this one, µs (a call takes the host about 4.4): 2×128 channels 6×6 6.6 / 4.4, 15×64 40×40 6.7 / 4.5, 32×32 56×56
// 6.7 / 5.4, 32×128 56×56 11.0 / 9.5, 17×512 66×66 24.9 / 23.0.  A wavefront waits for an image before it asks for the next: of many, see
// launch_conv2d_grad_bias_f32.
__global__ __launch_bounds__(1024) void conv_grad_bias_channel_kernel(int batch, int c_out, int spatial, int parts, const float *grad_output,
                                                                      float scale, float *out)
{
    __shared__ float stage[16];
    typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, channel = blockIdx.x;
    const int part_len = ((spatial + parts - 1) / parts + 3) / 4 * 4;
    f32x4_a4 sums[4] = {};
    float rest = 0.0f;
    for (int item = wave; item < batch * parts; item += 16) {
        const int image = item / parts, first = (item - image * parts) * part_len, end = min(first + part_len, spatial);
        const float *src = grad_output + (static_cast<size_t>(image) * c_out + channel) * spatial;
        int i = first + lane * 4;
        for (; i + 772 <= end; i += 1024) {
            f32x4_a4 t[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) t[u] = *reinterpret_cast<const f32x4_a4 *>(src + i + 256 * u);
#pragma unroll
            for (int u = 0; u < 4; ++u) sums[u] += t[u];
        }
        for (; i + 4 <= end; i += 256) {
            // (The sums take turns: many small planes would all go into one.)
            const f32x4_a4 next = sums[0] + *reinterpret_cast<const f32x4_a4 *>(src + i);
            sums[0] = sums[1];
            sums[1] = sums[2];
            sums[2] = sums[3];
            sums[3] = next;
        }
        for (int e = i; e < min(i + 4, end); ++e) rest += src[e];  // (one lane's, the last quad's)
    }
    const f32x4_a4 all = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    const float sum = wave_sum64(((all[0] + all[1]) + (all[2] + all[3])) + rest);
    if (lane == 0) stage[wave] = sum;
    __syncthreads();
    if (threadIdx.x != 0) return;
    float total[16];
#pragma unroll
    for (int w = 0; w < 16; ++w) total[w] = stage[w];
#pragma unroll
    for (int step = 8; step > 0; step >>= 1)
#pragma unroll
        for (int w = 0; w < step; ++w) total[w] += total[w + step];
    out[channel] = total[0] * scale;
}

// out[i] = scale · Σ_c partial[c][i] in a fixed order: 16 outputs per workgroup, sixteen groups of lanes take every
// sixteenth chunk (four loads in flight each) and their partial sums are added through LDS.
__global__ __launch_bounds__(256) void conv_reduce_chunks_kernel(int chunks, size_t count, const float *partial, float scale,
                                                                 float *out)
{
    __shared__ float stage[16][17];
    const int col = threadIdx.x & 15, sub = threadIdx.x >> 4;
    const size_t i = static_cast<size_t>(blockIdx.x) * 16 + col;
    float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (i < count) {
        int c = sub;
        for (; c + 48 < chunks; c += 64) {
            float t[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) t[u] = partial[static_cast<size_t>(c + 16 * u) * count + i];
#pragma unroll
            for (int u = 0; u < 4; ++u) sum[u] += t[u];
        }
        for (; c < chunks; c += 16) sum[0] += partial[static_cast<size_t>(c) * count + i];
    }
    stage[sub][col] = (sum[0] + sum[1]) + (sum[2] + sum[3]);
    __syncthreads();
    if (sub == 0 && i < count) {
        float total = stage[0][col];
#pragma unroll
        for (int k = 1; k < 16; ++k) total += stage[k][col];
        out[i] = total * scale;
    }
}

// The same sum, 128 bits per lane (count a multiple of 4, 16-byte aligned buffers): 128 outputs per workgroup, 32
// lanes side by side read 512 contiguous bytes of a chunk, eight groups of lanes take every eighth chunk (four loads
// in flight each), and the eight partial sums are added through LDS in a fixed order.
__global__ __launch_bounds__(256) void conv_reduce_chunks_vec_kernel(int chunks, size_t count4, const float4 *partial,
                                                                     float scale, float4 *out)
{
    __shared__ float4 stage[8][33];
    const int col = threadIdx.x & 31, sub = threadIdx.x >> 5;
    const size_t i = static_cast<size_t>(blockIdx.x) * 32 + col;
    float4 sum[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) sum[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    auto add = [](float4 &a, const float4 &b) { a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w; };
    if (i < count4) {
        int c = sub;
        for (; c + 24 < chunks; c += 32) {
            float4 t[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) t[u] = partial[static_cast<size_t>(c + 8 * u) * count4 + i];
#pragma unroll
            for (int u = 0; u < 4; ++u) add(sum[u], t[u]);
        }
        for (; c < chunks; c += 8) add(sum[0], partial[static_cast<size_t>(c) * count4 + i]);
    }
    add(sum[0], sum[1]);
    add(sum[2], sum[3]);
    add(sum[0], sum[2]);
    stage[sub][col] = sum[0];
    __syncthreads();
    if (sub == 0 && i < count4) {
        float4 total = stage[0][col];
#pragma unroll
        for (int k = 1; k < 8; ++k) add(total, stage[k][col]);
        out[i] = make_float4(total.x * scale, total.y * scale, total.z * scale, total.w * scale);
    }
}

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));

struct GradWeightArgs {
    const float *input;        // (N, C_in, H, W)
    const float *grad_output;  // (N, C_out, OH, OW)
    float *partial;            // (chunks, C_out, S)
    ConvShape s;
    int S;                     // c_in * kh * kw
    int spatial;               // oh * ow
    int tiles_s;
    int steps_per_chunk;       // 16-pixel steps (numbered image by image) per workgroup
    int workgroups;            // tiles × chunks; the launch grid is this rounded up to a multiple of 8
};

// One workgroup: a (64·TM output channels) × (64·TN reduction columns s) tile of grad_weight, summed over the pixels
// of its images; four wavefronts in a 2×2 arrangement, each owning TM×TN 32×32 accumulators.  The f32 operands are held as
// three exact bf16 pieces (split_product.h), cut here: per 16-pixel step the G tile (pixel-contiguous in NCHW) and the patch
// tile (gathered: a thread owns TN columns s, whose channel/tap offsets are fixed for the whole kernel) are fetched into
// registers two steps ahead, and cut and written to the other LDS stage among the matrix instructions of the step before.
//
// On the f32 matrix instruction the step was bound by it (94 of 150 µs for 32 images, 64 -> 128 channels, 56×56, 3×3); the six
// piece products take 36 µs, and the kernel now 104: one wavefront a SIMD, whose 36 matrix instructions a step cover the 190
// vector instructions of cutting and addressing (written into their gaps: 2.2 instead of 2.7 thousand cycles), and which then
// waits for its first LDS reads behind the barrier.  The whole call, two launches, old / new µs (and the error against float64,
// 3.6e-7 / 2.1e-7 and the like): that layer 158 / 113, 128 -> 128 at 28×28 90 / 63, 256 -> 256 at 14×14 176 / 75, 512 -> 512 at
// 7×7 235 / 106, 8 × 64 -> 64 at 56×56 (the small tile) 39.5 / 31, 4 × 24 -> 96 at 28×28 20 / 14.4, 14 × 64 -> 16 at 46×47 41 / 28.
//
// The big tile (TM = 2, TN = 3: 128 × 192, three of which span a 3×3 layer's 576 columns exactly for 64 input channels)
// cuts 20 values a thread for 36 matrix instructions of a wavefront, 8 for 6 in the small one.
template <int TM, int TN>
constexpr int kGradWeightStages = 2 * 3 * (64 * (TM + TN) * 32 + 256);  // two stages of three pieces (or of f32 rows)

// How a thread gets its four pixels of a row or column: one 16-byte load of the window under them (buffer loads need four-byte
// alignment only), or four loads.
enum class Gather {
    kValues,   // G and patches value by value: a G below four values an image
    kTaps,     // patches value by value
    kWindows,  // patches by windows: no stride, and rows that are a multiple of four pixels or the whole image
    kRows,     // by a window where the four pixels lie in one row, else value by value: no stride
};

template <Gather GATHER, int TM, int TN>
__device__ __forceinline__ void conv_grad_weight_body(const GradWeightArgs &p, unsigned char *lds)
{
    constexpr int BM = 64 * TM, BN = 64 * TN, BK = 16;
    constexpr bool kByWindow = GATHER == Gather::kWindows || GATHER == Gather::kRows;
    // Both tiles are kept pixel-contiguous (row = channel or patch column, 16 pixels + 4 words of padding), so that a
    // lane's four k-values of either operand are one conflict-free 128-bit LDS read.
    constexpr int A_STRIDE = BK + 4, B_STRIDE = BK + 4;
    constexpr int A_STAGE = BM * A_STRIDE, B_STAGE = BN * B_STRIDE;

    // A stage as pieces: [piece][half][row][8 pixels]: a lane's operand is sixteen bytes, those of 32 rows side by side.  (32 bytes
    // a row cost four cycles of bank conflicts a read and twelve a write of the gathered columns.)  The 64 bytes between the halves
    // keep the two that a quad of lanes of the G tile writes on different banks.
    constexpr int A_HALF = BM * 16 + 64, B_HALF = BN * 16 + 64;
    constexpr int A_PIECE = 2 * A_HALF, B_PIECE = 2 * B_HALF, PIECES_STAGE = 3 * (A_PIECE + B_PIECE);
    constexpr int STAGES_BYTES = kGradWeightStages<TM, TN>;
    static_assert(2 * PIECES_STAGE <= STAGES_BYTES && (2 * A_STAGE + 2 * B_STAGE) * 4 <= STAGES_BYTES, "two stages of either kind");
    __shared__ int beyond;

    float *const As = reinterpret_cast<float *>(lds), *const Bs = As + 2 * A_STAGE;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: the pixel bookkeeping below stays off the VALU
    const int wm = wave >> 1, wn = wave & 1;
    const int li = lane & 31, lh = lane >> 5;
    const ConvShape &s = p.s;
    const int H = s.h, W = s.w;

    // Workgroup ids go round-robin over the 8 XCDs; give each XCD a contiguous run of (chunk, tile) pairs so that
    // the tiles that share a chunk's pixels find them in the same L2.
    // (The grid is padded to a multiple of 8; the padding workgroups leave at once.)
    int bid = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (bid >= p.workgroups) return;
    const int tile_s = bid % p.tiles_s;
    bid /= p.tiles_s;
    const int tiles_oc = (s.c_out + BM - 1) / BM;
    const int tile_oc = bid % tiles_oc;
    const int chunk = bid / tiles_oc;
    const int oc0 = tile_oc * BM, s0 = tile_s * BN;

    // This thread's patch columns (lane + 64·j) and their fixed taps.
    const int khw = s.kh * s.kw;
    bool col_valid[TN];
    int dy[TN], dx[TN], tap_offset[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int col = s0 + j * 64 + lane;
        col_valid[j] = col < p.S;
        const int ic = col_valid[j] ? col / khw : 0;
        const int rem = col_valid[j] ? col - ic * khw : 0;
        const int ky = rem / s.kw, kx = rem - ky * s.kw;
        dy[j] = ky * s.dil_h - s.pad_h;
        dx[j] = kx * s.dil_w - s.pad_w;
        tap_offset[j] = kByWindow ? ic * H * W + dy[j] * W + dx[j] : ic * H * W;
        if (kByWindow && !col_valid[j]) dy[j] = -(1 << 30);  // no row of the image
    }
    const int prow0 = wave * 4;  // patch rows prow0 .. prow0+3 of a step: four consecutive pixels, the same for all lanes

    // G tile: a thread loads 4 consecutive pixels of the channel rows a_row + 64·i.
    const int a_row = tid >> 2, a_c4 = (tid & 3) * 4;

    // hi·hi and the five small products accumulate apart: one rounding against the large sum every sixteen terms.
    f32x16 acc[TM][TN], fine[TM][TN];
    const int steps_per_image = (p.spatial + BK - 1) / BK;
    const int first_step = chunk * p.steps_per_chunk;
    const int total_steps = max(0, min(s.batch * steps_per_image, first_step + p.steps_per_chunk) - first_step);

    // (oy, ox) of this wavefront's first pixel of the step being loaded, advanced by 16 pixels per step without
    // divisions.  Memory is addressed through per-image buffer descriptors with 32-bit offsets; anything outside
    // (padding, pixels past the end, channels past C_out) gets an out-of-range offset and reads as zero.
    int load_image, load_step, oy, ox;
    auto start = [&]() {
        load_image = first_step / steps_per_image;
        load_step = first_step - load_image * steps_per_image;
        const int first_pixel = load_step * BK + prow0;
        oy = first_pixel / s.ow;
        ox = first_pixel - oy * s.ow;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = fine[i][j] = f32x16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    };
    const unsigned image_bytes = static_cast<unsigned>(s.c_in) * H * W * 4u;
    const unsigned grad_bytes = static_cast<unsigned>(s.c_out) * p.spatial * 4u;
    constexpr unsigned kOutside = 0x80000000u;
    const int last_window = s.c_in * H * W - 4;
    const unsigned edge_from = max(W - 3, 0);
    const int last_g_window = s.c_out * p.spatial - 4;
    const bool a_valid[2] = {oc0 + a_row < s.c_out, oc0 + a_row + 64 < s.c_out};
    int a_base[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) a_base[i] = (oc0 + a_row + 64 * i) * p.spatial + a_c4;

    // This thread's values of a step.  A window may reach over the left or right border (edge: some lane's does) or over an end
    // of the image, and is then loaded from inside it (clamped: some lane's was moved, by moved floats).  ox: the window's first output
    // column.  pixel: the step's first one in the image.
    struct Raw {
        u32x4_t a[TM], b[TN];
        int pixel, ox, a_moved[TM], moved[TN];
        bool edge, clamped;
    };
    // The offset of the four floats under a lane's window, whether any of them is wanted, and the floats that the load is moved by to
    // stay inside the image (0 but at its two ends).
    auto window = [&](int j, int row, int col, int &off, int &moved) {
        const int at = tap_offset[j] + (row * W + col);
        off = min(max(at, 0), last_window);
        moved = off - at;
        return (static_cast<unsigned>(row + dy[j]) < static_cast<unsigned>(H)) & (static_cast<unsigned>(col + dx[j] + 3) < static_cast<unsigned>(W + 3));
    };
    // No branch and the same number of loads whatever the step is, also behind the last one (descriptors of no bytes): a load
    // that only some paths make has every later wait count for the path without it, and the values of two steps ahead were
    // waited for in each step (1.75 µs a step against 0.5 µs of matrix instructions).
    auto load_global = [&](Raw &raw, bool live) {
        const int p0 = load_step * BK;
        const __amdgpu_buffer_rsrc_t rsrc_g = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(p.grad_output + static_cast<size_t>(load_image) * s.c_out * p.spatial), 0,
            live ? static_cast<int>(grad_bytes) : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t rsrc_x = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(p.input + static_cast<size_t>(load_image) * s.c_in * H * W), 0,
            live ? static_cast<int>(image_bytes) : 0, 0x00020000);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if (GATHER != Gather::kValues) {
                const int at = a_base[i] + p0, off = min(at, last_g_window);
                raw.a_moved[i] = off - at;
                raw.a[i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_g, a_valid[i] ? static_cast<unsigned>(off) * 4u : kOutside, 0, 0);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bool inside = a_valid[i] & (p0 + a_c4 + e < p.spatial);
                    raw.a[i][e] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_g, inside ? static_cast<unsigned>(a_base[i] + p0 + e) * 4u : kOutside, 0, 0);
                }
            }
        }
        raw.pixel = p0;
        // The four pixels are the same for every lane of the wavefront (lanes differ in their taps).
        if (kByWindow) {
            raw.ox = ox;
            raw.edge = raw.clamped = false;
        }
        if (GATHER == Gather::kWindows || (GATHER == Gather::kRows && ox + 3 < s.ow && p0 + prow0 + 3 < p.spatial)) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                int off;
                const bool wanted = window(j, oy, ox, off, raw.moved[j]) & (p0 + prow0 < p.spatial);
                raw.b[j] = __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, wanted ? static_cast<unsigned>(off) * 4u : kOutside, 0, 0);
                raw.edge |= __builtin_amdgcn_ballot_w64(wanted & (static_cast<unsigned>(ox + dx[j]) >= edge_from)) != 0;
                raw.clamped |= __builtin_amdgcn_ballot_w64(wanted & (raw.moved[j] != 0)) != 0;
            }
        } else {
            int py = oy, px = ox;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int sy = GATHER == Gather::kRows ? py : py * s.stride_h, sx = GATHER == Gather::kRows ? px : px * s.stride_w;
                    const int iy = sy + dy[j], ix = sx + dx[j];
                    const bool inside = col_valid[j] & (p0 + prow0 + r < p.spatial) &
                                        (static_cast<unsigned>(iy) < static_cast<unsigned>(H)) &
                                        (static_cast<unsigned>(ix) < static_cast<unsigned>(W));
                    const int at = GATHER == Gather::kRows ? tap_offset[j] + (sy * W + sx) : tap_offset[j] + iy * W + ix;
                    const unsigned off = inside ? static_cast<unsigned>(at) * 4u : kOutside;
                    raw.b[j][r] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_x, off, 0, 0);
                }
                const bool wrap = ++px == s.ow;
                px = wrap ? 0 : px;
                py += wrap ? 1 : 0;
            }
        }
    };
    auto advance = [&]() {  // to the next step, possibly the next image's first
        if (++load_step == steps_per_image) {
            load_step = 0;
            ++load_image;
            oy = prow0 / s.ow;
            ox = prow0 - oy * s.ow;
        } else {
            ox += BK;
            while (ox >= s.ow) {
                ox -= s.ow;
                ++oy;
            }
        }
    };
    // Values in their places where a load was moved, zeros for what lies outside the row of the image or behind the last pixel.
    auto put_back = [](u32x4_t &values, int moved) {
        const u32x4_t got = values;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            unsigned value = got[r];
#pragma unroll
            for (int from = 0; from < 4; ++from) value = from + moved == r ? got[from] : value;
            values[r] = value;
        }
    };
    auto settle = [&](Raw &raw) {
        if (GATHER != Gather::kValues && raw.pixel + BK > p.spatial) {
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                put_back(raw.a[i], raw.a_moved[i]);
#pragma unroll
                for (int r = 0; r < 4; ++r) raw.a[i][r] = raw.pixel + a_c4 + r < p.spatial ? raw.a[i][r] : 0u;
            }
        }
        if (!kByWindow) return;
        if (raw.clamped) {
#pragma unroll
            for (int j = 0; j < TN; ++j) put_back(raw.b[j], raw.moved[j]);
        }
        if (raw.edge) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    raw.b[j][r] = static_cast<unsigned>(raw.ox + dx[j] + r) < static_cast<unsigned>(W) ? raw.b[j][r] : 0u;
        }
    };
    // Four neighbouring pixels of a row in pieces.
    auto split4 = [](unsigned char *dst, int piece_bytes, const u32x4_t &bits) {
        const f32x4 x = __builtin_bit_cast(f32x4, bits);
        uint32_t piece[3][2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float a = x[2 * e] * kSplitScale, b = x[2 * e + 1] * kSplitScale;
            piece[0][e] = pack_bf16x2_rne(a, b);
            const float ra = a - __uint_as_float(piece[0][e] << 16), rb = b - __uint_as_float(piece[0][e] & 0xffff0000u);
            piece[1][e] = pack_bf16x2_rne(ra, rb);
            const float la = ra - __uint_as_float(piece[1][e] << 16), lb = rb - __uint_as_float(piece[1][e] & 0xffff0000u);
            piece[2][e] = pack_bf16x2_rne(la, lb);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint2 *>(dst + i * piece_bytes) = make_uint2(piece[i][0], piece[i][1]);
    };
    auto store_pieces = [&](int stage, const Raw &raw) {
        unsigned char *const as = lds + stage * PIECES_STAGE, *const bs = as + 3 * A_PIECE;
#pragma unroll
        for (int i = 0; i < TM; ++i)
            split4(as + (a_c4 >> 3) * A_HALF + (a_row + 64 * i) * 16 + (a_c4 & 4) * 2, A_PIECE, raw.a[i]);
#pragma unroll
        for (int j = 0; j < TN; ++j) split4(bs + (prow0 >> 3) * B_HALF + (j * 64 + lane) * 16 + (prow0 & 4) * 2, B_PIECE, raw.b[j]);
    };
    // the six piece products, smallest first: (piece of G, piece of the patches)
    auto compute_pieces = [&](int stage, auto &&between) {
        constexpr int kFirst[6] = {2, 0, 1, 1, 0, 0}, kSecond[6] = {0, 2, 1, 0, 1, 0};  // (the first three name all pieces)
        const unsigned char *const as = lds + stage * PIECES_STAGE + (wm * 32 * TM + li) * 16 + lh * A_HALF;
        const unsigned char *const bs = lds + stage * PIECES_STAGE + 3 * A_PIECE + (wn * 32 * TN + li) * 16 + lh * B_HALF;
        bf16x8 fa[TM][3], fb[TN][3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {  // in the order of their first use
#pragma unroll
            for (int j = 0; j < TN; ++j) fb[j][kSecond[q]] = *reinterpret_cast<const bf16x8 *>(bs + kSecond[q] * B_PIECE + j * 512);
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[i][kFirst[q]] = *reinterpret_cast<const bf16x8 *>(as + kFirst[q] * A_PIECE + i * 512);
        }
        between();
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    f32x16 &sum = q < 5 ? fine[i][j] : acc[i][j];
                    sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][kFirst[q]], fb[j][kSecond[q]], sum, 0, 0, 0);
                }
    };
    auto store_lds = [&](int stage, const Raw &raw) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
            *reinterpret_cast<u32x4_t *>(&As[stage * A_STAGE + (a_row + 64 * i) * A_STRIDE + a_c4]) = raw.a[i];
#pragma unroll
        for (int j = 0; j < TN; ++j)
            *reinterpret_cast<u32x4_t *>(&Bs[stage * B_STAGE + (j * 64 + lane) * B_STRIDE + prow0]) = raw.b[j];
    };
    auto compute = [&](int stage, auto &&between) {
        between();
        const float *as = As + stage * A_STAGE;
        const float *bs = Bs + stage * B_STAGE;
#pragma unroll
        for (int kk = 0; kk < BK / 8; ++kk) {
            f32x4 av[TM], bv[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i)
                av[i] = *reinterpret_cast<const f32x4 *>(&as[(wm * 32 * TM + i * 32 + li) * A_STRIDE + kk * 8 + lh * 4]);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                bv[j] = *reinterpret_cast<const f32x4 *>(&bs[(wn * 32 * TN + j * 32 + li) * B_STRIDE + kk * 8 + lh * 4]);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i][t], bv[j][t], acc[i][j], 0, 0, 0);
        }
    };

    // Step t is computed from LDS while the values of step t + 1 wait in registers and those of t + 2 are on their way.
    auto sum_steps = [&](auto &&store, auto &&compute_step) {
        start();
        Raw raw[2];
        load_global(raw[0], total_steps > 0);
        if (total_steps <= 1) {  // nothing to run ahead of (0.4 µs of the smallest layers' 8)
            settle(raw[0]);
            store(0, raw[0]);
            __syncthreads();
            compute_step(0, [] {});
            return;
        }
        advance();
        load_global(raw[1], true);
        advance();
        settle(raw[0]);
        store(0, raw[0]);
        load_global(raw[0], total_steps > 2);
        __syncthreads();
        auto step = [&](int t, Raw &next) {
            compute_step(t & 1, [&] {
                settle(next);
                advance();
                store((t + 1) & 1, next);
                load_global(next, t + 3 < total_steps);
            });
            // The cutting and addressing of the two steps ahead into the gaps between the matrix instructions.  (The small tile has
            // four wavefronts a SIMD for that.)
            if constexpr (TM * TN > 1) {
#pragma unroll
                for (int g = 0; g < 6 * TM * TN; ++g) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
                    __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                }
            }
            __syncthreads();
        };
        // the last step has none to prepare
        int t = 0;
        for (; t + 2 < total_steps; t += 2) {
            step(t, raw[1]);
            step(t + 1, raw[0]);
        }
        if (t + 1 < total_steps) step(t++, raw[1]);
        if (t < total_steps) compute_step(t & 1, [] {});
    };
    if (threadIdx.x == 0) beyond = 0;
    sum_steps(store_pieces, compute_pieces);
    // A value the scaled pieces cannot carry, or a sum that overflows, leaves an infinity or NaN behind, which no later term takes
    // away: the tile is then summed again on the f32 matrix instruction, from the original values.
    bool finite = true;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] += fine[i][j][r];
                finite = finite && fabsf(acc[i][j][r]) < INFINITY;
                acc[i][j][r] *= kSplitUnscale;
            }
    if (!finite) beyond = 1;
    __syncthreads();
    if (beyond) sum_steps(store_lds, compute);

    float *dst = p.partial + static_cast<size_t>(chunk) * s.c_out * p.S;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int out_col = s0 + wn * 32 * TN + j * 32 + li;
        if (out_col >= p.S) continue;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int oc = oc0 + wm * 32 * TM + i * 32 + (r >> 2) * 8 + lh * 4 + (r & 3);
                if (oc < s.c_out) dst[static_cast<size_t>(oc) * p.S + out_col] = acc[i][j][r];
            }
    }
}

template <Gather GATHER>
__global__ __launch_bounds__(256, 4) void conv_grad_weight_kernel(GradWeightArgs p)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char grad_weight_lds[];
    conv_grad_weight_body<GATHER, 1, 1>(p, grad_weight_lds);
}

template <Gather GATHER>
__global__ __launch_bounds__(256, 1) void conv_grad_weight_big_kernel(GradWeightArgs p)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char grad_weight_lds[];
    conv_grad_weight_body<GATHER, 2, 3>(p, grad_weight_lds);
}

}  // namespace

namespace {
// grad_input as a forward problem: grad_output is the image, input positions are the output pixels.  True when the
// forward kernels can run it (stride 1 and a non-negative adjoint padding); `t` is that problem either way, with
// the original stride/padding when the adjoint gather has to run instead.
bool grad_input_as_forward(const ConvShape &shape, ConvShape &t)
{
    const int adj_pad_h = shape.dil_h * (shape.kh - 1) - shape.pad_h;
    const int adj_pad_w = shape.dil_w * (shape.kw - 1) - shape.pad_w;
    const bool as_forward = shape.stride_h == 1 && shape.stride_w == 1 && adj_pad_h >= 0 && adj_pad_w >= 0;
    t = shape;
    t.c_in = shape.c_out;
    t.h = shape.oh;
    t.w = shape.ow;
    t.c_out = shape.c_in;
    t.oh = shape.h;
    t.ow = shape.w;
    if (as_forward) {
        t.pad_h = adj_pad_h;
        t.pad_w = adj_pad_w;
    }
    return as_forward;
}
}  // namespace

namespace {
// Strided (or over-padded) layers: the adjoint gather kernel tests every (channel, tap) for every input position,
// although only one tap in stride_h·stride_w can contribute, and its output-channel tiles hold 64 or 128 input
// channels — the ViT patch embedding (3 channels, 16×16 at stride 16) took 1.3 s that way.  The reference's own route,
// the product grad_outputᵀ·W followed by col2im, does the forward's flops once: per image an f32 GEMM with the
// transposed-A kernel (grad_output of an image is C_out × OH·OW, i.e. k × m), its result gathered into grad_input.
// Images are processed in groups whose products fit kCol2imWorkspaceBytes.  Chosen when the gather's wasted work
// (stride product × channel-tile padding) exceeds a factor of three; the allocation-free entry point keeps the gather.
constexpr size_t kCol2imWorkspaceBytes = 256u << 20;
bool grad_input_by_col2im(const ConvShape &shape)
{
    const double tile = shape.c_in > 64 ? 128.0 : 64.0;
    const double padded = std::ceil(shape.c_in / tile) * tile / shape.c_in;
    const size_t image_cols = static_cast<size_t>(shape.oh) * shape.ow * shape.c_in * shape.kh * shape.kw * sizeof(float);
    return static_cast<double>(shape.stride_h) * shape.stride_w * padded > 3.0 && image_cols <= kCol2imWorkspaceBytes &&
           image_cols > 0;
}
}  // namespace

int planned_conv_grad_input_kernel(const ConvShape &shape)
{
    ConvShape t;
    if (!grad_input_as_forward(shape, t)) return grad_input_by_col2im(shape) ? ST_HIP_CONV_KERNEL_COL2IM : ST_HIP_CONV_KERNEL_ADJOINT;
    return planned_conv_kernel(t, true, true);
}

bool conv2d_split_served(const ConvShape &shape, bool grad_input, ConvShape *computed)
{
    *computed = shape;
    if (grad_input && !grad_input_as_forward(shape, *computed)) return false;
    return conv2d_f32_split_preferred(*computed, true, true, grad_input);
}

hipError_t launch_conv2d_grad_input_f32(const ConvShape &shape, const float *grad_output, const float *weight,
                                        float *grad_input, hipStream_t stream, float *weight_scratch)
{
    if (shape.batch == 0 || shape.c_in == 0 || shape.h == 0 || shape.w == 0) return hipSuccess;
    const size_t weight_count = static_cast<size_t>(shape.c_out) * shape.c_in * shape.kh * shape.kw;
    ConvShape t;
    const bool as_forward = grad_input_as_forward(shape, t);
    hipError_t rc;
    if (as_forward && weight_scratch == nullptr && conv2d_f32_split_preferred(t, true, (reinterpret_cast<uintptr_t>(grad_input) & 15u) == 0, true)) {
        rc = launch_conv2d_f32_split(t, ST_HIP_ACT_NONE, grad_output, weight, true, nullptr, grad_input, stream);
        if (!scratch_unavailable(rc)) return rc;
    }
    if (!as_forward && weight_scratch == nullptr && grad_input_by_col2im(shape)) {
        const size_t m = static_cast<size_t>(shape.oh) * shape.ow, S = static_cast<size_t>(shape.c_in) * shape.kh * shape.kw;
        const size_t image_cols = m * S;
        const size_t group = std::max<size_t>(1, std::min<size_t>(shape.batch, kCol2imWorkspaceBytes / (image_cols * sizeof(float))));
        void *workspace = nullptr;
        rc = stream_workspace(stream, group * image_cols * sizeof(float), &workspace);
        if (rc != hipSuccess) return rc;
        float *cols = static_cast<float *>(workspace);
        const size_t image_in = static_cast<size_t>(shape.c_in) * shape.h * shape.w;
        for (size_t first = 0; first < static_cast<size_t>(shape.batch); first += group) {
            const size_t images = std::min(group, static_cast<size_t>(shape.batch) - first);
            // cols_i (OH·OW × S) = G_iᵀ · W with G_i = grad_output of image i, C_out × OH·OW (k × m), W = C_out × S: one
            // launch for the group's images (a launch per image cost 5 µs each whatever its size).
            rc = launch_gemm_f32_batched(images, m, S, static_cast<size_t>(shape.c_out), true,
                                         grad_output + first * shape.c_out * m, static_cast<size_t>(shape.c_out) * m, weight, cols,
                                         image_cols, stream);
            if (rc != hipSuccess) return rc;
            const size_t total = images * image_in;
            hipLaunchKernelGGL(conv_col2im_gather_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, stream,
                               shape, static_cast<int>(images), cols, grad_input + first * image_in);
            rc = hipGetLastError();
            if (rc != hipSuccess) return rc;
        }
        return hipSuccess;
    }
    if (as_forward && launch_conv2d_strip_adjoint(t, grad_output, weight, grad_input, stream, weight_scratch == nullptr, &rc)) return rc;
    float *adjoint_weight = weight_scratch;  // room for weight_count values, owned by the caller
    // The re-laid weights sit at the front of the stream's scratch buffer; a forward launch that cuts its reduction
    // into slices keeps its partial sums behind them (sized here, so the buffer does not move in between).
    const size_t weight_bytes = (weight_count * sizeof(float) + 255) & ~static_cast<size_t>(255);
    if (adjoint_weight == nullptr) {
        void *workspace = nullptr;
        const size_t behind = as_forward ? conv2d_scratch_bytes(t, true, (reinterpret_cast<uintptr_t>(grad_input) & 15u) == 0) : 0;
        rc = stream_workspace(stream, weight_bytes + behind, &workspace);
        if (rc != hipSuccess) return rc;
        adjoint_weight = static_cast<float *>(workspace);
    }
    hipLaunchKernelGGL(conv_weight_to_adjoint_kernel, dim3(static_cast<unsigned>((weight_count + 255) / 256)), dim3(256), 0,
                       stream, shape.c_out, shape.c_in, shape.kh, shape.kw, as_forward ? 1 : 0, weight, adjoint_weight);
    rc = hipGetLastError();
    if (rc != hipSuccess) return rc;
    if (as_forward)
        return launch_conv2d_f32(t, ST_HIP_ACT_NONE, grad_output, adjoint_weight, nullptr, grad_input, stream,
                                 weight_scratch ? kConvScratchNone : kConvScratchStream, weight_bytes);
    return launch_conv2d_adjoint_f32(t, grad_output, adjoint_weight, grad_input, stream);
}

hipError_t launch_conv2d_grad_bias_f32(const ConvShape &shape, const float *grad_output, float scale, float *grad_bias,
                                       hipStream_t stream)
{
    if (shape.c_out == 0) return hipSuccess;
    const size_t planes = static_cast<size_t>(shape.batch) * shape.c_out;
    const int spatial = shape.oh * shape.ow;
    // One launch or two (two / one, µs).  Many images are a chain in each of a channel's wavefronts, where two launches spread the planes over
    // the chip: 64×64 40×40 7.0 / 8.0, 65×128 28×28 7.7 / 9.3, 112×64 28×28 6.9 / 12.3, 256×64 7×7 6.9 / 9.7, 512×16 7×7 6.8 / 17.0, 2048×64 7×7 34 / 101, 4096×16 4×4
    // 27 / 90; 64×64 28×28 7.3 / 5.9, 112×64 20×20 7.0 / 5.6, 128×64 14×14 7.0 / 5.3.  Channels that give every unit a workgroup, or two, hide that: 256×256 10×10
    // 13.0 / 11.1, 512×256 5×5 23.0 / 26.5, 1024×512 5×5 86 / 67, 2048×512 7×7 169 / 131.  Fewer of many values leave units idle: 32×16 112×112 10.7
    // / 17.3, 48×64 50×50 7.1 / 8.5, 40×64 43×43 6.6 / 8.0, 32×64 61×61 7.3 / 8.5; 32×64 56×56 7.4 / 6.6, 16×64 90×90 9.8 / 8.8, 32×128 56×56 11.1
    // / 9.8.  Planes of less than a quad add up in one sum: the error of 1024×512 1×1 would be 1.6e-7 of the sums (1.0e-7).
    const int images_most = spatial < 4 ? 48 : shape.c_out >= 512 ? shape.batch : shape.c_out >= 256 ? 256 : spatial <= 400 ? 128 : spatial <= 800 ? 64 : 48;
    const bool all = shape.batch <= 16 || shape.c_out >= 256 || (shape.c_out >= 128 && shape.batch <= 32);
    const size_t values_most = all ? 128u << 10 : shape.batch <= 32 ? 104u << 10 : 64u << 10;
    const bool one = planes > 0 && shape.batch <= images_most && static_cast<size_t>(shape.batch) * spatial <= values_most;
    void *workspace = nullptr;
    hipError_t rc = one ? hipSuccess : stream_workspace(stream, (planes ? planes : 1) * sizeof(float), &workspace);
    if (rc != hipSuccess && !(planes > 0 && scratch_unavailable(rc))) return rc;
    if (workspace == nullptr) {  // (the one launch needs no scratch)
        const int parts = shape.batch >= 16 ? 1 : 16 / shape.batch;
        hipLaunchKernelGGL(conv_grad_bias_channel_kernel, dim3(static_cast<unsigned>(shape.c_out)), dim3(1024), 0, stream, shape.batch, shape.c_out, spatial, parts,
                           grad_output, scale, grad_bias);
        return hipGetLastError();
    }
    float *partial = static_cast<float *>(workspace);
    if (planes > 0) {
        hipLaunchKernelGGL(conv_grad_bias_partial_kernel, dim3(static_cast<unsigned>((planes + 3) / 4)), dim3(256), 0, stream,
                           static_cast<int>(planes), spatial, grad_output, partial);
        rc = hipGetLastError();
        if (rc != hipSuccess) return rc;
    }
    hipLaunchKernelGGL(conv_reduce_chunks_kernel, dim3(static_cast<unsigned>((shape.c_out + 15) / 16)), dim3(256), 0, stream,
                       shape.batch, static_cast<size_t>(shape.c_out), partial, scale, grad_bias);
    return hipGetLastError();
}

hipError_t launch_conv2d_grad_weight_f32(const ConvShape &shape, const float *input, const float *grad_output, float scale,
                                         float *grad_weight, hipStream_t stream)
{
    const int S = shape.c_in * shape.kh * shape.kw;
    const size_t count = static_cast<size_t>(shape.c_out) * S;
    if (count == 0) return hipSuccess;
    // One image of the input and of grad_output is addressed through 32-bit byte offsets.
    const size_t image_floats = static_cast<size_t>(shape.c_in) * shape.h * shape.w;
    if (image_floats * 4 >= (1ull << 31) || static_cast<size_t>(shape.c_out) * shape.oh * shape.ow * 4 >= (1ull << 31))
        return hipErrorInvalidValue;
    GradWeightArgs args;
    args.input = input;
    args.grad_output = grad_output;
    args.s = shape;
    args.S = S;
    args.spatial = shape.oh * shape.ow;
    const bool unit = shape.stride_h == 1 && shape.stride_w == 1;
    // A kernel of one tap that reads every pixel: the image is one long row, whose end is its only border.
    const bool one_row = unit && shape.kh == 1 && shape.kw == 1 && shape.pad_h == 0 && shape.pad_w == 0;
    if (one_row) {
        args.s.h = args.s.oh = 1;
        args.s.w = args.s.ow = args.spatial;
    }
    // 128 × 192 tiles when they waste little (every output channel and column a tile covers beyond the matrix is
    // arithmetic thrown away), 64 × 64 tiles otherwise.
    const long long big_cover = static_cast<long long>((shape.c_out + 127) / 128 * 128) * ((S + 191) / 192 * 192);
    // Nor where they have little to sum, or run in rounds of 256 workgroups of which the last is mostly empty (the small ones, four a
    // unit, take a third more time a value).  Big / small, µs, batch × channels, side: 1×64 -> 128, 4, 3×3 11.0 / 7.5; 4×512 -> 256, 4, 3×3
    // 21.3 / 15.5; 16×512 -> 512, 7, 3×3 (64 steps) 65.8 / 80.0.  With a step or less for each of 256 workgroups 20.8 / 14.0 (1×64 -> 512, 18, 3×3
    // and 92 other layers of 17 to 128 steps), with two to four 25 / 20, four to six 28.6 / 24.6, six to ten 32.6 / 29.6, ten to twenty
    // 41 / 42, beyond 69 / 76.  With 268 tiles 2×512 -> 512, 7, 5×5 61 / 49 and 32 images 365 / 289; with 524
    // 2×512 -> 512, 2×7, 7×7 72 / 61 and 32 images of 7 554 / 510.
    const long long steps_per_image = (args.spatial + 15) / 16, total_steps = steps_per_image * shape.batch;
    const long long big_tiles = static_cast<long long>((shape.c_out + 127) / 128) * ((S + 191) / 192);
    const bool full_rounds = big_tiles <= 256 || (big_tiles + 255) / 256 * 256 * 5 <= big_tiles * 6;
    const bool big = big_cover * 10 <= static_cast<long long>(count) * 12 && total_steps > 16 && total_steps * big_tiles >= 6 * 256 &&
                     full_rounds;  // (of 107 channels at least: never kValues)
    const int bm = big ? 128 : 64, bn = big ? 192 : 64;
    args.tiles_s = (S + bn - 1) / bn;
    const int tiles = args.tiles_s * ((shape.c_out + bm - 1) / bm);
    // The reduction (all 16-pixel steps of all images, numbered image by image) is cut into chunks so that the
    // launch is about one round of resident workgroups (four small tiles or one big tile per compute unit).
    const long long slots = big ? 256 : 1024;
    long long chunks = slots / tiles;  // rounded down: one workgroup too many would run as a round of its own
    if (chunks > total_steps) chunks = total_steps;
    if (chunks < 1) chunks = 1;
    args.steps_per_chunk = static_cast<int>(total_steps > 0 ? (total_steps + chunks - 1) / chunks : 1);
    chunks = total_steps > 0 ? (total_steps + args.steps_per_chunk - 1) / args.steps_per_chunk : 1;
    void *workspace = nullptr;
    hipError_t rc = stream_workspace(stream, static_cast<size_t>(chunks) * count * sizeof(float), &workspace);
    if (rc != hipSuccess) return rc;
    args.partial = static_cast<float *>(workspace);
    const size_t workgroups = static_cast<size_t>(tiles) * static_cast<size_t>(chunks);
    if (workgroups > 0x7ffffff0u) return hipErrorInvalidConfiguration;
    args.workgroups = static_cast<int>(workgroups);
    const dim3 grid(static_cast<unsigned>((workgroups + 7) / 8 * 8));
    // Windows need the four pixels of a thread in one output row (of one row, the last ones may lie beyond it: the input's column is then
    // beyond its row as well) and neighbouring columns of the input, and an image that holds one.
    // (Rows of other widths as two windows, the second for the pixels in the next row: 111 instead of 75 µs for 256 -> 256 channels at
    // 14×14, and between 4 % less and 10 % more in the small tile.)
    const bool windows = unit && (one_row || shape.ow % 4 == 0) && image_floats >= 4;
    // In the small tile each four pixels of such layers take a window where they lie in one row, by a branch of the whole wavefront: value by
    // value a wavefront asks for four times as many cache lines.  Value by value / this, over 330 layers: of launches above 50 µs
    // with rows of 40 and more 1 / 0.83 (30×256 -> 64 at 74×74, 3×1, 235 / 168 µs),
    // 20 to 40 1 / 0.86, below 12 level.  In the big tile, one wavefront a SIMD, the branch's waits are not covered.
    const bool rows = unit && !big && !windows && shape.ow > 4 && image_floats >= 4;
    const Gather gather = static_cast<size_t>(shape.c_out) * args.spatial < 4 ? Gather::kValues
                          : windows                                          ? Gather::kWindows
                          : rows                                             ? Gather::kRows
                                                                             : Gather::kTaps;
    auto kernel = gather == Gather::kValues    ? conv_grad_weight_kernel<Gather::kValues>
                  : gather == Gather::kRows    ? conv_grad_weight_kernel<Gather::kRows>
                  : gather == Gather::kWindows ? (big ? conv_grad_weight_big_kernel<Gather::kWindows> : conv_grad_weight_kernel<Gather::kWindows>)
                                               : (big ? conv_grad_weight_big_kernel<Gather::kTaps> : conv_grad_weight_kernel<Gather::kTaps>);
    const size_t lds_bytes = big ? kGradWeightStages<2, 3> : kGradWeightStages<1, 1>;
    static_assert(kGradWeightStages<2, 3> <= 64 * 1024, "what a launch may take unasked");
    hipLaunchKernelGGL(kernel, grid, dim3(256), lds_bytes, stream, args);
    rc = hipGetLastError();
    if (rc != hipSuccess) return rc;
    if (count % 4 == 0 && ((reinterpret_cast<uintptr_t>(args.partial) | reinterpret_cast<uintptr_t>(grad_weight)) & 15u) == 0)
        hipLaunchKernelGGL(conv_reduce_chunks_vec_kernel, dim3(static_cast<unsigned>((count / 4 + 31) / 32)), dim3(256), 0, stream,
                           static_cast<int>(chunks), count / 4, reinterpret_cast<const float4 *>(args.partial), scale,
                           reinterpret_cast<float4 *>(grad_weight));
    else
        hipLaunchKernelGGL(conv_reduce_chunks_kernel, dim3(static_cast<unsigned>((count + 15) / 16)), dim3(256), 0, stream,
                           static_cast<int>(chunks), count, args.partial, scale, grad_weight);
    return hipGetLastError();
}

}  // namespace sthip
