// The main loop of products of f32 operands held as three exact bf16 pieces (hi, mid, lo), shared by the f32 GEMM and the
// f32 convolution: see gemm_f32_split.hip for the arithmetic and its error.
#pragma once

#include <type_traits>

#include "device_math.h"

namespace sthip {

#define ST_SPLIT_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (7 << 4) | (15 << 8) | ((((n) >> 4) & 3) << 14))
#define ST_SPLIT_FENCE() __builtin_amdgcn_sched_barrier(0)

// The largest magnitude among eight values and `so_far`, as f32 bits (ordered like the magnitudes, infinities and NaN above
// everything else), and over a wavefront.
__device__ __forceinline__ unsigned split_top(const float (&x)[8], unsigned so_far)
{
#pragma unroll
    for (int e = 0; e < 8; ++e) so_far = max(so_far, __float_as_uint(x[e]) & 0x7fffffffu);
    return so_far;
}
__device__ __forceinline__ unsigned wave_top(unsigned top)
{
#pragma unroll
    for (int mask = 32; mask > 0; mask >>= 1) top = max(top, static_cast<unsigned>(__shfl_xor(static_cast<int>(top), mask)));
    return top;
}

// Operands are scaled by 2^24 before they are split, and sums by 2^-48 behind the products: the last bit any f32 value can
// have, 2^-149, is then a normal bf16 number, and the three pieces are exact for every value, however small.
constexpr int kSplitScaleBits = 24;
constexpr float kSplitScale = 0x1p24f, kSplitUnscale = 0x1p-48f;

// Whether the piece products can stand for sums of `terms` products of values up to `top_a` and `top_b`: finite values below
// 2^127 when scaled, and no partial sum that could pass 2^127.  (Where one overflows, mid·hi overflows as well, with the
// sign of the mid piece, and Inf - Inf comes out where f32 sums give an infinity.)
__device__ __forceinline__ bool split_in_range(unsigned top_a, unsigned top_b, int terms)
{
    const int a = static_cast<int>(top_a >> 23), b = static_cast<int>(top_b >> 23);  // values below 2^(a - 126)
    return max(a, b) <= 253 - kSplitScaleBits && a + b - 252 + 2 * kSplitScaleBits + (32 - __clz(terms)) <= 127;
}

// 2^24·x = hi + mid + lo for eight values, packed in pairs: piece[0] hi, [1] mid, [2] lo.
__device__ __forceinline__ void split_pieces(const float (&x)[8], uint32_t (&piece)[3][4])
{
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float a = x[2 * e] * kSplitScale, b = x[2 * e + 1] * kSplitScale;
        piece[0][e] = pack_bf16x2_rne(a, b);
        const float ra = a - __uint_as_float(piece[0][e] << 16), rb = b - __uint_as_float(piece[0][e] & 0xffff0000u);
        piece[1][e] = pack_bf16x2_rne(ra, rb);
        const float la = ra - __uint_as_float(piece[1][e] << 16), lb = rb - __uint_as_float(piece[1][e] & 0xffff0000u);
        piece[2][e] = pack_bf16x2_rne(la, lb);
    }
}

// A tile's operands go through LDS in stages of one 16-term step: (BM + BN) / 32 blocks of three 1 KB fragments, A's
// first.  Piece q of a stage is fragment q % 3 of block q / 3; wavefront w loads pieces w·LOADS .. + LOADS - 1.
template <int BM, int BN, int WM, int WN, int STAGES>
struct SplitTile {
    static constexpr int WAVES = WM * WN, WTM = BM / WM, WTN = BN / WN, TM = WTM / 32, TN = WTN / 32;
    static constexpr int PIECES = (BM + BN) / 32 * 3;
    static constexpr int LOADS = (PIECES + WAVES - 1) / WAVES;
    static constexpr int STAGE = PIECES * 1024;
};

// acc[tm][tn] = the wavefront's sums over `steps` (even) steps, not scaled back.  `locate(t)` is called once for every step in
// order and says where step t's data lies; `load(stage, i, where)` requests this wavefront's i-th piece of it into a stage
// (past the last step too: those loads read nothing that is used).  `check()` runs under the first loads; its result is
// returned.
template <int BM, int BN, int WM, int WN, int STAGES, class Locate, class Load, class Check>
__device__ __forceinline__ bool split_product_loop(unsigned char *lds_bytes, int wave, int lane, int steps,
                                                   f32x16 (&acc)[BM / WM / 32][BN / WN / 32], Locate &&locate, Load &&load,
                                                   Check &&check)
{
    using Tile = SplitTile<BM, BN, WM, WN, STAGES>;
    constexpr int TM = Tile::TM, TN = Tile::TN, LOADS = Tile::LOADS, STAGE = Tile::STAGE;
    constexpr int SLOTS = TM * TN, SPREAD = TM + TN;
    const int wm = wave / WN, wn = wave % WN;
    const unsigned lane_off = lane * 16;

    // hi·hi and the five small products accumulate apart and are added at the end: a small product then never rounds
    // against the large sum, and the result carries one rounding per sixteen terms.
    f32x16 fine[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
            acc[a][b] = fine[a][b] = f32x16{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

    bf16x8 a_hi[TM], a_mid[TM], a_lo[TM], b_hi[2][TN], b_mid[TN], b_lo[TN];
    const unsigned a_frag = wm * TM * 3072 + lane_off, b_frag = (BM / 32 + wn * TN) * 3072 + lane_off;
    auto frag_a = [&](int stage, int t, int plane) {
        return *reinterpret_cast<const bf16x8 *>(lds_bytes + stage * STAGE + a_frag + t * 3072 + plane * 1024);
    };
    auto frag_b = [&](int stage, int t, int plane) {
        return *reinterpret_cast<const bf16x8 *>(lds_bytes + stage * STAGE + b_frag + t * 3072 + plane * 1024);
    };
    // The product is formed transposed (B's fragment first), so register 4g + j of lane (li, lh) is
    // C[32·tm + li][32·tn + 8g + 4·lh + j]: four neighbouring columns of a row.
    auto product = [&](f32x16 (&sum)[TM][TN], const bf16x8 (&a)[TM], const bf16x8 (&b)[TN], auto &&memory) {
#pragma unroll
        for (int slot = 0; slot < SLOTS; ++slot) {
            sum[slot / TN][slot % TN] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[slot % TN], a[slot / TN], sum[slot / TN][slot % TN], 0, 0, 0);
            ST_SPLIT_FENCE();
            memory(slot);
            ST_SPLIT_FENCE();
        }
    };

    // Step t (16 terms).  On entry the fragments lo and mid of A and hi and mid of B are in registers; the rest is read
    // during the first product, so that every LDS read of a stage is behind its barrier, after which the stage takes
    // the loads of step t + STAGES.  Behind the barrier come those loads and the next step's fragments, each into
    // registers whose last use is past: one memory instruction behind an MFMA, never a burst.
    int stage = 0;
    auto iteration = [&](auto buf_tag, int t) {
        constexpr int BUF = decltype(buf_tag)::value;
        const int next = stage + 1 == STAGES ? 0 : stage + 1;
        product(fine, a_lo, b_hi[BUF], [&](int slot) {
            if (slot < SPREAD) {
                if (slot < TM) a_hi[slot] = frag_a(stage, slot, 0);
                else b_lo[slot - TM] = frag_b(stage, slot - TM, 2);
            }
            if (SLOTS < SPREAD && slot == SLOTS - 1) {
#pragma unroll
                for (int i = SLOTS; i < SPREAD; ++i) {
                    if (i < TM) a_hi[i] = frag_a(stage, i, 0);
                    else b_lo[i - TM] = frag_b(stage, i - TM, 2);
                }
            }
        });
        product(fine, a_mid, b_hi[BUF], [&](int) {});
        // This wavefront's loads of step t + 1 have landed, and its LDS reads of step t have returned; the barrier extends
        // both to every wavefront.
        ST_SPLIT_WAIT_VMCNT((STAGES - 2) * LOADS);
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        // Past the last step the fragments read are never used: every step runs the same code.
        const auto where = locate(t + STAGES);
        // the memory instructions of the last four products: loads, then A's lo and B's hi, spread over three of them ...
        auto tail = [&](int slot) {
            constexpr int ALL = LOADS + SPREAD, PER = (ALL + 3 * SLOTS - 1) / (3 * SLOTS);
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                const int i = slot * PER + e, r = i - LOADS;
                if (i < LOADS) load(stage, i, where);
                else if (r < TM) a_lo[r] = frag_a(next, r, 2);
                else if (r < SPREAD) b_hi[BUF ^ 1][r - TM] = frag_b(next, r - TM, 0);
            }
        };
        product(fine, a_mid, b_mid, [&](int slot) { tail(slot); });
        product(fine, a_hi, b_mid, [&](int slot) { tail(SLOTS + slot); });
        product(fine, a_hi, b_lo, [&](int slot) { tail(2 * SLOTS + slot); });
        // ... and the mid fragments behind the last one that reads them
        product(acc, a_hi, b_hi[BUF], [&](int slot) {
            constexpr int PER = (SPREAD + SLOTS - 1) / SLOTS;
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                const int i = slot * PER + e;
                if (i < TM) a_mid[i] = frag_a(next, i, 1);
                else if (i < SPREAD) b_mid[i - TM] = frag_b(next, i - TM, 1);
            }
        });
        stage = next;
    };

#pragma unroll
    for (int s = 0; s < STAGES; ++s) {
        const auto where = locate(s);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) load(s, i, where);
    }
    const bool bad = check();
    ST_SPLIT_WAIT_VMCNT(0);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        a_lo[i] = frag_a(0, i, 2);
        a_mid[i] = frag_a(0, i, 1);
    }
#pragma unroll
    for (int i = 0; i < TN; ++i) {
        b_hi[0][i] = frag_b(0, i, 0);
        b_mid[i] = frag_b(0, i, 1);
    }
    for (int t = 0; t < steps; t += 2) {
        iteration(std::integral_constant<int, 0>{}, t);
        iteration(std::integral_constant<int, 1>{}, t + 1);
    }

#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] += fine[a][b];
    ST_SPLIT_WAIT_VMCNT(0);  // the loads past the last step have written their stages: the caller may use the LDS behind a barrier
    return bad;
}

}  // namespace sthip
