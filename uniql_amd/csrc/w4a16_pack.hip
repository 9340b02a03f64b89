// Producer side of the packed layout on the device: group-128 quantisation of an fp16 weight
// matrix into int4 codes + fp16 scales, and the packing of codes into the kernel's word order.
// Bit-exact with the host arithmetic of the reference (fp16 tensors on the CPU: every operation rounds its
// fp32 result to fp16).
#include "common.hpp"

namespace uniql {

// fp16 result of an fp16 x fp32-constant product, an fp16 / fp16 quotient and an fp16 + 8 sum,
// each computed in fp32 and rounded once to fp16, as torch does for half tensors on the CPU
__device__ __forceinline__ half_t half_div(half_t a, half_t b) { return (half_t)((float)a / (float)b); }

// Position of column n's scale inside a permuted scale row (group-128 case): inside every 64
// columns, position 8 i + j holds column i + 8 j.
__device__ __forceinline__ int64_t group_scale_pos(int n) { return (n & ~63) + 8 * (n & 7) + ((n & 63) >> 3); }

// code of one weight; `gptq`: the scales were handed over and the reference computes
// round(w / s + 8) (quantize_helpers.py:216-217) instead of round(w / s) + 8 (:114).
// A quotient that is not finite (0/0 in an all-zero group, x/0 when the scale underflowed)
// becomes INT_MIN in the reference's float -> int conversion and so code 0 after the clamp.
__device__ __forceinline__ uint32_t quantize_code(half_t w, half_t s, bool gptq) {
    const half_t q = half_div(w, s);
    float r;
    if (gptq) {
        const half_t shifted = (half_t)((float)q + 8.0f);
        if (!__builtin_isfinite((float)shifted)) return 0u;
        r = __builtin_rintf((float)shifted);
    } else {
        if (!__builtin_isfinite((float)q)) return 0u;
        r = __builtin_rintf((float)q) + 8.0f;
    }
    return (uint32_t)fminf(fmaxf(r, 0.0f), 15.0f);
}

// One workgroup quantises 64 columns (one chunk of the packed layout) x one group of 128 K values in one pass:
// every weight is read once, 32 bytes per column and thread, and stays in registers between the group's
// maximum and its codes.  Thread t takes packed row r = t % 8 of the columns 16 j + c8 and 16 j + 8 + c8
// (c8 = (t / 8) % 8, j = t / 64): their 2 x 16 values are exactly the four words (j of the pieces (c8, kq),
// kq = 0..3) of that row, and the eight threads of a column pair are neighbours, so a group's maximum is three lane
// exchanges.  The words leave through LDS as whole 16-byte pieces.
//
// Bound by memory: 14336 x 4096 (150 MB) takes 32 us = 4.7 TB/s, the rate of a large copy; a kernel for the scales (one wave
// per group, 107 us) and one for the words (each gathering its eight weights, 71 us) took 178.  The quotient decides that: the
// compiler's correctly rounded fp32 division costs ten instructions per weight, more than the memory time, where
// three give the same fp16 quotient.  With w and s of 11 bits and m a midpoint of two fp16 numbers (12 bits),
// w / s differs from m by at least 2^-23 of itself (|w - m s| is at least one unit of a product below 2^23, and never
// zero: an odd 12-bit m times s has more than 11 bits), so every approximation closer than that rounds to the same fp16
// number: the product with a reciprocal refined once, corrected by its own remainder, is within 2^-24 and a bit.
// Columns with a scale or weights outside of what that covers (zero, negative or non-finite scales, non-finite
// weights, quotients that leave fp16) take the plain division.
constexpr int kPackLdsRow = 132;  // words per packed row in LDS: 128 + 4, rows on different banks

// 16 codes (bits 4 lo .. of two words' worth of one column are placed by the caller) of 16 weights w with scale s
template <bool GPTQ>
__device__ __forceinline__ void quantize_sixteen(const h8 (&w)[2], half_t s, bool fast, float rcp, uint32_t (&code)[8]) {
    // code[p]: codes of K values 2 p (low half) and 2 p + 1 (high half)
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        const half_t w0 = w[p >> 2][2 * (p & 3)], w1 = w[p >> 2][2 * (p & 3) + 1];
        if (fast) {
            const float f0 = (float)w0, f1 = (float)w1, sf = (float)s;
            float q0 = f0 * rcp, q1 = f1 * rcp;
            q0 = __builtin_fmaf(__builtin_fmaf(-q0, sf, f0), rcp, q0);
            q1 = __builtin_fmaf(__builtin_fmaf(-q1, sf, f1), rcp, q1);
            h2 q = h2{(half_t)q0, (half_t)q1};
            // clamping first, then adding 1536 (spacing 1: the addition rounds to the nearest integer, ties to even)
            // gives clamp(rint(q) + 8) or, with the scales handed over, clamp(rint(fp16(q + 8))) in the low bits
            if (GPTQ) {
                q = q + h2{(half_t)8.0f, (half_t)8.0f};
                q = __builtin_elementwise_min(__builtin_elementwise_max(q, h2{(half_t)0.0f, (half_t)0.0f}), h2{(half_t)15.0f, (half_t)15.0f});
                q = q + h2{(half_t)1536.0f, (half_t)1536.0f};
            } else {
                q = __builtin_elementwise_min(__builtin_elementwise_max(q, h2{(half_t)-8.0f, (half_t)-8.0f}), h2{(half_t)7.0f, (half_t)7.0f});
                q = q + h2{(half_t)1544.0f, (half_t)1544.0f};
            }
            code[p] = h2_to_bits(q) & 0x000f000fu;
        } else {
            code[p] = quantize_code(w0, s, GPTQ) | (quantize_code(w1, s, GPTQ) << 16);
        }
    }
}

// Quantises and stores one tile; load(n, w) fetches the thread's 16 K values (from 128 g + 16 r on) of column n, zeros
// where there is none.
template <bool GPTQ, class Load>
__device__ __forceinline__ void quantize_tile(const Load& load, uint32_t* words, half_t* scales, const half_t* __restrict__ given,
                                              half_t* __restrict__ S, uint32_t* __restrict__ B, int out_features, int n_pad,
                                              int g, int chunk, bool out_ok) {
    const int tid = threadIdx.x;
    const int r = tid & 7, c8 = (tid >> 3) & 7, j = tid >> 6;
    uint32_t out[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
        const int n = 64 * chunk + 16 * j + 8 * blk + c8;
        h8 w[2];
        load(n, w);
        h2 m = h2{(half_t)0.0f, (half_t)0.0f};
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 8; e += 2) m = __builtin_elementwise_max(m, __builtin_elementwise_abs(h2{w[i][e], w[i][e + 1]}));
        float own = fmaxf((float)m.x, (float)m.y);
        bool finite = true;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const u32x4 bits = __builtin_bit_cast(u32x4, w[i]);
#pragma unroll
            for (int e = 0; e < 4; ++e)  // an exponent of all ones in either half carries into bit 15 of that half
                finite = finite && (((bits[e] & 0x7c007c00u) + 0x04000400u) & 0x80008000u) == 0u;
        }
        half_t s = (half_t)0.0f;
        if (GPTQ) {
            if (n < out_features) s = given[(size_t)g * out_features + n];
        } else {
            float amax = own;
#pragma unroll
            for (int d = 1; d < 8; d <<= 1) amax = fmaxf(amax, __shfl_xor(amax, d, kWave));
            s = scaled_to_half(amax, (float)(2.0 / 15.0));   // fp32 product, then one rounding to fp16
        }
        if (n >= out_features) s = (half_t)0.0f;
        if (r == 0) scales[8 * c8 + 2 * j + blk] = s;
        const float sf = (float)s;
        const bool fast = finite && sf > 0.0f && sf <= 65504.0f && own <= 32768.0f * sf;
        float rcp = __builtin_amdgcn_rcpf(fast ? sf : 1.0f);
        rcp = __builtin_fmaf(__builtin_fmaf(-sf, rcp, 1.0f), rcp, rcp);
        uint32_t code[8];
        if (n < out_features) {
            if (__builtin_expect(fast, 1)) quantize_sixteen<GPTQ>(w, s, true, rcp, code);
            else quantize_sixteen<GPTQ>(w, s, false, rcp, code);
        } else {  // padding columns: code 0 (and scale 0)
#pragma unroll
            for (int p = 0; p < 8; ++p) code[p] = 0u;
        }
        // word kq: K values 2 kq, 2 kq + 1 (code[kq]) at bits 8 blk and 16 + 8 blk, 2 kq + 8, 2 kq + 9 (code[kq + 4]) four bits up
#pragma unroll
        for (int kq = 0; kq < 4; ++kq) out[kq] |= (code[kq] | (code[kq + 4] << 4)) << (8 * blk);
    }
#pragma unroll
    for (int kq = 0; kq < 4; ++kq) words[r * kPackLdsRow + (4 * c8 + kq) * 4 + j] = out[kq];
    __syncthreads();
    // eight packed rows x 512 bytes, 16 bytes per thread; the chunk's 64 scales
    const int row = tid >> 5, piece = tid & 31;
    const u32x4 v = *reinterpret_cast<const u32x4*>(words + row * kPackLdsRow + 4 * piece);
    uint32_t* to = B + (size_t)(8 * g + row) * 2 * n_pad + 128 * (size_t)chunk + 4 * piece;
    half_t* scale_to = S + (size_t)g * n_pad + 64 * (size_t)chunk;
    if (out_ok) {
        *reinterpret_cast<u32x4*>(to) = v;
        if (tid < 8) *reinterpret_cast<u32x4*>(scale_to + 8 * tid) = *reinterpret_cast<const u32x4*>(scales + 8 * tid);
    } else {  // a caller's buffers off the 16-byte grid
#pragma unroll
        for (int i = 0; i < 4; ++i) to[i] = v[i];
        if (tid < 64) scale_to[tid] = scales[tid];
    }
}

template <bool GPTQ>
__global__ __launch_bounds__(256) void w4a16_quantize_kernel(const half_t* __restrict__ W, int64_t ldw, int vec_ok,
                                                            const half_t* __restrict__ given, half_t* __restrict__ S,
                                                            uint32_t* __restrict__ B, int out_features, int in_features,
                                                            int n_pad, int groups, int out_ok) {
    __shared__ __attribute__((aligned(16))) uint32_t words[8 * kPackLdsRow];
    __shared__ __attribute__((aligned(16))) half_t scales[64];
    const int g = blockIdx.x % groups, chunk = blockIdx.x / groups;  // neighbours read on along the same rows
    const int k0 = 128 * g + 16 * (threadIdx.x & 7);
    const auto load = [&](int n, h8 (&w)[2]) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const half_t* src = W + (size_t)n * ldw + k0 + 8 * i;
            if (n < out_features && k0 + 8 * i + 8 <= in_features && vec_ok) {
                w[i] = *reinterpret_cast<const h8*>(src);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) w[i][e] = n < out_features && k0 + 8 * i + e < in_features ? src[e] : (half_t)0.0f;
            }
        }
    };
    quantize_tile<GPTQ>(load, words, scales, given, S, B, out_features, n_pad, g, chunk, out_ok != 0);
}

// Keeps rows of a packed matrix that no longer line up with the groups, and quantises them again: what dequantising, gathering
// the rows, transposing and the kernel above give, without the fp16 matrix and its two copies.  Kept row i is row
// (i / kept) full + i % kept.  One workgroup takes 64 columns x one group of the
// OUTPUT: tasks of kept rows x eight columns (one 16-byte piece holds them; neighbouring rows read the same
// pieces, from the first-level cache) expand into LDS, from where every thread takes its 2 x 16 values.
// Bound by vector instructions.  PAIRED: runs of an even number of rows, an even distance apart, so that kept rows 2 p and 2 p + 1
// are the two halves of the same words: a task is two rows, expanded in packed arithmetic (the same values: code - 8 is
// exact, one rounding), and the division by `kept` is a product with its rounded inverse.
// Out of cache, one row a task -> this: 4096 x 4096, 32 heads of 128 cut to 108 rows, 13.0 -> 10.2 us; 8192 x 4096, 128 of 64
// to 48, 19.4 -> 15.3; 14336 x 4096, one run of 14000, 39.5 -> 29.7.
constexpr int kCutLdsRow = 136;  // fp16 values per column in LDS: 128 + 8, 16-byte reads of eight columns on different banks

template <bool PAIRED>
__global__ __launch_bounds__(256) void w4a16_cut_rows_kernel(const uint32_t* __restrict__ Bin, const half_t* __restrict__ Sin,
                                                            half_t* __restrict__ S, uint32_t* __restrict__ B, int n, int k_kept,
                                                            int full, int kept, unsigned kept_inverse, int per_column, int vec_ok,
                                                            int n_real, int n_pad, int groups) {
    __shared__ __attribute__((aligned(16))) uint32_t words[8 * kPackLdsRow];
    __shared__ __attribute__((aligned(16))) half_t scales[64];
    __shared__ __attribute__((aligned(16))) half_t values[64 * kCutLdsRow];
    const int g = blockIdx.x % groups, chunk = blockIdx.x / groups;
    const int tid = threadIdx.x, c8 = tid & 7;
    if (PAIRED && 64 * chunk < n_real) {  // n_real <= n: the chunk exists in the source
        NibbleMagic magic;
        magic.init();
        u32x4 q4[2];
        h8 s[2];
        int down[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int i = 128 * g + 64 * t + 2 * (tid >> 3), at = i < k_kept ? i : k_kept - 2;
            const int unit = (int)__umulhi((unsigned)at, kept_inverse), k = unit * full + (at - unit * kept);
            q4[t] = *reinterpret_cast<const u32x4*>(Bin + (size_t)(k >> 4) * 2 * n + 128 * (size_t)chunk + 16 * c8 + 4 * ((k >> 1) & 3));
            s[t] = *reinterpret_cast<const h8*>(Sin + (size_t)(k >> 7) * n + 64 * chunk + 8 * c8);
            down[t] = 4 * ((k >> 3) & 1);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int row = 64 * t + 2 * (tid >> 3);
            const bool real = 128 * g + row < k_kept;
#pragma unroll
            for (int e = 0; e < 8; ++e) {  // column 8 e + c8
                const h2 v = magic.pair_low((q4[t][e >> 1] >> down[t]) >> (8 * (e & 1))) * h2{s[t][e], s[t][e]};
                *reinterpret_cast<uint32_t*>(values + (8 * e + c8) * kCutLdsRow + row) = real ? h2_to_bits(v) : 0u;
            }
        }
    } else if (64 * chunk < n_real) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int row = 32 * t + (tid >> 3), i = 128 * g + row;
            h8 v = {};
            if (i < k_kept) {
                const int k = (i / kept) * full + i % kept;
                const u32x4 q4 = *reinterpret_cast<const u32x4*>(Bin + (size_t)(k >> 4) * 2 * n + 128 * (size_t)chunk + 16 * c8 +
                                                                 4 * ((k >> 1) & 3));
                const int bit = 16 * (k & 1) + 4 * ((k >> 3) & 1);
                const half_t* sp = Sin + (per_column ? 0 : (size_t)(k >> 7) * n);
                h8 s;
                if (!per_column && vec_ok) {
                    s = *reinterpret_cast<const h8*>(sp + 64 * chunk + 8 * c8);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        s[e] = per_column ? sp[single_scale_pos(64 * chunk + 8 * e + c8)] : sp[64 * chunk + 8 * c8 + e];
                }
#pragma unroll
                for (int e = 0; e < 8; ++e)  // column 8 e + c8: word e / 2, bits 8 (e % 2) up
                    v[e] = (half_t)(float)((int)((q4[e >> 1] >> (bit + 8 * (e & 1))) & 15u) - 8);
                v *= s;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) values[(8 * e + c8) * kCutLdsRow + row] = v[e];
        }
    }
    __syncthreads();
    const int r = tid & 7;
    const auto load = [&](int col, h8 (&w)[2]) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            w[i] = col < n_real ? *reinterpret_cast<const h8*>(values + (col & 63) * kCutLdsRow + 16 * r + 8 * i) : h8{};
    };
    quantize_tile<false>(load, words, scales, nullptr, S, B, n_real, n_pad, g, chunk, true);
}

// Keeps columns of a packed matrix, as they are: kept columns are up to five runs of `units` x (`kept` of every `full`
// columns, from `base` on: the first `split`, and the others `skip` columns further on); columns behind them have code 0,
// those from n_scaled on scale 0; rows from k_real on get code 0.  A column's four codes of a word are two of its bytes,
// so nothing is unpacked: a 16-byte piece of the output
// takes eight 4-byte loads and a byte selection each, or, where its 64 columns are one source chunk (a kept prefix),
// one load.  A workgroup resolves its chunk's 64 source columns once and keeps them for `per` groups of 128 rows.
// Bound by memory and, for the small projections, by the launch; so the eight loads are all in flight together (columns
// without a source load, too, and are masked: skipped loads had been waited for one by one), quotients are products with
// rounded inverses, and registers stay within 64 for eight waves a SIMD (with 75 the kept prefix took 15 us).  Out of cache,
// before and now: 4096 x 14336 cut to 12160 (53 MB) 13.4 -> 12.8 us, 112 heads of 128 to 108 22.6 -> 17.0; 4096 x 18688 of
// two runs of 64 to 48 25.8 -> 18.6; 4096 x 4096 to 3456 8.3 -> 7.5; 1024 columns 4.9 -> 4.3.  Requesting the next group's words
// ahead: 19.2, 24.6, 28.8, 10.3 (registers).
struct ColumnRuns {
    int count;
    int base[5], units[5], full[5], kept[5], split[5], skip[5];
    unsigned inverse[5];  // 2^32 / kept, rounded up, where that gives the exact quotients; else 0
};

__global__ __launch_bounds__(256, 8) void w4a16_cut_columns_kernel(const uint32_t* __restrict__ Bin, const half_t* __restrict__ Sin,
                                                               uint32_t* __restrict__ B, half_t* __restrict__ S, int n,
                                                               int groups, int k_real, ColumnRuns runs, int n_scaled, int n_pad,
                                                               int per) {
    __shared__ int source[64];
    __shared__ int whole_chunk;
    const int tid = threadIdx.x;
    const int steps = (groups + per - 1) / per;
    const int chunk = blockIdx.x / steps, g0 = (blockIdx.x % steps) * per;
    if (tid < 64) {
        int i = 64 * chunk + tid, col = -1;
#pragma unroll
        for (int s = 0; s < 5; ++s) {
            if (s < runs.count && col < 0) {
                const int len = runs.units[s] * runs.kept[s];
                if (i < len) {
                    const int unit = runs.inverse[s] ? (int)__umulhi((unsigned)i, runs.inverse[s]) : i / runs.kept[s];
                    const int at = i - unit * runs.kept[s];
                    col = runs.base[s] + unit * runs.full[s] + at + (at >= runs.split[s] ? runs.skip[s] : 0);
                }
                i -= len;
            }
        }
        source[tid] = col;
        const int first = __shfl(col, 0, kWave);
        const bool same = first >= 0 && (first & 63) == 0 && col - tid == first;
        const unsigned long long all = __ballot(same);
        if (tid == 0) whole_chunk = all == ~0ull ? first >> 6 : -1;
    }
    __syncthreads();
    const int piece = tid & 31, row = tid >> 5, c8 = piece >> 2, kq = piece & 3;
    const int from = whole_chunk;
    // columns 8 e + c8: word of a packed row, bits to go down, and what of it counts (nothing where there is no source
    // column: every load is made, since one that is skipped waits for those in front of it)
    unsigned word[8];
    int shift[8], counts = 0;  // counts: bit e
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int col = source[8 * e + c8], real = col < 0 ? 0 : col;
        word[e] = 128 * (real >> 6) + 16 * (real & 7) + 4 * kq + ((real & 63) >> 4);
        shift[e] = 8 * ((real >> 3) & 1);
        counts |= col < 0 ? 0 : 1 << e;
    }
    int scale_from = 0;
    bool scaled = false;
    if (tid < 64) {  // the scale at position tid of a chunk belongs to column (tid / 8) + 8 (tid % 8)
        const int at = 8 * (tid & 7) + (tid >> 3), col = source[at];
        scaled = col >= 0 && 64 * chunk + at < n_scaled;
        scale_from = scaled ? (int)group_scale_pos(col) : 0;
    }
    const int g1 = g0 + per < groups ? g0 + per : groups;
    for (int g = g0; g < g1; ++g) {
        const uint32_t* src = Bin + (size_t)(8 * g + row) * 2 * n;
        half_t sv = (half_t)0.0f;
        if (tid < 64) sv = Sin[(size_t)g * n + scale_from];
        u32x4 v;
        if (from >= 0) {
            v = *reinterpret_cast<const u32x4*>(src + 128 * (size_t)from + 4 * piece);
        } else {
            uint32_t q[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) q[e] = src[word[e]];
#pragma unroll
            for (int e = 0; e < 8; ++e) q[e] = (q[e] >> shift[e]) & 0x00ff00ffu & (uint32_t)__builtin_amdgcn_sbfe(counts, e, 1);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = q[2 * j] | (q[2 * j + 1] << 8);
        }
        const int k0 = 128 * g + 16 * row + 2 * kq;  // K rows k0, k0 + 1 (nibbles 0 and 4 of a 16-bit half's pairs), k0 + 8, k0 + 9
        if (k0 + 9 >= k_real) {
            const uint32_t mask = (k0 < k_real ? 0x00000f0fu : 0u) | (k0 + 1 < k_real ? 0x0f0f0000u : 0u) |
                                  (k0 + 8 < k_real ? 0x0000f0f0u : 0u) | (k0 + 9 < k_real ? 0xf0f00000u : 0u);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] &= mask;
        }
        *reinterpret_cast<u32x4*>(B + (size_t)(8 * g + row) * 2 * n_pad + 128 * (size_t)chunk + 4 * piece) = v;
        if (tid < 64) S[(size_t)g * n_pad + 64 * (size_t)chunk + tid] = scaled ? sv : (half_t)0.0f;
    }
}

// Ready codes[k][n] -> packed words, one thread per 32-bit word.  Word j of piece (c8, kq) of chunk c of packed row r
// holds, in nibble 4 lo + 2 blk + hi, K row 16 r + 2 kq + 8 hi + lo of column 64 c + 16 j + 8 blk + c8.
__global__ __launch_bounds__(256) void w4a16_pack_kernel(const uint8_t* __restrict__ codes, uint32_t* __restrict__ B,
                                                        int out_features, int in_features, int n_pad, int k_pad) {
    const int64_t words_per_row = 2 * (int64_t)n_pad;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)(k_pad >> 4) * words_per_row) return;
    const int r = (int)(idx / words_per_row);
    const int c = (int)(idx % words_per_row);
    const int chunk = c >> 7, piece = (c >> 2) & 31, j = c & 3;
    const int c8 = piece >> 2, kq = piece & 3;
    uint32_t word = 0u;
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
        const int n = 64 * chunk + 16 * j + 8 * blk + c8;
#pragma unroll
        for (int hi = 0; hi < 2; ++hi) {
#pragma unroll
            for (int lo = 0; lo < 2; ++lo) {
                const int k = 16 * r + 2 * kq + 8 * hi + lo;
                uint32_t code = 0u;  // columns past out_features: code 0 (and scale 0)
                if (n < out_features) code = k < in_features ? (uint32_t)(codes[(size_t)k * out_features + n] & 15u) : 8u;
                word |= code << (4 * (4 * lo + 2 * blk + hi));
            }
        }
    }
    B[idx] = word;
}

// natural-order scales [groups][n] -> permuted rows of width n_pad (zeros in the padding)
__global__ __launch_bounds__(256) void w4a16_permute_scales_kernel(const half_t* __restrict__ src,
                                                                  half_t* __restrict__ S, int n, int n_pad,
                                                                  int groups) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)groups * n_pad) return;
    const int g = (int)(idx / n_pad), col = (int)(idx % n_pad);
    S[(size_t)g * n_pad + group_scale_pos(col)] = col < n ? src[(size_t)g * n + col] : (half_t)0.0f;
}

int quantize_launch(const void* W, int64_t ldw, const void* given_scales, void* B, void* S, int out_features,
                    int in_features, int n_pad, int k_pad, hipStream_t stream) {
    const int groups = k_pad / 128;
    const int64_t grid = (int64_t)groups * (n_pad / 64);
    if (grid > 0x7fffffffLL) return UNIQL_E_SHAPE;
    const int vec_ok = ldw % 8 == 0 && (reinterpret_cast<uintptr_t>(W) & 15u) == 0 ? 1 : 0;
    const int out_ok = ((reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(S)) & 15u) == 0 ? 1 : 0;
    auto kern = given_scales ? &w4a16_quantize_kernel<true> : &w4a16_quantize_kernel<false>;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), 0, stream, reinterpret_cast<const half_t*>(W), ldw, vec_ok,
                       reinterpret_cast<const half_t*>(given_scales), reinterpret_cast<half_t*>(S),
                       reinterpret_cast<uint32_t*>(B), out_features, in_features, n_pad, groups, out_ok);
    return hipGetLastError() == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
}

int pack_launch(const uint8_t* codes, const void* scales, void* B, void* S, int n, int k, int n_pad, int k_pad,
                hipStream_t stream) {
    const int groups = k_pad / 128;
    const int64_t sc = (int64_t)groups * n_pad;
    hipLaunchKernelGGL(w4a16_permute_scales_kernel, dim3((unsigned)((sc + 255) / 256)), dim3(256), 0, stream,
                       reinterpret_cast<const half_t*>(scales), reinterpret_cast<half_t*>(S), n, n_pad, groups);
    const int64_t words = (int64_t)(k_pad / 16) * 2 * n_pad;
    hipLaunchKernelGGL(w4a16_pack_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, stream, codes,
                       reinterpret_cast<uint32_t*>(B), n, k, n_pad, k_pad);
    return hipGetLastError() == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
}

int cut_rows_launch(const void* B, const void* S, int n, int groups_in, int units, int full, int kept, int n_real, void* B_out,
                    void* S_out, int n_pad, hipStream_t stream) {
    const int k_kept = units * kept, groups = (k_kept + 127) / 128;
    const int64_t grid = (int64_t)groups * (n_pad / 64);
    if (grid > 0x7fffffffLL) return UNIQL_E_SHAPE;
    const bool vec_ok = (reinterpret_cast<uintptr_t>(S) & 15u) == 0;
    // floor(i / kept) = floor(i inverse / 2^32) while i times the inverse's rounding, less than kept, stays below 2^32
    const bool paired = kept % 2 == 0 && full % 2 == 0 && groups_in != 1 && vec_ok && (int64_t)k_kept * kept < (1LL << 32);
    const unsigned inverse = paired ? (unsigned)(((1ULL << 32) + kept - 1) / kept) : 0u;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), 0, stream, reinterpret_cast<const uint32_t*>(B),
                           reinterpret_cast<const half_t*>(S), reinterpret_cast<half_t*>(S_out), reinterpret_cast<uint32_t*>(B_out),
                           n, k_kept, full, kept, inverse, groups_in == 1 ? 1 : 0, vec_ok ? 1 : 0, n_real, n_pad, groups);
    };
    if (paired) go(w4a16_cut_rows_kernel<true>);
    else go(w4a16_cut_rows_kernel<false>);
    return hipGetLastError() == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
}

int cut_columns_launch(const void* B, const void* S, int n, int k, int k_real, const int* runs, int n_runs, int n_scaled,
                       void* B_out, void* S_out, int n_pad, hipStream_t stream) {
    ColumnRuns r = {};
    r.count = n_runs;
    for (int i = 0; i < n_runs; ++i) {
        r.base[i] = runs[6 * i];
        r.units[i] = runs[6 * i + 1];
        r.full[i] = runs[6 * i + 2];
        r.kept[i] = runs[6 * i + 3];
        r.split[i] = runs[6 * i + 4];
        r.skip[i] = runs[6 * i + 5];
        const int64_t kept = r.kept[i];
        r.inverse[i] = kept > 1 && r.units[i] * kept * kept < (1LL << 32) ? (unsigned)(((1LL << 32) + kept - 1) / kept) : 0u;
    }
    const int groups = k / 128;
    const int64_t tiles = (int64_t)groups * (n_pad / 64);
    // Four groups per workgroup share the resolved columns once the chip (2048 workgroups at a time) is filled all the same.
    const int per = tiles >= 4 * 2048 ? 4 : 1;
    const int64_t grid = (int64_t)((groups + per - 1) / per) * (n_pad / 64);
    if (grid > 0x7fffffffLL) return UNIQL_E_SHAPE;
    hipLaunchKernelGGL(w4a16_cut_columns_kernel, dim3((unsigned)grid), dim3(256), 0, stream, reinterpret_cast<const uint32_t*>(B),
                       reinterpret_cast<const half_t*>(S), reinterpret_cast<uint32_t*>(B_out), reinterpret_cast<half_t*>(S_out),
                       n, groups, k_real, r, n_scaled, n_pad, per);
    return hipGetLastError() == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
}

}  // namespace uniql
