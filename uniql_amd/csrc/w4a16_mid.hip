// W4A16 kernel for 9 to 64 rows (a batch of sequences that advance together, a short prompt):
// D[M,N] = X[M,K] . dequant(B)[K,N].
//
// The weights are streamed as in the kernel for few rows (w4a16_stream.hip): a unit is 128 columns x one group of
// 128 K, a wave loads it with eight 16-byte loads per lane whose registers hold, per word, the codes of two MFMA
// operand columns, expands every weight once to the reference's fp16 value and multiplies it with ALL rows, 16 of them
// per v_mfma_f32_16x16x32_f16.  The weights never touch LDS; X goes through LDS in operand order, each wave its own
// group (the waves of a workgroup split K and meet in LDS at the end), so the loop has no workgroup barrier.
//
// What bounds it: vector instructions.  A SIMD takes one shift, packed multiply-add or MFMA issue every four clocks from
// however many waves (an MFMA occupies two issue slots, its other clocks pass under them; 2 clocks only for plain AND / fp32
// adds), so a unit of 392 of them and 32 MQ MFMAs is 2080 clocks at 32 rows, 2340 at 48, beside 14 clocks for a load and
// 12 for an LDS access that another wave has to fill: hence two waves a SIMD up to 32 rows (226 registers), one with
// the next unit's loads spread over the current one above (360 to 448).  A 32x32x16 form (half the MFMAs) was no faster:
// it multiplies 64 rows where there are 33 to 48, at a lower clock.
//   us, weights out of cache:          17 rows        32 rows        48 rows
//   4096 ->  6144 (tiled -> this)   10.7 ->  7.7   11.0 ->  8.3   12.6 -> 10.6
//   4096 ->  4096                    9.9 ->  7.4   10.1 ->  7.8   10.6 -> 10.2
//   4096 -> 28672                   20.0 -> 16.6   20.8 -> 17.5   27.1 -> 21.6
//  14336 ->  4096                   16.5 -> 11.8   17.2 -> 13.0   19.7 -> 16.3
// and at 16 rows, against the streaming kernel, 9.0 -> 7.1, 8.5 -> 6.8, the third no faster, 12.8 -> 10.7; 64 rows over
// 4096 -> 512 9.6 -> 9.2.
//
// How exact its sums are: the distance from float64 in front of the fp16 rounding is 0.81 to 1.00 x the streaming
// kernel's at 9 to 16 rows, 0.60 to 1.03 x the tiled kernel's above (216 drawn calls, 0.87 on average).  It grows with the
// number of products that enter one accumulator one after another, hence two sets of accumulators (SETS, mid_sets) and
// mid_plan's longest_chain, and sums of waves and workgroups in pairs, up to 16 rows in 64 bits: the streaming kernel adds its
// workgroups' sums as integers.  With one set and the sums added in a row it was up to 1.39 x.
#include <type_traits>

#include "common.hpp"
#include "mid_plan.hpp"

namespace uniql {

constexpr int kMidXStride = 68;    // dwords per staged row of X: 64 + 4
constexpr int kMidRedStride = 132; // floats per row of a partial tile in LDS

struct MidArgs {
    const u32x4* B;
    const half_t* S;
    const half_t* X;
    void* D;
    unsigned long long* accum;  // an arrival count per strip and wave (splits > 1), zero on entry and exit
    void* part;                 // [strip][split] partial tiles (splits > 1), any contents
    int64_t ldx;
    int M, N, G;
    int per_column;
    int upw;           // groups per wave
    int splits;
    int k_valid;       // columns of X that exist (multiple of 8); the rest of K counts as zeros
    unsigned x_bytes;  // bytes from X to the end of its last row
    Epilogue epi;
};

constexpr int kMidNonTemporal = 2;   // cache policy bit nt
constexpr int kMidDeviceScope = 16;  // cache policy bit sc1: as relaxed device-scope loads and stores compile to

// How sums from several waves and workgroups are added.  In pairs of pairs: a term goes through as few roundings as there
// are levels.
struct TreeSums {
    typedef f4 Total;
    template <int N>
    static __device__ __forceinline__ void add(f4& total, f4 (&v)[N]) {
#pragma unroll
        for (int h = 1; h < N; h <<= 1)
#pragma unroll
            for (int i = 0; i + h < N; i += 2 * h) v[i] += v[i + h];
        total += v[0];
    }
    static __device__ __forceinline__ f4 rounded(f4 total) { return total; }
};
// In 64 bits, one rounding at the end.
struct DoubleSums {
    typedef double Total __attribute__((ext_vector_type(4)));
    template <int N>
    static __device__ __forceinline__ void add(Total& total, const f4 (&v)[N]) {
#pragma unroll
        for (int j = 0; j < N; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) total[i] += (double)v[j][i];
    }
    static __device__ __forceinline__ f4 rounded(Total total) { return f4{(float)total[0], (float)total[1], (float)total[2], (float)total[3]}; }
};

template <int MQ, int WAVES>
struct MidLds {
    static constexpr size_t kBytes = (size_t)WAVES * 16 * MQ * kMidRedStride * 4;  // an area per wave
};

// MQ: 16-row tiles (M <= 16 MQ).  SETS: the products of the low and of the high code pairs go to accumulators of their own (2)
// or to the same ones.  EXT: the call uses something beyond the plain product, as in w4a16_stream.hip.
template <int MQ, int WAVES, int SETS, bool EXT>
__global__ __launch_bounds__(64 * WAVES, WAVES / 4) void w4a16_mid_kernel(const MidArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    constexpr int MR = 16 * MQ, XQ = 4 * MQ;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slot = lane & 15;
    const int kq = lane >> 4;
    const int c8 = slot & 7;
    const int strip = blockIdx.x;
    const int split = blockIdx.y;
    const bool gated = EXT && a.epi.gated != 0;  // uniform
    // a strip of nothing but padding columns
    if (EXT && (gated ? 64 : 128) * strip >= a.epi.n_store) return;

    const int N4 = a.N >> 1;
    const int g_begin = (split * WAVES + w) * a.upw;
    const int g_end = (g_begin + a.upw < a.G) ? (g_begin + a.upw) : a.G;
    const uint32_t piece_off = (uint32_t)((slot >> 3) * 32 + 4 * c8 + kq);
    const uint32_t scale_off = (uint32_t)((slot >> 3) * 64 + 8 * c8);
    const u32x4* strip_w = a.B + (size_t)strip * 64;
    const half_t* strip_s = a.S + (size_t)strip * 128;

    // acc[set][mq][jb][v]: row 16 mq + slot, column slot 4 kq + v of column block jb
    typedef typename std::conditional<MQ == 1, DoubleSums, TreeSums>::type Sums;
    f4 acc[SETS][MQ][8];

    // this wave's area: the staged rows of X, at the end its partial tile
    uint32_t* area = lds + (size_t)w * (MR * kMidRedStride);
    // Staged row layout (dwords): the pair of K values 32 rq + 8 i + kq' + 4 c of the group (packed row 4 rq + i, low
    // (c = 0) or high code pairs) at dword 32 rq + 16 c + 4 kq' + i: an operand is one 16-byte read.
    const uint32_t* xread = area + slot * kMidXStride + 4 * kq;
    uint32_t* xwrite = area + kq * kMidXStride + 32 * (slot >> 3) + 16 * (slot & 1) + ((slot & 7) >> 1);
    NibbleMagic magic;
    magic.init();

    struct {
        u32x4 wq[8];
        u32x4 sc;
    } unit;
    u32x4 xv[XQ];
    // A load brings four rows; rows and columns of X that do not exist lie beyond the descriptor and read as zeros.
    const uint32_t x_lane = (uint32_t)kq * (uint32_t)a.ldx * 2u + 16u * (uint32_t)slot, x_step = 8u * (uint32_t)a.ldx;
    // What a unit needs from memory.  Every load goes through a descriptor that covers what exists of its group, and none
    // of them brings anything for the group behind a wave's last one, so that all units run the same loop body: X and the
    // scales by a descriptor of no bytes at scalar offset zero, the packed rows, which have scalar offsets, by a lane offset
    // behind a descriptor of full size.  So no load leaves its descriptor, however the bounds check counts a scalar offset.
    const uint32_t packed_row_bytes = 16u * (uint32_t)N4;
    auto x_of = [&](int g, bool real) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(a.X) + (size_t)128 * g, 0,
                                                 __builtin_amdgcn_readfirstlane(mid_x_records(a.x_bytes, g, real)), 0x00020000);
    };
    auto w_of = [&](int g) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<u32x4*>(strip_w + (size_t)(8 * g) * N4), 0, (unsigned)mid_group_bytes(a.N), 0x00020000);
    };
    auto s_of = [&](int g, bool real) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(strip_s + (size_t)(a.per_column ? 0 : g) * a.N), 0, real ? 256u : 0u, 0x00020000);
    };
    auto load_x = [&](__amdgpu_buffer_rsrc_t rsrc, int g, int i) __attribute__((always_inline)) {
        const bool real = !EXT || 128 * g + 8 * slot < a.k_valid;
        const uint32_t off = x_lane + (uint32_t)i * x_step;
        xv[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, real ? off : kMidNoLoad, 0, 0));
    };
    auto load_row = [&](__amdgpu_buffer_rsrc_t rsrc, int row, bool real) __attribute__((always_inline)) {
        unit.wq[row] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, real ? 16u * piece_off : kMidNoLoad, (uint32_t)row * packed_row_bytes, kMidNonTemporal));
    };
    auto load_scales = [&](__amdgpu_buffer_rsrc_t rsrc) __attribute__((always_inline)) {
        unit.sc = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, 2u * scale_off, 0, 0));
    };
    auto load_unit = [&](int g) __attribute__((always_inline)) {
        const auto xr = x_of(g, true), wr = w_of(g);
#pragma unroll
        for (int i = 0; i < XQ; ++i) load_x(xr, g, i);
        load_scales(s_of(g, true));
#pragma unroll
        for (int row = 0; row < 8; ++row) load_row(wr, row, true);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto fence = [&]() __attribute__((always_inline)) {
        // LDS operations of one wave complete in issue order, and every wave has its own rows
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    auto stage = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XQ; ++i) {
#pragma unroll
            for (int p = 0; p < 4; ++p) xwrite[4 * i * kMidXStride + 4 * p] = xv[i][p];
        }
        fence();
        __builtin_amdgcn_sched_barrier(0);
    };
    u32x4 sc_fixed = u32x4{0u, 0u, 0u, 0u};

    // The sixteen operand pairs of a unit (quad rq of packed rows, column block jb), each expanded while the previous
    // one is multiplied.  The scheduling barriers keep the compiler from expanding further ahead than there are
    // registers for.
    auto multiply = [&](auto&& pairs, auto&& prefetch) __attribute__((always_inline)) {
        h8 xl[MQ], xh[MQ], bl, bh;
        auto expand = [&](int b, h8& low, h8& high) __attribute__((always_inline)) {
            h2 el[4], eh[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) pairs(unit.wq[4 * (b >> 3) + i][(b & 7) >> 1], (b & 7) >> 1, b & 1, el[i], eh[i]);
            low = h8{el[0].x, el[0].y, el[1].x, el[1].y, el[2].x, el[2].y, el[3].x, el[3].y};
            high = h8{eh[0].x, eh[0].y, eh[1].x, eh[1].y, eh[2].x, eh[2].y, eh[3].x, eh[3].y};
        };
        expand(0, bl, bh);
#pragma unroll
        for (int b = 0; b < 16; ++b) {
            const int rq = b >> 3, jb = b & 7;
            if (jb == 0) {
#pragma unroll
                for (int mq = 0; mq < MQ; ++mq) {
                    xl[mq] = __builtin_bit_cast(h8, *reinterpret_cast<const u32x4*>(xread + 16 * mq * kMidXStride + 32 * rq));
                    xh[mq] = __builtin_bit_cast(h8, *reinterpret_cast<const u32x4*>(xread + 16 * mq * kMidXStride + 32 * rq + 16));
                }
            }
            h8 nl = bl, nh = bh;
            prefetch(b);
            if (b < 15) expand(b + 1, nl, nh);
#pragma unroll
            for (int mq = 0; mq < MQ; ++mq) acc[0][mq][jb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bl, xl[mq], acc[0][mq][jb], 0, 0, 0);
#pragma unroll
            for (int mq = 0; mq < MQ; ++mq) acc[SETS - 1][mq][jb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bh, xh[mq], acc[SETS - 1][mq][jb], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 2 * MQ; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                 // one MFMA,
                __builtin_amdgcn_sched_group_barrier(0x002, MQ == 2 ? 5 : (MQ == 3 ? 4 : 3), 0);   // a share of the expansion
            }
            __builtin_amdgcn_sched_barrier(0);
            bl = nl;
            bh = nh;
        }
        fence();  // the next group's staging must not overtake this group's reads
    };

    // One unit against the staged rows.  A code left where it is, everything else masked away, is the fp16 number
    // c 2^-20; with S = s 2^20, fma(c 2^-20, S, -8 s) = fp16_rn((c - 8) s), the reference's weight, for every scale
    // whose S is finite: |s| < 2^-4, zeros and subnormals included.  A unit with a larger scale is left out (its
    // scales and its X count as zeros, since an infinite X times zero would be NaN) and done behind the others.
    bool left_out = false;
    auto too_large = [&](const u32x4& scales) __attribute__((always_inline)) {
        uint32_t large = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) large |= (scales[j] & 0x7fff7fffu) + 0x54005400u;  // a half's top bit: |s| >= 2^-4
        return __builtin_amdgcn_ballot_w64((large & 0x80008000u) != 0) != 0ull;
    };
    auto process = [&](auto&& prefetch) __attribute__((always_inline)) {
        const u32x4 scales = a.per_column ? sc_fixed : unit.sc;
        const bool large = too_large(scales);
        left_out |= large;
        if (__builtin_expect(large, 0)) {  // uniform
#pragma unroll
            for (int i = 0; i < XQ; ++i) {
#pragma unroll
                for (int p = 0; p < 4; ++p) xwrite[4 * i * kMidXStride + 4 * p] = 0u;
            }
            fence();
        }
        h2 s20[4], m8[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const h2 pr = bits_to_h2(large ? 0u : scales[j]);
            s20[j] = pr * h2{(half_t)1024.0f, (half_t)1024.0f} * h2{(half_t)1024.0f, (half_t)1024.0f};
            m8[j] = pr * h2{(half_t)-8.0f, (half_t)-8.0f};
        }
        multiply([&](uint32_t q, int j, int blk, h2& el, h2& eh) __attribute__((always_inline)) {
            const h2 sv = blk ? h2{s20[j].y, s20[j].y} : h2{s20[j].x, s20[j].x};
            const h2 mv = blk ? h2{m8[j].y, m8[j].y} : h2{m8[j].x, m8[j].x};
            const uint32_t low = blk ? (q >> 4) : (q << 4), high = blk ? (q >> 8) : q;
            el = __builtin_elementwise_fma(bits_to_h2(low & magic.mask_high), sv, mv);
            eh = __builtin_elementwise_fma(bits_to_h2(high & magic.mask_high), sv, mv);
        }, prefetch);
    };
    // the same for any scale: code - 8 exactly, then the reference's multiplication
    auto process_any = [&]() __attribute__((always_inline)) {
        const u32x4 scales = a.per_column ? sc_fixed : unit.sc;
        multiply([&](uint32_t q, int j, int blk, h2& el, h2& eh) __attribute__((always_inline)) {
            const h2 pr = bits_to_h2(scales[j]);
            const h2 sv = blk ? h2{pr.y, pr.y} : h2{pr.x, pr.x};
            const uint32_t pq = blk ? (q >> 8) : q;
            el = magic.pair_low(pq) * sv;
            eh = magic.pair_high(pq) * sv;
        }, [](int) {});
    };

    // ---- the waves' partial tiles meet in LDS ---------------------------------------------
    auto red_of = [&](int tile) __attribute__((always_inline)) { return reinterpret_cast<float*>(lds) + tile * (MR * kMidRedStride); };
    auto put = [&](auto&& value) __attribute__((always_inline)) {
        float* red = red_of(w) + slot * kMidRedStride + 64 * (kq >> 1) + 4 * (kq & 1);
#pragma unroll
        for (int mq = 0; mq < MQ; ++mq)
#pragma unroll
            for (int jb = 0; jb < 8; ++jb)
                *reinterpret_cast<f4*>(red + 16 * mq * kMidRedStride + 16 * (jb >> 1) + 8 * (jb & 1)) = value(mq, jb);
    };
    if (g_begin >= g_end) {
        put([](int, int) { return f4{0.f, 0.f, 0.f, 0.f}; });
    } else {
        load_unit(g_begin);
        // Zeros while the first unit is on its way.  (They are hidden from the compiler: it takes a sum that starts as a
        // constant apart into scalars, which then wander between accumulator and vector registers all through the loop.)
        f4 zeros = f4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+v"(zeros));
#pragma unroll
        for (int set = 0; set < SETS; ++set)
#pragma unroll
            for (int mq = 0; mq < MQ; ++mq)
#pragma unroll
                for (int jb = 0; jb < 8; ++jb) acc[set][mq][jb] = zeros;
        if (a.per_column) {  // uniform, rare
            uint32_t t[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const int n0 = strip * 128 + (slot >> 3) * 64 + c8 + 8 * (2 * p), n1 = n0 + 8;
                const uint16_t lo = *reinterpret_cast<const uint16_t*>(a.S + single_scale_pos(n0));
                const uint16_t hi = *reinterpret_cast<const uint16_t*>(a.S + single_scale_pos(n1));
                t[p] = (uint32_t)lo | ((uint32_t)hi << 16);
            }
            sc_fixed = u32x4{t[0], t[1], t[2], t[3]};
        }
        if constexpr (WAVES == 8) {
            // two waves a SIMD: one's loads pass under the other's arithmetic
            stage();
            process([](int) {});
            for (int g = g_begin + 1; g < g_end; ++g) {
                load_unit(g);
                stage();
                process([](int) {});
            }
        } else {
            // One wave a SIMD: the next unit's loads go out while the current one is multiplied, into registers that are
            // free again by then: X from the start, the first four packed rows behind the expansion of the first quad,
            // the rest at the end.
            for (int g = g_begin; g < g_end; ++g) {
                stage();
                const bool more = g + 1 < g_end;
                const auto xr = x_of(g + 1, more), wr = w_of(g + 1), sr = s_of(g + 1, more);
                process([&](int b) __attribute__((always_inline)) {
#pragma unroll
                    for (int i = 2 * b; i < 2 * b + 2; ++i)
                        if (i < XQ) load_x(xr, g + 1, i);
                    if (b == 8) load_scales(sr);
                    if (b >= 9 && b < 13) load_row(wr, b - 9, more);
                });
#pragma unroll
                for (int row = 4; row < 8; ++row) load_row(wr, row, more);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (__builtin_expect(left_out, 0)) {
            for (int g = g_begin; g < g_end; ++g) {
                load_unit(g);
                if (!too_large(a.per_column ? sc_fixed : unit.sc)) continue;
                stage();
                process_any();
            }
        }
        put([&](int mq, int jb) { return SETS == 2 ? acc[0][mq][jb] + acc[SETS - 1][mq][jb] : acc[0][mq][jb]; });
    }
    __syncthreads();
    // four rows are a unit; wave w finishes units w, w + WAVES ..: lane l row l / 16, columns 8 (l % 16) ..
    constexpr int UT = (XQ + WAVES - 1) / WAVES;
    if (4 * w >= a.M) return;
    // the residual of the wave's units, requested in front of the sums
    u32x4 ahead[UT];
    auto request_residual = [&]() __attribute__((always_inline)) {
        if constexpr (EXT) {
            if (!a.epi.residual_vec) return;  // uniform
            const __amdgpu_buffer_rsrc_t rows = residual_rows(a.epi, 0, a.M, 128 * strip);
#pragma unroll
            for (int t = 0; t < UT; ++t) ahead[t] = residual_load(a.epi, rows, 4 * (w + t * WAVES) + kq, 8 * slot);
        }
    };
    if (a.splits == 1) request_residual();
    f4 lo[UT], hi[UT];
#pragma unroll
    for (int t = 0; t < UT; ++t) {
        const int u = w + t * WAVES < XQ ? w + t * WAVES : w;
        const float* src = red_of(0) + (4 * u + kq) * kMidRedStride + 8 * slot;
        f4 l[WAVES], h[WAVES];
#pragma unroll
        for (int ww = 0; ww < WAVES; ++ww) {
            l[ww] = *reinterpret_cast<const f4*>(src + ww * MR * kMidRedStride);
            h[ww] = *reinterpret_cast<const f4*>(src + ww * MR * kMidRedStride + 4);
        }
        typename Sums::Total sum_lo{}, sum_hi{};
        Sums::add(sum_lo, l);
        Sums::add(sum_hi, h);
        lo[t] = Sums::rounded(sum_lo);
        hi[t] = Sums::rounded(sum_hi);
    }
    if (a.splits > 1) {  // uniform
        // K split over workgroups.  Every wave exchanges its own quarter of the rows: it writes its sums to the
        // quarter's slot, waits until the memory side has acknowledged them and counts itself in; the wave that
        // completes the count adds the slots, in an order that does not depend on it.  The accesses and what they rely on are those of the
        // 128-column kernel's exchange (w4a16_tile.hip); no workgroup barrier, since nobody else's stores matter.
        constexpr int kSlotBytes = WAVES * UT * 2048;
        char* tile = reinterpret_cast<char*>(a.part) + (size_t)strip * a.splits * kSlotBytes;
        // (The slot is the descriptor's base and not a scalar offset, as in that kernel: see there.)
        const __amdgpu_buffer_rsrc_t slot_rsrc = __builtin_amdgcn_make_buffer_rsrc(tile + (size_t)split * kSlotBytes, 0, (unsigned)kSlotBytes, 0x00020000);
        const uint32_t mine = (uint32_t)(UT * 2048 * w) + 16u * (uint32_t)lane;
#pragma unroll
        for (int t = 0; t < UT; ++t) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, lo[t]), slot_rsrc, mine + 2048u * t, 0, kMidDeviceScope);
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, hi[t]), slot_rsrc, mine + 2048u * t + 1024u, 0, kMidDeviceScope);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        unsigned long long* count = a.accum + WAVES * (size_t)strip + w;
        int arrived = 0;
        if (lane == 0) arrived = (int)__hip_atomic_fetch_add(count, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        arrived = __builtin_amdgcn_readfirstlane(arrived);
        if (arrived != a.splits - 1) return;
        asm volatile("" ::: "memory");
        if (lane == 0) __hip_atomic_store(count, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        request_residual();
        // Slots are requested up to eight together; those that do not exist lie beyond the descriptor and read as zeros.
        typename Sums::Total total_lo[UT], total_hi[UT];
#pragma unroll
        for (int t = 0; t < UT; ++t) total_lo[t] = total_hi[t] = typename Sums::Total{};
        auto gather = [&](int first, auto batch) __attribute__((always_inline)) {
            constexpr int N = decltype(batch)::value;
            const __amdgpu_buffer_rsrc_t slots = __builtin_amdgcn_make_buffer_rsrc(
                tile + (size_t)first * kSlotBytes, 0, (unsigned)((a.splits - first) * kSlotBytes), 0x00020000);
            f4 v[2 * UT][N];
#pragma unroll
            for (int b = 0; b < N; ++b)
#pragma unroll
                for (int t = 0; t < 2 * UT; ++t)
                    v[t][b] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(slots, mine + (uint32_t)(b * kSlotBytes) + 1024u * t, 0, kMidDeviceScope));
#pragma unroll
            for (int t = 0; t < UT; ++t) {
                Sums::add(total_lo[t], v[2 * t]);
                Sums::add(total_hi[t], v[2 * t + 1]);
            }
        };
        for (int first = 0; first < a.splits; first += 8) {
            const int rest = a.splits - first;  // uniform
            if (rest > 4) gather(first, std::integral_constant<int, 8>{});
            else if (rest > 2) gather(first, std::integral_constant<int, 4>{});
            else gather(first, std::integral_constant<int, 2>{});
        }
#pragma unroll
        for (int t = 0; t < UT; ++t) {
            lo[t] = Sums::rounded(total_lo[t]);
            hi[t] = Sums::rounded(total_hi[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < UT; ++t) {
        const int m = 4 * (w + t * WAVES) + kq;
        if (EXT) {
            if (gated) {
                // the up value of gate columns 8 slot .. (slot < 8) is eight lanes on
                f4 ulo, uhi;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    ulo[i] = __shfl_down(lo[t][i], 8, kWave);
                    uhi[i] = __shfl_down(hi[t][i], 8, kWave);
                }
                if (m < a.M && slot < 8) store_eight_gated(a.epi, a.D, m, 64 * strip + 8 * slot, lo[t], hi[t], ulo, uhi);
            } else if (m < a.M) {
                store_eight<true>(a.epi, a.D, m, 128 * strip + 8 * slot, lo[t], hi[t], ahead[t]);
            }
        } else if (m < a.M) {
            const size_t o = (size_t)m * a.N + 128 * strip + 8 * slot;
            if (a.epi.out_f32) {
                float* d = reinterpret_cast<float*>(a.D) + o;
                *reinterpret_cast<f4*>(d) = lo[t];
                *reinterpret_cast<f4*>(d + 4) = hi[t];
            } else {
                const h2 r0 = h2{(half_t)lo[t][0], (half_t)lo[t][1]}, r1 = h2{(half_t)lo[t][2], (half_t)lo[t][3]};
                const h2 r2 = h2{(half_t)hi[t][0], (half_t)hi[t][1]}, r3 = h2{(half_t)hi[t][2], (half_t)hi[t][3]};
                *reinterpret_cast<u32x4*>(reinterpret_cast<half_t*>(a.D) + o) =
                    u32x4{h2_to_bits(r0), h2_to_bits(r1), h2_to_bits(r2), h2_to_bits(r3)};
            }
        }
    }
}

// ---------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------
template <int MQ, int WAVES, int SETS>
static bool mid_allow_lds_rows() {
    return allow_lds(&w4a16_mid_kernel<MQ, WAVES, SETS, false>, MidLds<MQ, WAVES>::kBytes) &&
           allow_lds(&w4a16_mid_kernel<MQ, WAVES, SETS, true>, MidLds<MQ, WAVES>::kBytes);
}
bool mid_allow_lds() {
    return mid_allow_lds_rows<1, 8, 2>() && mid_allow_lds_rows<2, 8, 2>() && mid_allow_lds_rows<3, 4, 1>() &&
           mid_allow_lds_rows<3, 4, 2>() && mid_allow_lds_rows<4, 4, 1>();
}

template <int MQ, int WAVES, int SETS>
static hipError_t mid_launch_rows(const MidArgs& a, bool ext, hipStream_t stream) {
    const dim3 grid(a.N / 128, a.splits), block(64 * WAVES);
    constexpr size_t shmem = MidLds<MQ, WAVES>::kBytes;
    if (ext) hipLaunchKernelGGL((w4a16_mid_kernel<MQ, WAVES, SETS, true>), grid, block, shmem, stream, a);
    else hipLaunchKernelGGL((w4a16_mid_kernel<MQ, WAVES, SETS, false>), grid, block, shmem, stream, a);
    return hipGetLastError();
}

// Rows, and the 32-bit offsets of the loads: row strides and packed weights as far as the tiled kernels take them, and
// descriptors of X and of a group's packed rows that end in front of kMidNoLoad.
bool mid_shape_ok(int m, int n, int k, int64_t lda) {
    return m >= kMidMinRows && m <= kMidMaxRows && lda < (1LL << 24) && ((int64_t)(m - 1) * lda + k) * 2 < (1LL << 31) &&
           (int64_t)k * n / 2 < (1LL << 32) && mid_group_bytes(n) <= (int64_t)kMidNoLoad;
}

int mid_launch(const void* A, int64_t lda, int k_valid, const void* B, const void* S, void* D, const Epilogue& epi, void* accum,
               void* part, int m, int n, int k, int groups, const MidPlan& plan, hipStream_t stream) {
    if (plan.splits > 1 && (!accum || !part)) return UNIQL_E_WORKSPACE;
    MidArgs a;
    a.B = reinterpret_cast<const u32x4*>(B);
    a.S = reinterpret_cast<const half_t*>(S);
    a.X = reinterpret_cast<const half_t*>(A);
    a.D = D;
    a.accum = reinterpret_cast<unsigned long long*>(accum);
    a.part = part;
    a.ldx = lda;
    a.M = m;
    a.N = n;
    a.G = k / 128;
    a.per_column = (groups == 1) ? 1 : 0;
    a.upw = plan.upw;
    a.splits = plan.splits;
    a.k_valid = k_valid;
    a.x_bytes = (unsigned)(((int64_t)(m - 1) * lda + k_valid) * 2);
    a.epi = epi;
    const bool ext = epi.gated || epi.bias || epi.residual || epi.relu2 || epi.transpose || epi.n_store != n ||
                     epi.ldd != n || k_valid != k || !epi.vec_ok;
    hipError_t e;
    switch (mid_row_tiles(m)) {
        case 1: e = mid_launch_rows<1, 8, 2>(a, ext, stream); break;
        case 2: e = mid_launch_rows<2, 8, 2>(a, ext, stream); break;
        case 3: e = mid_sets(m, plan.upw) == 2 ? mid_launch_rows<3, 4, 2>(a, ext, stream) : mid_launch_rows<3, 4, 1>(a, ext, stream); break;
        default: e = mid_launch_rows<4, 4, 1>(a, ext, stream); break;
    }
    return e == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
}

}  // namespace uniql
