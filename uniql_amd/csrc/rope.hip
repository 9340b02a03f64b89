// Rotary position embedding with per-head gathered frequencies, in place on the projections'
// outputs.  Attention heads pruned to fewer than the original head_dim columns keep, per
// key/value head, the list of the original columns they retained; column j of such a head is
// rotated with the frequency of original column indices[head][j].
//
// One thread rotates up to eight neighbouring column pairs (j, j + d/2) of one head of one token
// with 16-byte loads and stores (4- or 2-byte ones when the head width does not allow more),
// consecutive lanes on consecutive columns.  Every value is read once and written once; cos /
// sin rows are shared by all heads of a token and stay in cache.
//
// Arithmetic: out = x * cos_g + rotate_half(x) * sin_g with both products and the sum rounded to
// fp16 one after the other, which is what the tensor expression of the reference computes on
// fp16 tensors.
#include "common.hpp"

namespace uniql {

struct RopeArgs {
    half_t* q;
    half_t* k;
    const half_t* cos;
    const half_t* sin;
    const void* indices;  // [n_kh][hd], index_bytes wide
    int64_t q_row_stride, k_row_stride, cos_row_stride;
    int seq_len, cos_batch, n_qh, n_kh, hd, index_bytes;
    unsigned rows;
    int per_head, group;                       // work items of a head, query heads of a key / value head
    unsigned per_head_inverse, group_inverse;  // 2^32 / divisor, rounded up: quotients without a division
    int kh;                                    // key / value heads of a workgroup
};
constexpr unsigned kRopeGridRows = 65535;

__device__ __forceinline__ int load_index(const void* base, int index_bytes, int pos) {
    if (index_bytes == 1) return (int)reinterpret_cast<const uint8_t*>(base)[pos];
    if (index_bytes == 4) return reinterpret_cast<const int32_t*>(base)[pos];
    return (int)reinterpret_cast<const int64_t*>(base)[pos];
}

// one column pair: (lo, hi) = (x[j], x[j + d/2]) with their own table columns
__device__ __forceinline__ void rotate_pair(half_t& lo, half_t& hi, half_t c_lo, half_t s_lo, half_t c_hi,
                                            half_t s_hi) {
    // no fused multiply-add: the reference rounds each product before the sum
#pragma clang fp contract(off)
    const float x1 = (float)lo, x2 = (float)hi;
    const half_t a_lo = (half_t)(x1 * (float)c_lo), r_lo = (half_t)(-x2 * (float)s_lo);
    const half_t a_hi = (half_t)(x2 * (float)c_hi), r_hi = (half_t)(x1 * (float)s_hi);
    lo = (half_t)((float)a_lo + (float)r_lo);
    hi = (half_t)((float)a_hi + (float)r_hi);
}

// Several column pairs at once in packed fp16 arithmetic.  An fp16 product or sum computed in fp32 and rounded to fp16 equals
// the fp16 operation's own single rounding (fp32's 24 bits are at least 2 x 11 + 2), so these are the values of
// rotate_pair bit for bit, at a fifth of its instructions: the conversions made the kernel for many tokens compute-bound.
template <typename V>
__device__ __forceinline__ void rotate_pairs(half_t* to_lo, half_t* to_hi, V lo, V hi, V c_lo, V s_lo, V c_hi, V s_hi) {
#pragma clang fp contract(off)
    const V a_lo = lo * c_lo, r_lo = (-hi) * s_lo;
    const V a_hi = hi * c_hi, r_hi = lo * s_hi;
    *reinterpret_cast<V*>(to_lo) = a_lo + r_lo;
    *reinterpret_cast<V*>(to_hi) = a_hi + r_hi;
}

template <int VEC>
struct HalfVec;  // VEC fp16 values moved with one access
template <>
struct HalfVec<8> { typedef h8 type; };
template <>
struct HalfVec<2> { typedef h2 type; };
template <>
struct HalfVec<1> { typedef half_t type; };

// the indices of VEC neighbouring columns, I bytes each (of eight the low word counts)
template <int VEC, int I>
__device__ __forceinline__ void load_indices(const void* base, int pos, int (&out)[VEC]) {
    typedef uint32_t words4 __attribute__((ext_vector_type(4), aligned(8)));
    typedef uint32_t words2 __attribute__((ext_vector_type(2), aligned(4)));
    if constexpr (VEC == 2 && I == 8) {
        const words4 v = *reinterpret_cast<const words4*>(reinterpret_cast<const uint64_t*>(base) + pos);
        out[0] = (int)v[0];
        out[1] = (int)v[2];
    } else if constexpr (VEC == 2 && I == 4) {
        const words2 v = *reinterpret_cast<const words2*>(reinterpret_cast<const uint32_t*>(base) + pos);
        out[0] = (int)v[0];
        out[1] = (int)v[1];
    } else {
#pragma unroll
        for (int v = 0; v < VEC; ++v) out[v] = load_index(base, I, pos + v);
    }
}

// Few tokens: VEC columns per thread and half of the head.  A block covers 256 consecutive work items of one token.
// Bound by latency: kernel arguments, indices, table values and the store follow each other, and every instruction in
// front of the first load is paid in full (four clocks each; a division is forty of them, a 64-bit one two hundred).
// So no divisions, one round of
// scalar loads, and a thread's indices in two loads: one token 2.6 -> 2.2 us, 48 tokens 2.75 -> 2.4 (heads of 128), 3.1 -> 2.8
// (of 108).
// DIVIDE: sizes for which the rounded inverses are not exact.
template <int VEC, int I, bool DIVIDE>
__global__ __launch_bounds__(256) void rope_indices_kernel(const RopeArgs a) {
    typedef typename HalfVec<VEC>::type vec_t;
    // the kernel arguments in one round of scalar loads
    const int hd = a.hd, half = hd >> 1, n_qh = a.n_qh, n_kh = a.n_kh, per_head = a.per_head;
    const unsigned per_head_inverse = a.per_head_inverse, group_inverse = a.group_inverse;
    half_t *const q = a.q, *const k = a.k;
    const half_t *const cos = a.cos, *const sin = a.sin;
    const void* const indices = a.indices;
    const unsigned rows = a.rows;
    const int64_t q_stride = a.q_row_stride, k_stride = a.k_row_stride, cos_stride = a.cos_row_stride;
    const unsigned seq_len = a.cos_batch == 1 && rows != (unsigned)a.seq_len ? (unsigned)a.seq_len : 0u;
    asm volatile("" ::"s"(q), "s"(k), "s"(cos), "s"(sin), "s"(indices), "s"(per_head_inverse), "s"(group_inverse), "s"(q_stride),
                 "s"(k_stride), "s"(cos_stride), "s"(seq_len));
    const int t = (int)blockIdx.x * 256 + (int)threadIdx.x;
    if (t >= (n_qh + n_kh) * per_head) return;
    const int head = DIVIDE ? t / per_head : (int)__umulhi((unsigned)t, per_head_inverse);
    const int j = (t - head * per_head) * VEC;
    const bool is_q = head < n_qh;
    const int of_q = DIVIDE ? head / a.group : (a.group == 1 ? head : (int)__umulhi((unsigned)head, group_inverse));
    const int kv_head = is_q ? of_q : head - n_qh;
    int i_lo[VEC], i_hi[VEC];
    load_indices<VEC, I>(indices, kv_head * hd + j, i_lo);
    load_indices<VEC, I>(indices, kv_head * hd + half + j, i_hi);
    for (unsigned row = blockIdx.y; row < rows; row += kRopeGridRows) {
        half_t* x = is_q ? q + row * q_stride + (int64_t)head * hd : k + row * k_stride + (int64_t)(head - n_qh) * hd;
        const int64_t table_row = seq_len == 1 ? 0 : (seq_len != 0 ? row % seq_len : row);
        const half_t *cos_row = cos + table_row * cos_stride, *sin_row = sin + table_row * cos_stride;
        const vec_t lo_v = *reinterpret_cast<const vec_t*>(x + j), hi_v = *reinterpret_cast<const vec_t*>(x + half + j);
        if constexpr (VEC == 1) {
            half_t lo = lo_v, hi = hi_v;
            rotate_pair(lo, hi, cos_row[i_lo[0]], sin_row[i_lo[0]], cos_row[i_hi[0]], sin_row[i_hi[0]]);
            x[j] = lo;
            x[half + j] = hi;
        } else {
            vec_t c_lo, s_lo, c_hi, s_hi;
#pragma unroll
            for (int v = 0; v < VEC; ++v) {
                c_lo[v] = cos_row[i_lo[v]];
                s_lo[v] = sin_row[i_lo[v]];
                c_hi[v] = cos_row[i_hi[v]];
                s_hi[v] = sin_row[i_hi[v]];
            }
            rotate_pairs<vec_t>(x + j, x + half + j, lo_v, hi_v, c_lo, s_lo, c_hi, s_hi);
        }
    }
}

// Many tokens: a workgroup builds a token's gathered (cos, sin) pairs once per
// key/value head in LDS (kh x head_dim entries of 4 bytes) and every query head of the
// group reads them from there, instead of every element gathering from the tables in memory.
// The phases of a workgroup wait for each other, so a token's heads are shared out to several (see the launch): 32 + 32 heads of
// 128, one workgroup a token -> four: 333 tokens 7.6 -> 4.8 us, 1024 12.2 -> 9.0, 4096 30.0 -> 23.8; 32 + 8, two: 333 3.9 -> 3.6,
// of 126 6.7 -> 5.3.
// DIVIDE as above; without the divisions 1024 tokens of heads of 108 take 6.0 us instead of 7.05, 333 4.55 instead of 5.2.
template <int VEC, bool DIVIDE>
__global__ __launch_bounds__(256) void rope_indices_lds_kernel(const RopeArgs a, int cos_dim) {
    typedef typename HalfVec<VEC>::type vec_t;
    extern __shared__ __attribute__((aligned(16))) uint32_t rope_lds[];
    uint16_t* trow = reinterpret_cast<uint16_t*>(rope_lds);  // the token's cos row, then its sin row
    // gathered tables: entry (kv head, column) of the cosines, then the same of the sines, as fp16
    uint16_t* tab_cos = reinterpret_cast<uint16_t*>(rope_lds + ((cos_dim + 3) & ~3));
    uint16_t* tab_sin = tab_cos + a.kh * a.hd;
    const int tid = threadIdx.x;
    const unsigned row = blockIdx.x;
    const int first_kv = (int)blockIdx.y * a.kh, qh = a.kh * a.group;
    const int64_t table_row = a.cos_batch == 1 && a.rows != (unsigned)a.seq_len ? row % (unsigned)a.seq_len : row;
    const uint16_t* cos_row = reinterpret_cast<const uint16_t*>(a.cos + table_row * a.cos_row_stride);
    const uint16_t* sin_row = reinterpret_cast<const uint16_t*>(a.sin + table_row * a.cos_row_stride);
    // Everything the token needs from memory is requested before the first barrier: the (cos, sin)
    // row, the thread's first four index entries and its first two work items' q / k values are three
    // independent loads, and issued one behind a barrier behind the other they would cost three
    // memory round trips in a launch that lasts little longer than that.
    const int entries = a.kh * a.hd, first_entry = first_kv * a.hd;
    const int half = a.hd >> 1;
    const int per_head = half / VEC;
    const int per_row = (qh + a.kh) * per_head;
    constexpr int kIdxAhead = 4;
    int idx_ahead[kIdxAhead];
#pragma unroll
    for (int i = 0; i < kIdxAhead; ++i) {
        const int e = tid + 256 * i;
        idx_ahead[i] = e < entries ? load_index(a.indices, a.index_bytes, first_entry + e) : 0;
    }
    auto item = [&](int t, half_t*& x, int& kv_head, int& j) __attribute__((always_inline)) {
        const int head = DIVIDE ? t / per_head : (int)__umulhi((unsigned)t, a.per_head_inverse);
        j = (t - head * per_head) * VEC;
        const bool is_q = head < qh;
        kv_head = is_q ? (DIVIDE ? head / a.group : (a.group == 1 ? head : (int)__umulhi((unsigned)head, a.group_inverse))) : head - qh;
        x = is_q ? a.q + row * a.q_row_stride + (int64_t)(first_kv * a.group + head) * a.hd
                 : a.k + row * a.k_row_stride + (int64_t)(first_kv + head - qh) * a.hd;
    };
    constexpr int kItemsAhead = 2;  // 32 + 8 heads of 128 are 320 work items of eight column pairs: two per thread at most
    half_t* x0[kItemsAhead];
    int kv0[kItemsAhead], j0[kItemsAhead];
    vec_t lo0[kItemsAhead], hi0[kItemsAhead];
#pragma unroll
    for (int i = 0; i < kItemsAhead; ++i) {
        x0[i] = nullptr;
        kv0[i] = j0[i] = 0;
        lo0[i] = hi0[i] = vec_t();
        if (tid + 256 * i < per_row) {
            item(tid + 256 * i, x0[i], kv0[i], j0[i]);
            lo0[i] = *reinterpret_cast<const vec_t*>(x0[i] + j0[i]);
            hi0[i] = *reinterpret_cast<const vec_t*>(x0[i] + half + j0[i]);
        }
    }
    for (int i = tid; i < cos_dim; i += 256) {
        trow[i] = cos_row[i];
        trow[cos_dim + i] = sin_row[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kIdxAhead; ++i) {
        const int e = tid + 256 * i;
        if (e < entries) {
            tab_cos[e] = trow[idx_ahead[i]];
            tab_sin[e] = trow[cos_dim + idx_ahead[i]];
        }
    }
    for (int e = tid + 256 * kIdxAhead; e < entries; e += 256) {
        const int i = load_index(a.indices, a.index_bytes, first_entry + e);
        tab_cos[e] = trow[i];
        tab_sin[e] = trow[cos_dim + i];
    }
    __syncthreads();
    auto rotate_item = [&](half_t* x, int kv_head, int j, vec_t lo_v, vec_t hi_v) __attribute__((always_inline)) {
        const int e0 = kv_head * a.hd + j;
        if constexpr (VEC > 1) {
            rotate_pairs<vec_t>(x + j, x + half + j, lo_v, hi_v, *reinterpret_cast<const vec_t*>(tab_cos + e0),
                                *reinterpret_cast<const vec_t*>(tab_sin + e0), *reinterpret_cast<const vec_t*>(tab_cos + e0 + half),
                                *reinterpret_cast<const vec_t*>(tab_sin + e0 + half));
        } else {
            half_t lo = lo_v, hi = hi_v;
            rotate_pair(lo, hi, __builtin_bit_cast(half_t, tab_cos[e0]), __builtin_bit_cast(half_t, tab_sin[e0]),
                        __builtin_bit_cast(half_t, tab_cos[e0 + half]), __builtin_bit_cast(half_t, tab_sin[e0 + half]));
            *reinterpret_cast<vec_t*>(x + j) = lo;
            *reinterpret_cast<vec_t*>(x + half + j) = hi;
        }
    };
#pragma unroll
    for (int i = 0; i < kItemsAhead; ++i)
        if (tid + 256 * i < per_row) rotate_item(x0[i], kv0[i], j0[i], lo0[i], hi0[i]);
    for (int t = tid + 256 * kItemsAhead; t < per_row; t += 256) {
        half_t* x;
        int kv_head, j;
        item(t, x, kv_head, j);
        const vec_t lo_v = *reinterpret_cast<const vec_t*>(x + j), hi_v = *reinterpret_cast<const vec_t*>(x + half + j);
        rotate_item(x, kv_head, j, lo_v, hi_v);
    }
}

template <int VEC, int I>
static void rope_indices_bytes(const RopeArgs& a, bool divide, dim3 grid, hipStream_t stream) {
    if (divide) hipLaunchKernelGGL((rope_indices_kernel<VEC, I, true>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((rope_indices_kernel<VEC, I, false>), grid, dim3(256), 0, stream, a);
}
template <int VEC>
static void rope_indices_go(const RopeArgs& a, bool divide, dim3 grid, hipStream_t stream) {
    if (a.index_bytes == 1) rope_indices_bytes<VEC, 1>(a, divide, grid, stream);
    else if (a.index_bytes == 4) rope_indices_bytes<VEC, 4>(a, divide, grid, stream);
    else rope_indices_bytes<VEC, 8>(a, divide, grid, stream);
}

template <int VEC>
static void rope_tables_go(const RopeArgs& a, bool divide, int cos_dim, size_t lds_bytes, hipStream_t stream) {
    const dim3 grid(a.rows, (unsigned)(a.n_kh / a.kh));
    if (divide) hipLaunchKernelGGL((rope_indices_lds_kernel<VEC, true>), grid, dim3(256), lds_bytes, stream, a, cos_dim);
    else hipLaunchKernelGGL((rope_indices_lds_kernel<VEC, false>), grid, dim3(256), lds_bytes, stream, a, cos_dim);
}

int rope_indices_launch(void* q, int64_t q_row_stride, void* k, int64_t k_row_stride, const void* cos, const void* sin,
                        int64_t cos_row_stride, const void* indices, int index_bytes, int64_t rows, int seq_len,
                        int cos_batch, int n_qh, int n_kh, int hd, int cos_dim, hipStream_t stream) {
    RopeArgs a;
    a.q = reinterpret_cast<half_t*>(q);
    a.k = reinterpret_cast<half_t*>(k);
    a.cos = reinterpret_cast<const half_t*>(cos);
    a.sin = reinterpret_cast<const half_t*>(sin);
    a.indices = indices;
    a.q_row_stride = q_row_stride;
    a.k_row_stride = k_row_stride;
    a.cos_row_stride = cos_row_stride;
    a.seq_len = seq_len;
    a.cos_batch = cos_batch;
    a.n_qh = n_qh;
    a.n_kh = n_kh;
    a.hd = hd;
    a.index_bytes = index_bytes;
    if (rows == 0) return UNIQL_OK;
    const int half = hd / 2;
    // the widest access every offset (head start, half-head start, row start) is aligned for
    const uintptr_t bases = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k);
    int vec = 1;
    if (half % 8 == 0 && q_row_stride % 8 == 0 && k_row_stride % 8 == 0 && (bases & 15u) == 0) vec = 8;
    else if (half % 2 == 0 && q_row_stride % 2 == 0 && k_row_stride % 2 == 0 && (bases & 3u) == 0) vec = 2;
    // From 128 tokens on workgroups build a token's tables in LDS (where they fit), below that every pair gathers its
    // own values, two columns at a time: more threads in flight hide the dependent index -> table loads better than wide
    // accesses do (32 + 8 heads of 108: 96 tokens 3.15 us against 3.1, 128 3.4 against 3.1, 192 4.1 against 3.3; of 126, one column
    // at a time, 128 3.4 against 3.8, 192 3.7 against 3.9, 512 6.65 against 6.0: from 192 on).
    // A token's key / value heads are halved between workgroups while their number is even and a workgroup has more than eight, or, up
    // to 1024 tokens, more than 24 heads with its query heads (an odd number, as 9 or 5 x 9 heads, stays together: 32 + 8 heads of
    // 128: eight key / value heads 6.2 us at 1024 tokens and 8.8 at 2048, four 5.8 and 9.2, two 7.0 and 11.2; 32 + 32: sixteen 9.5 and
    // 16.3, eight 9.0 and 14.1, four 11.2 and 18.5), and while half of them is enough for a workgroup: 128 work items, and beyond 1024
    // tokens 768 gathered entries (heads of 64: 32 + 32 at 2048 tokens sixteen 8.2, eight 10.2; 40 + 40 forty 9.6, twenty 9.5, five 15.7;
    // 40 + 10 at 4096 ten 9.1, five 10.8; 40 + 40 of 96 at 4096 forty 27.5, ten 21.8, five 30.4).  Left: 64 + 8 heads of 128 at 1024 tokens,
    // eight 6.9, two as here 7.6 (at 2048 11.6 either way).
    a.group = n_qh / n_kh;
    a.kh = n_kh;
    const int64_t items = (int64_t)(a.group + 1) * (half / vec);  // of a key / value head and its query heads
    while (a.kh % 2 == 0 && (a.kh > 8 || (rows <= 1024 && a.kh * (a.group + 1) > 24)) && a.kh / 2 * items >= 128 &&
           (rows <= 1024 || (int64_t)(a.kh / 2) * hd >= 768))
        a.kh /= 2;
    const size_t lds_bytes = ((size_t)((cos_dim + 3) & ~3) + (size_t)a.kh * hd) * 4;
    const bool tables = rows >= (vec == 1 ? 192 : 128) && lds_bytes <= 32 * 1024 && rows <= 0x7fffffffLL && n_kh / a.kh <= 65535;
    if (!tables && vec == 8) vec = 2;
    a.per_head = half / vec;
    const int64_t per_row = (int64_t)(n_qh + n_kh) * a.per_head, blocks = (per_row + 255) / 256;
    if (!tables && (per_row > 0x7fffff00LL || rows * blocks > 0x7fffffffLL)) return UNIQL_E_SHAPE;
    a.rows = (unsigned)rows;
    // floor(t / d) = floor(t inverse / 2^32) while t times the inverse's rounding, less than d, stays below 2^32
    auto exact = [](int64_t dividends, int64_t divisor) { return dividends * divisor < (1LL << 32); };
    auto inverse = [](int divisor) { return (unsigned)(((1ULL << 32) + divisor - 1) / divisor); };
    const bool divide = a.per_head == 1 || !exact(256 * blocks, a.per_head) || !exact(n_qh + n_kh, a.group);
    a.per_head_inverse = divide ? 0u : inverse(a.per_head);
    a.group_inverse = divide || a.group == 1 ? 0u : inverse(a.group);
    if (tables) {
        if (vec == 8) rope_tables_go<8>(a, divide, cos_dim, lds_bytes, stream);
        else if (vec == 2) rope_tables_go<2>(a, divide, cos_dim, lds_bytes, stream);
        else rope_tables_go<1>(a, divide, cos_dim, lds_bytes, stream);
    } else {
        const dim3 grid((unsigned)blocks, rows < (int64_t)kRopeGridRows ? (unsigned)rows : kRopeGridRows);
        if (vec == 2) rope_indices_go<2>(a, divide, grid, stream);
        else rope_indices_go<1>(a, divide, grid, stream);
    }
    return hipGetLastError() == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
}

}  // namespace uniql
