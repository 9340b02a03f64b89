// extern "C" surface: argument checks and dispatch.  Nothing here allocates,
// synchronises or throws.
#include <atomic>
#include <mutex>

#include "common.hpp"
#include "mid_plan.hpp"
#include "tile_plan.hpp"
#include "uniql_amd_diag.h"

namespace uniql {
int stream_launch(const void* A, int64_t lda, int k_valid, const void* B, const void* S, void* D,
                  const Epilogue& epi, void* accum, int m, int n, int k, int groups, int had_mode, float had_scale,
                  unsigned tune, hipStream_t stream);
bool stream_rotates_rows(int m, int k);
size_t stream_accum_bytes(int m, int n, int k, unsigned tune);
size_t stream_accum_bound(int m, int n, int k);
bool stream_shape_ok(int k, int64_t lda);
int read_floor_launch(const void* B, const void* S, void* sink, int m, int n, int k, unsigned tune, hipStream_t stream);
size_t read_floor_sink_bytes(int m, int n, int k, unsigned tune);
int tile_launch(const void* A, int64_t lda, int k_valid, const void* B, const void* S, void* D, const Epilogue& epi, void* accum,
                size_t accum_bytes, void* part, size_t part_bytes, int m, int n, int k, int groups, int first, int columns,
                const TilePlan& plan, hipStream_t stream);
bool tile_shape_ok(int m, int n, int k, int64_t ldx, int columns, const TilePlan& plan);
int mid_launch(const void* A, int64_t lda, int k_valid, const void* B, const void* S, void* D, const Epilogue& epi, void* accum,
               void* part, int m, int n, int k, int groups, const MidPlan& plan, hipStream_t stream);
bool mid_shape_ok(int m, int n, int k, int64_t lda);
int pad_rows_launch(const void* A, int64_t lda, int k_in, void* dst, int k, int m, hipStream_t stream);
int wide_launch(const void* A, int64_t lda, int k_valid, const void* B, const void* S, void* D, const Epilogue& epi, int m, int n,
                int k, int groups, int first, int columns, hipStream_t stream);
bool wide_shape_ok(int m, int n, int k, int groups, int64_t ldx);
int dequant_launch(const void* B, const void* S, void* W, uint8_t* codes, int n, int k, int groups,
                   hipStream_t stream);
int embedding_launch(const int64_t* ids, int64_t ntokens, const void* weight, const void* scales, void* out,
                     int64_t vocab, int dim, hipStream_t stream);
int embedding_quantize_launch(const void* W, int64_t ldw, void* packed, void* scales, int64_t vocab, int dim,
                              hipStream_t stream);
int rope_indices_launch(void* q, int64_t q_row_stride, void* k, int64_t k_row_stride, const void* cos, const void* sin,
                        int64_t cos_row_stride, const void* indices, int index_bytes, int64_t rows, int seq_len,
                        int cos_batch, int n_qh, int n_kh, int hd, int cos_dim, hipStream_t stream);
int fwht_launch(const void* x, void* y, int64_t rows, int dim, int block, float scale, int dtype,
                hipStream_t stream);
int fwht_composite_launch(const void* x, void* y, int64_t rows, int dim, int base, float scale, int dtype,
                          hipStream_t stream);
int fwht_columns_launch(const void* x, void* y, int rows, int cols, float scale, int dtype, hipStream_t stream);
int quantize_launch(const void* W, int64_t ldw, const void* given_scales, void* B, void* S, int out_features,
                    int in_features, int n_pad, int k_pad, hipStream_t stream);
int pack_launch(const uint8_t* codes, const void* scales, void* B, void* S, int n, int k, int n_pad, int k_pad,
                hipStream_t stream);
int cut_columns_launch(const void* B, const void* S, int n, int k, int k_real, const int* runs, int n_runs, int n_scaled,
                       void* B_out, void* S_out, int n_pad, hipStream_t stream);
int cut_rows_launch(const void* B, const void* S, int n, int groups_in, int units, int full, int kept, int n_real, void* B_out,
                    void* S_out, int n_pad, hipStream_t stream);
bool stream_allow_lds();
bool mid_allow_lds();
bool tile_allow_lds();
bool wide_allow_lds();
bool fwht_allow_lds();
}  // namespace uniql

using namespace uniql;

static inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
static inline bool is_pow2(int v) { return v > 0 && (v & (v - 1)) == 0; }
static inline size_t round256(size_t v) { return (v + 255) & ~(size_t)255; }

// More than 64 KiB of LDS is a property of (kernel, device) that may not be set while a stream is capturing, and which kernel
// a layer call launches follows from all of its sizes: so the first call on a device sets it for every kernel of these calls
// (it takes 13.5 to 14 ms, nearly all of it to load code; 12.9 while the tiled kernel had 12 instantiations in place of 30).
static bool prepare_device() {
    static std::atomic<unsigned long long> done{0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    const unsigned long long bit = dev < 64 ? 1ull << dev : 0ull;  // further devices: set again on every call
    if (done.load(std::memory_order_acquire) & bit) return true;
    if (!stream_allow_lds() || !mid_allow_lds() || !tile_allow_lds() || !wide_allow_lds() || !fwht_allow_lds()) return false;
    done.fetch_or(bit, std::memory_order_release);
    return true;
}

static int check_linear_shape(int m, int n, int k, int groups) {
    if (m < 0 || n <= 0 || k <= 0) return UNIQL_E_SHAPE;
    if (n % 128 != 0 || k % 128 != 0) return UNIQL_E_SHAPE;
    if (!(groups == 1 || groups == k / 128)) return UNIQL_E_SHAPE;
    return UNIQL_OK;
}

extern "C" {

int uniql_abi_version(void) { return UNIQL_ABI_VERSION; }

int uniql_stream_capture_id(void* stream, unsigned long long* id) {
    if (!id) return UNIQL_E_NULL;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long capture = 0;
    if (hipStreamGetCaptureInfo(reinterpret_cast<hipStream_t>(stream), &status, &capture) != hipSuccess)
        return UNIQL_E_LAUNCH;
    *id = status == hipStreamCaptureStatusActive ? capture : 0;
    return UNIQL_OK;
}

const char* uniql_status_string(int code) {
    switch (code) {
        case UNIQL_OK: return "ok";
        case UNIQL_E_NULL: return "a required pointer is NULL";
        case UNIQL_E_SHAPE: return "sizes violate the packed layout (k % 128, n % 128, groups, dim, block)";
        case UNIQL_E_ALIGN: return "pointer or leading dimension not 16-byte aligned";
        case UNIQL_E_WORKSPACE: return "workspace, accum or temp buffer too small";
        case UNIQL_E_UNSUPPORTED: return "request not supported by this build";
        case UNIQL_E_LAUNCH: return "HIP runtime rejected the kernel launch";
        case UNIQL_E_STATIC_LIMIT:
            return "the call needs more scratch memory than the library's static buffer holds "
                   "(uniql_w4a16_gemm_static_limit); use uniql_w4a16_gemm with caller-provided buffers";
        default: return "unknown status";
    }
}

// rows up to this many take the weight-streaming kernel, more take the tiled one
static constexpr int kStreamMaxM = 16;

// Which kernels a call goes to: the streaming kernel, or (see mid_for_few_rows) the one for 9 to 64 rows in its place, or those of
// the plan below.
static bool takes_stream_kernel(int m, unsigned flags) {
    bool use_stream = m <= kStreamMaxM;
    if (flags & UNIQL_F_FORCE_SKINNY) use_stream = true;
    if (flags & UNIQL_F_FORCE_TILED) use_stream = false;
    return use_stream;
}

// How the streaming kernel itself applies a rotation: 1 the 128-block one while staging, 2 whole
// rows (block = k, a power of two, few rows, input not shorter than k), 0 not at all: then the
// transform kernel runs first, into `temp`.
static int fused_rotation(int m, int k, int k_in, int had_block, bool use_stream, unsigned flags) {
    if (!use_stream || had_block == 0) return 0;
    if (had_block == 128) return 1;
    if (flags & UNIQL_F_SEPARATE_ROTATION) return 0;
    return (had_block == k && k_in == k && stream_rotates_rows(m, k)) ? 2 : 0;
}

// bytes of the rotated or zero-padded copy of the activations at the start of `temp`, at most: every
// rotation that is not fused into the streaming kernel, and padding in front of a rotation or where
// the rows are too far apart for the tiled kernels to read short ones as they are (the stride is not known here)
static size_t activation_copy_bytes(int m, int k, int k_in, int had_block, bool use_stream, unsigned flags) {
    const bool rotate_first = had_block != 0 && fused_rotation(m, k, k_in, had_block, use_stream, flags) == 0;
    const bool pad_first = k_in != k && (rotate_first || !use_stream);
    return (rotate_first || pad_first) ? round256((size_t)m * k * sizeof(half_t)) : 0;
}

static constexpr size_t kStaticAccumBytes = (size_t)4 << 20;   // the static area: exchange words, 16 rows x 32768 columns
static constexpr size_t kStaticTempBytes = (size_t)12 << 20;   //                  rotated rows / partial tiles

// Partial tiles of any call fit the static area (with more splits than that the exchange costs more than it gives);
// the static entry asks for less where the copy of the activations needs the room.
static constexpr size_t kPartialCap = kStaticTempBytes;

// What one layer call needs, decided in ONE place for the argument checks, the launch and the
// entry point that brings its own scratch memory: which kernels take the call, whether the
// activations are copied (rotated / zero-padded) into `temp` first, and the bytes of `accum` and
// `temp` that follow from that.  The 256 x 256 kernel needs neither buffer; two launches of the 128-column
// kernel run one after the other and share theirs.
struct LinearNeeds {
    bool use_stream, rotate_first, pad_first;
    int had_mode;
    int64_t ld_kernel;   // row stride the product kernel will see
    LinearPlan plan;     // of the tiled kernels
    MidPlan mid[2];      // the kernel for 9 to 64 rows, where it takes a launch of the plan (upw > 0)
    size_t accum_bytes;  // rounded to 256
    size_t act_bytes;    // copy of the activations at the start of temp (rounded to 256), or 0
    size_t part_bytes;   // the tiled kernel's partial tiles behind it, or 0
};
// The kernel for 9 to 64 rows (w4a16_mid.hip) for one launch of a call: upw = 0 where it does not take it.
static const MidPlan kNoMid = {0, 0, 0, 0.0};

// In place of the streaming kernel: from 9 rows on that kernel's one atomic per output element and K split costs more than
// the exchange of partial tiles, and its single row tile does not use what the second wave of a SIMD hides.  us at 9 / 16 rows,
// there and here: 1024 -> 4096 0.69 / 0.56 x; 4096 -> 512 6.4 / 6.6 and 6.3 / 6.2; 4096 -> 4096 7.5 / 8.5 and 6.5 / 6.8; 14336 -> 4096
// 10.7 / 12.2 and 10.0 / 10.3.  Not for few columns over a long K, where more than eight partial tiles meet (9984 -> 2560 8.0 / 9.0 and
// 8.7 / 9.1, 11904 -> 512 1.22 / 1.03 x; 8192 -> 2560 0.90 / 0.84 x, 11904 -> 3072 9.75 / 10.8 and 8.9 / 9.2), and not from 144
// strips on, where the streaming kernel mostly splits nothing (4096 -> 28672 within 3 %, 4096 -> 128256 46.0 / 48.6 and 48.7 /
// 52.0).  Rows that are rotated stay with the streaming kernel, which rotates blocks of 128 and short rows while it stages them.
static MidPlan mid_for_few_rows(int m, int n, int k, int had_block, unsigned flags, size_t part_cap) {
    if (m < kMidMinRows || m > kStreamMaxM || had_block != 0 || (flags & (UNIQL_F_FORCE_SKINNY | UNIQL_F_FORCE_TILED)) || (flags >> 8) != 0)
        return kNoMid;
    return n / 128 < 144 && (k <= 8192 || n >= 3072) ? mid_plan(m, n, k, 0, part_cap) : kNoMid;
}

// In place of a launch of the tiled kernels, where it is expected to be faster.  Over a short K of fewer than 12 groups the tiled
// kernels' expected times are the better ones from 33 rows on.  Plans that add longer chains of products than the tiled kernel's own are left out: a sum
// is no less exact here than there (8192 -> 512 at 56 rows with two groups a wave: 1.1 x the distance from float64).
// Drawn calls: 17 to 32 rows 1.26 x faster on average, 33 to 48 1.17, 49 to 64 1.03.
// short_rows: fewer columns of X than K.  Up to 32 rows the tiled kernels' form for those is slower than its expected time: of 49
// drawn calls of 17 to 32 rows for which the tiled kernels are rated up to 2 us better 35 are faster here by more than 2 % and 4
// there (1744 -> 28032 at 25 rows 9.4 us against 11.5, 14280 -> 9216 at 17 21.2 against 22.4), of 27 of 33 to 48 rows 5 and 13, of 324 of
// more 29 and 211.
static MidPlan mid_for_tiles(const RowPart& part, int n, int k, bool short_rows, unsigned flags, size_t part_cap) {
    if (part.rows < kMidMinRows || part.rows > kMidMaxRows) return kNoMid;
    if (((flags >> 16) & 0xfu) == 9) return mid_plan(part.rows, n, k, (int)((flags >> 8) & 0xffu), part_cap);  // asked for
    if (part.rows <= kStreamMaxM || (part.rows > 32 && k < 12 * 128)) return kNoMid;
    if ((flags & UNIQL_F_FORCE_TILED) || ((flags >> 8) & 0x3fffu) != 0) return kNoMid;
    const MidPlan p = mid_plan(part.rows, n, k, 0, part_cap, tile_chain(part.tile));
    return p.upw > 0 && p.us < part.tile.us + (short_rows && part.rows <= 32 ? 2.0 : 0.0) ? p : kNoMid;
}

// basic: neither the kernel for 9 to 64 rows nor columns in two launches, for callers whose scratch memory is enough for the
// other kernels only (none at all up to 16 rows, or sized by a library in front of those).
static LinearNeeds linear_needs(int m, int n, int k, int k_in, int64_t lda, int groups, int had_block, unsigned flags,
                                size_t part_cap = kPartialCap, bool basic = false) {
    LinearNeeds q;
    const unsigned tune = flags >> 8;
    q.use_stream = takes_stream_kernel(m, flags);
    q.had_mode = fused_rotation(m, k, k_in, had_block, q.use_stream, flags);
    q.rotate_first = had_block != 0 && q.had_mode == 0;
    // the transform kernel reads dense rows of k values: a strided or short input is first copied
    // (and zero-padded) into the temporary buffer, then rotated there in place; rows too far apart for the tiled kernels'
    // 32-bit offsets are copied as well where they are short
    q.pad_first = q.rotate_first ? (k_in != k || lda != k) : (k_in != k && !q.use_stream && lda >= (1LL << 24));
    q.ld_kernel = (q.rotate_first || q.pad_first) ? (int64_t)k : lda;
    q.plan.parts = q.plan.head_columns = 0;
    q.mid[0] = q.mid[1] = kNoMid;
    q.accum_bytes = q.part_bytes = 0;
    if (q.use_stream) {
        if (!basic && mid_shape_ok(m, n, k, lda)) q.mid[0] = mid_for_few_rows(m, n, k, had_block, flags, part_cap);
        if (q.mid[0].upw > 0) {
            q.use_stream = false;
            q.plan.parts = 1;
            q.plan.part[0] = RowPart{m, false, TilePlan{}};
        } else {
            q.accum_bytes = round256(stream_accum_bytes(m, n, k, tune));
        }
    } else {
        q.plan = basic ? linear_plan(m, n, k, wide_shape_ok(m, n, k, groups, q.ld_kernel), part_cap, tune)
                       : call_plan(m, n, k, wide_shape_ok(m, n & ~255, k, groups, q.ld_kernel), part_cap, tune);
        for (int i = 0; i < q.plan.parts; ++i)
            if (!basic && q.plan.head_columns == 0 && mid_shape_ok(q.plan.part[i].rows, n, k, q.rotate_first ? k : lda))
                q.mid[i] = mid_for_tiles(q.plan.part[i], n, k, k_in != k && !q.rotate_first, flags, part_cap);
    }
    for (int i = 0; i < q.plan.parts; ++i) {
        const RowPart& part = q.plan.part[i];
        const bool mid = q.mid[i].upw > 0;
        const int columns = part_columns(q.plan, i, n);
        const size_t acc = round256(mid ? mid_accum_bytes(n, q.mid[i]) : part.wide ? 0 : tile_accum_bytes(part.rows, columns, part.tile));
        const size_t tmp = mid ? mid_part_bytes(part.rows, n, q.mid[i]) : part.wide ? 0 : tile_part_bytes(part.rows, columns, part.tile);
        q.accum_bytes = acc > q.accum_bytes ? acc : q.accum_bytes;
        q.part_bytes = tmp > q.part_bytes ? tmp : q.part_bytes;
    }
    q.act_bytes = (q.rotate_first || q.pad_first) ? round256((size_t)m * k * sizeof(half_t)) : 0;
    return q;
}

// The most the kernels of a call may ask for, whichever of them its scales, strides and input width let take it.
static void call_workspace(int m, int n, int k, int had_block, unsigned flags, size_t* accum, size_t* part) {
    *accum = *part = 0;
    auto most = [&](int rows, const MidPlan& mid) {
        if (mid.upw == 0) return;
        const size_t a = mid_accum_bytes(n, mid), p = mid_part_bytes(rows, n, mid);
        *accum = a > *accum ? a : *accum;
        *part = p > *part ? p : *part;
    };
    if (takes_stream_kernel(m, flags)) {
        *accum = stream_accum_bytes(m, n, k, flags >> 8);
        most(m, mid_for_few_rows(m, n, k, had_block, flags, kPartialCap));
        return;
    }
    for (int wide = 0; wide < 2; ++wide) {
        const LinearPlan plan = call_plan(m, n, k, wide != 0 && wide_shape_ok(m, n & ~255, k, k / 128, k), kPartialCap, flags >> 8);
        const size_t a = plan_accum_bytes(plan, n), p = plan_part_bytes(plan, n);
        *accum = a > *accum ? a : *accum;
        *part = p > *part ? p : *part;
        for (int i = 0; i < plan.parts; ++i)
            for (int short_rows = 0; short_rows < 2; ++short_rows)
                most(plan.part[i].rows, mid_for_tiles(plan.part[i], n, k, short_rows != 0, flags, kPartialCap));
    }
}

int uniql_w4a16_linear_workspace(int m, int n, int k, int k_in, int had_block, unsigned flags, size_t* accum_bytes,
                                 size_t* temp_bytes) {
    if (!accum_bytes || !temp_bytes) return UNIQL_E_NULL;
    *accum_bytes = *temp_bytes = 0;
    if (m < 0 || n <= 0 || k <= 0 || n % 128 != 0 || k % 128 != 0) return UNIQL_E_SHAPE;
    if (m == 0) return UNIQL_OK;
    const bool use_stream = takes_stream_kernel(m, flags);
    // a strided input ahead of a separate rotation is compacted into the copy as well: count it
    const size_t act = had_block != 0 && fused_rotation(m, k, k_in, had_block, use_stream, flags) == 0
                           ? round256((size_t)m * k * sizeof(half_t))
                           : activation_copy_bytes(m, k, k_in, had_block, use_stream, flags);
    size_t accum, part;
    call_workspace(m, n, k, had_block, flags, &accum, &part);
    *accum_bytes = round256(accum);
    *temp_bytes = act + round256(part);
    return UNIQL_OK;
}

size_t uniql_w4a16_gemm_accum_bytes(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0 || n % 128 != 0 || k % 128 != 0) return 0;
    // enough for either kernel with its own plan (forced tuning fields: uniql_w4a16_linear_workspace)
    const size_t a = stream_accum_bound(m, n, k);
    size_t b, part;
    call_workspace(m, n, k, 0, 0, &b, &part);
    return round256(a > b ? a : b);
}

size_t uniql_w4a16_linear_temp_bytes(int m, int n, int k, int k_in, int had_block) {
    if (m <= 0 || n <= 0 || k <= 0 || n % 128 != 0 || k % 128 != 0) return 0;
    // the copy of the activations (as if the tiled kernel took the call: the larger case) and the
    // partial tiles of the tiled kernel's own plan
    const size_t act = (had_block != 0 || k_in != k) ? round256((size_t)m * k * sizeof(half_t)) : 0;
    size_t accum, part;
    call_workspace(m, n, k, had_block, 0, &accum, &part);
    return act + round256(part);
}

size_t uniql_w4a16_gemm_temp_bytes(int m, int n, int k, int had_block) {
    return uniql_w4a16_linear_temp_bytes(m, n, k, k, had_block);
}

// check_only: every argument check, then return before the first kernel is enqueued
static int linear_impl(const void* A, int64_t lda, int k_in, const void* B, const void* S, const void* bias,
                       const void* residual, int64_t ldr, void* D, int64_t ldd, int n_out, int epilogue,
                       const int32_t* workspace,
                       int64_t workspace_len, void* accum, size_t accum_bytes, void* temp, size_t temp_bytes, int m,
                       int n, int k, int groups, int had_block, float had_scale, unsigned flags, void* stream,
                       bool check_only, size_t part_cap) {
    const int rc = check_linear_shape(m, n, k, groups);
    if (rc != UNIQL_OK) return rc;
    const bool transpose = (flags & UNIQL_F_TRANSPOSE_OUT) != 0;
    if (epilogue != UNIQL_EPI_NONE && epilogue != UNIQL_EPI_SILU_MUL && epilogue != UNIQL_EPI_RELU2)
        return UNIQL_E_UNSUPPORTED;
    const bool gated = epilogue == UNIQL_EPI_SILU_MUL;
    if (k_in <= 0 || k_in > k || k - k_in >= 128 || (k_in % 8) != 0) return UNIQL_E_SHAPE;
    if (n_out <= 0 || n_out > (gated ? n / 2 : n) || ldd < (transpose ? m : n_out)) return UNIQL_E_SHAPE;
    if (m == 0) return UNIQL_OK;
    if (!A || !B || !S || !D) return UNIQL_E_NULL;
    if (lda < k_in || (lda % 8) != 0) return UNIQL_E_ALIGN;
    const bool out_f32 = (flags & UNIQL_F_OUT_F32) != 0;
    if (!aligned16(A) || !aligned16(B) || !aligned16(S)) return UNIQL_E_ALIGN;
    if (reinterpret_cast<uintptr_t>(D) % (out_f32 ? 4 : 2) != 0) return UNIQL_E_ALIGN;
    if (bias && (reinterpret_cast<uintptr_t>(bias) & 1u)) return UNIQL_E_ALIGN;
    if (residual) {
        if (epilogue != UNIQL_EPI_NONE) return UNIQL_E_UNSUPPORTED;  // activations feed the next layer, not the residual stream
        if (ldr < n_out) return UNIQL_E_SHAPE;
        if (reinterpret_cast<uintptr_t>(residual) & 1u) return UNIQL_E_ALIGN;
    }
    if (workspace && workspace_len < n / 128) return UNIQL_E_WORKSPACE;
    if (had_block != 0 && (!is_pow2(had_block) || had_block < 2 || had_block > 32768 || k % had_block != 0))
        return UNIQL_E_SHAPE;
    if ((accum && !aligned16(accum)) || (temp && !aligned16(temp))) return UNIQL_E_ALIGN;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const unsigned tune = flags >> 8;  // tuning fields, see the header
    LinearNeeds q = linear_needs(m, n, k, k_in, lda, groups, had_block, flags, part_cap);
    auto enough = [&]() {
        return (q.accum_bytes == 0 || (accum && accum_bytes >= q.accum_bytes)) &&
               (q.act_bytes + q.part_bytes == 0 || (temp && temp_bytes >= q.act_bytes + q.part_bytes));
    };
    if (!enough() && ((flags >> 16) & 0xfu) != 9)
        q = linear_needs(m, n, k, k_in, lda, groups, had_block, flags, part_cap, true);
    const bool use_stream = q.use_stream, rotate_first = q.rotate_first, pad_first = q.pad_first;
    const int had_mode = q.had_mode;
    const int64_t ld_kernel = q.ld_kernel;
    const void* Ain = A;
    int64_t ld = lda;
    int k_valid = k_in;
    if (!enough()) return UNIQL_E_WORKSPACE;
    // temp: the copy of the activations, then the partial tiles of a kernel that splits K
    const size_t act_bytes = q.act_bytes, part_bytes = q.part_bytes;
    void* part = part_bytes ? reinterpret_cast<char*>(temp) + act_bytes : nullptr;
    // last check before the first kernel is enqueued: whether the tiled kernel can take the shape
    for (int i = 0; i < q.plan.parts; ++i)
        if (!q.plan.part[i].wide && q.mid[i].upw == 0 && !tile_shape_ok(q.plan.part[i].rows, n, k, ld_kernel, part_columns(q.plan, i, n), q.plan.part[i].tile))
            return UNIQL_E_SHAPE;
    if (use_stream && !stream_shape_ok(k, ld_kernel)) return UNIQL_E_SHAPE;
    if (check_only) return UNIQL_OK;
    if (!prepare_device()) return UNIQL_E_LAUNCH;
    if (pad_first) {
        const int e = pad_rows_launch(A, lda, k_in, temp, k, m, st);
        if (e != UNIQL_OK) return e;
        Ain = temp;
        ld = k;
        k_valid = k;
    }
    if (rotate_first) {
        const int e = fwht_launch(Ain, temp, m, k, had_block, had_scale, UNIQL_DT_F16, st);
        if (e != UNIQL_OK) return e;
        Ain = temp;
        ld = k;
        k_valid = k;
    }
    Epilogue epi;
    epi.bias = reinterpret_cast<const half_t*>(bias);
    epi.residual = reinterpret_cast<const half_t*>(residual);
    epi.ldr = ldr;
    epi.ldd = ldd;
    epi.n_store = n_out;
    epi.gated = gated ? 1 : 0;
    epi.out_f32 = out_f32 ? 1 : 0;
    epi.transpose = transpose ? 1 : 0;
    epi.relu2 = epilogue == UNIQL_EPI_RELU2 ? 1 : 0;
    epi.vec_ok = (!transpose && ldd % 8 == 0 && aligned16(D)) ? 1 : 0;
    epi.residual_vec = residual && epi.vec_ok && !out_f32 && aligned16(residual) && ldr % 8 == 0 && ldr < (1 << 22) ? 1 : 0;
    if (use_stream)
        return stream_launch(Ain, ld, k_valid, B, S, D, epi, accum, m, n, k, groups, had_mode, had_scale, tune, st);
    int m0 = 0, first = 0;
    for (int i = 0; i < q.plan.parts; ++i) {
        const int columns = part_columns(q.plan, i, n);
        const RowPart& p = q.plan.part[i];
        const char* x = reinterpret_cast<const char*>(Ain) + (size_t)m0 * ld * sizeof(half_t);
        char* d = reinterpret_cast<char*>(D) + (size_t)m0 * (transpose ? 1 : ldd) * (out_f32 ? 4 : 2);
        epi.residual = residual ? reinterpret_cast<const half_t*>(residual) + (size_t)m0 * ldr : nullptr;
        const int e = q.mid[i].upw > 0
                          ? mid_launch(x, ld, k_valid, B, S, d, epi, accum, part, p.rows, n, k, groups, q.mid[i], st)
                      : p.wide ? wide_launch(x, ld, k_valid, B, S, d, epi, p.rows, n, k, groups, first, columns, st)
                               : tile_launch(x, ld, k_valid, B, S, d, epi, accum, accum_bytes, part, part_bytes, p.rows, n, k, groups, first, columns, p.tile, st);
        if (e != UNIQL_OK) return e;
        if (q.plan.head_columns == 0) m0 += p.rows;
        else first += columns;
    }
    return UNIQL_OK;
}

int uniql_w4a16_linear(const void* A, int64_t lda, int k_in, const void* B, const void* S, const void* bias,
                       const void* residual, int64_t ldr, void* D, int64_t ldd, int n_out, int epilogue,
                       const int32_t* workspace,
                       int64_t workspace_len, void* accum, size_t accum_bytes, void* temp, size_t temp_bytes, int m,
                       int n, int k, int groups, int had_block, float had_scale, unsigned flags, void* stream) {
    return linear_impl(A, lda, k_in, B, S, bias, residual, ldr, D, ldd, n_out, epilogue, workspace, workspace_len, accum,
                       accum_bytes, temp, temp_bytes, m, n, k, groups, had_block, had_scale, flags, stream, false, kPartialCap);
}

static int gemm_impl(const void* A, int64_t lda, const void* B, const void* S, void* D, const int32_t* workspace,
                     int64_t workspace_len, void* accum, size_t accum_bytes, void* temp, size_t temp_bytes, int m,
                     int n, int k, int groups, int had_block, float had_scale, unsigned flags, void* stream,
                     bool check_only, size_t part_cap) {
    if (D && !aligned16(D)) return UNIQL_E_ALIGN;
    // transposed: D is [n, m8] with m8 = m rounded up to 8, as the reference allocates it
    // (marlin_gemm_kernel.cuh:1023-1026)
    const int64_t ldd = (flags & UNIQL_F_TRANSPOSE_OUT) ? (int64_t)((m + 7) / 8) * 8 : n;
    return linear_impl(A, lda, k, B, S, nullptr, nullptr, 0, D, ldd, n, UNIQL_EPI_NONE, workspace, workspace_len, accum,
                       accum_bytes, temp, temp_bytes, m, n, k, groups, had_block, had_scale, flags, stream, check_only, part_cap);
}

int uniql_w4a16_gemm(const void* A, int64_t lda, const void* B, const void* S, void* D, const int32_t* workspace,
                     int64_t workspace_len, void* accum, size_t accum_bytes, void* temp, size_t temp_bytes, int m,
                     int n, int k, int groups, int had_block, float had_scale, unsigned flags, void* stream) {
    return gemm_impl(A, lda, B, S, D, workspace, workspace_len, accum, accum_bytes, temp, temp_bytes, m, n, k, groups,
                     had_block, had_scale, flags, stream, false, kPartialCap);
}

// ---- the entry point that allocates nothing --------------------------------------------------
// All the scratch memory a product needs (the zero-in / zero-out exchange words first, then the
// temporary area) lives in one array in this library's device image.  Each GPU holds its own copy
// at its own address; the name below is only a host-side handle for hipGetSymbolAddress, never a
// device address, so every use goes through the per-device pointer looked up once.
static __device__ __align__(256) unsigned char scratch[kStaticAccumBytes + kStaticTempBytes];

static constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mutex;
static unsigned char* g_scratch_ptr[kMaxDevices];  // zero-initialised: not looked up yet

// the current device's copy of the array, or nullptr
static unsigned char* static_scratch() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        g_scratch_ptr[dev] = reinterpret_cast<unsigned char*>(p);
    }
    return g_scratch_ptr[dev];
}

size_t uniql_w4a16_gemm_static_limit(int which) {
    return which == 0 ? kStaticAccumBytes : (which == 1 ? kStaticTempBytes : 0);
}

int uniql_w4a16_gemm_static(const void* A, int64_t lda, const void* B, const void* S, void* D,
                            const int32_t* workspace, int64_t workspace_len, int m, int n, int k, int groups,
                            int had_block, float had_scale, unsigned flags, void* stream) {
    const int rc = check_linear_shape(m, n, k, groups);
    if (rc != UNIQL_OK) return rc;
    if (m == 0) return UNIQL_OK;
    // (the sizes of the kernel that will really take the call: a long prefill on the 256 x 256 kernel needs
    // no scratch at all, whatever the 128-column kernel would have asked for)
    size_t part_cap = kPartialCap;
    LinearNeeds q = linear_needs(m, n, k, k, lda, groups, had_block, flags, part_cap);
    if (q.act_bytes <= kStaticTempBytes && q.act_bytes + round256(q.part_bytes) > kStaticTempBytes) {
        // the copy of the activations leaves less room for partial tiles: fewer K splits
        part_cap = kStaticTempBytes - q.act_bytes;
        q = linear_needs(m, n, k, k, lda, groups, had_block, flags, part_cap);
    }
    const size_t need_accum = q.accum_bytes, need_temp = q.act_bytes + round256(q.part_bytes);
    // (up to 16 rows the words of a K split have to fit, whether or not this call's plan makes one)
    const size_t words = takes_stream_kernel(m, flags) ? round256(stream_accum_bound(m, n, k)) : need_accum;
    if (words > kStaticAccumBytes || need_accum > kStaticAccumBytes || need_temp > kStaticTempBytes) return UNIQL_E_STATIC_LIMIT;
    if (!A || !B || !S || !D) return UNIQL_E_NULL;
    unsigned char* base = static_scratch();
    if (!base) return UNIQL_E_LAUNCH;
    void* accum = need_accum ? base : nullptr;
    void* temp = need_temp ? base + kStaticAccumBytes : nullptr;
    // every argument check of the product first: nothing is enqueued for a call that will be refused
    const int crc = gemm_impl(A, lda, B, S, D, workspace, workspace_len, accum, need_accum, temp, need_temp, m, n, k,
                              groups, had_block, had_scale, flags, stream, true, part_cap);
    if (crc != UNIQL_OK) return crc;
    // The exchange words must be zero on entry.  The kernels leave them zero, but the array is
    // shared by every call on this GPU, so the part this call uses is cleared by a small kernel
    // (a kernel, not a memset node: the call may be recorded into a graph).
    if (need_accum > 0) {
        const int e = uniql_clear(base, need_accum, stream);
        if (e != UNIQL_OK) return e;
    }
    return gemm_impl(A, lda, B, S, D, workspace, workspace_len, accum, need_accum, temp, need_temp, m, n, k, groups,
                     had_block, had_scale, flags, stream, false, part_cap);
}

int uniql_w4a16_read_floor(const void* B, const void* S, void* sink, size_t sink_bytes, int m, int n, int k,
                           unsigned flags, void* stream) {
    const int rc = check_linear_shape(m, n, k, k / 128);
    if (rc != UNIQL_OK) return rc;
    if (m <= 0) return UNIQL_E_SHAPE;
    if (!B || !S || !sink) return UNIQL_E_NULL;
    if (!aligned16(B) || !aligned16(S)) return UNIQL_E_ALIGN;
    if (sink_bytes < read_floor_sink_bytes(m, n, k, flags >> 8)) return UNIQL_E_WORKSPACE;
    return read_floor_launch(B, S, sink, m, n, k, flags >> 8, reinterpret_cast<hipStream_t>(stream));
}

size_t uniql_w4a16_read_floor_sink_bytes(int m, int n, int k, unsigned flags) {
    if (m <= 0 || n <= 0 || k <= 0 || n % 128 != 0 || k % 128 != 0) return 0;
    return read_floor_sink_bytes(m, n, k, flags >> 8);
}

int uniql_w4a16_dequant(const void* B, const void* S, void* W, uint8_t* codes, int n, int k, int groups,
                        void* stream) {
    const int rc = check_linear_shape(1, n, k, groups);
    if (rc != UNIQL_OK) return rc;
    if (!B || !S || (!W && !codes)) return UNIQL_E_NULL;
    if (!aligned16(B)) return UNIQL_E_ALIGN;
    return dequant_launch(B, S, W, codes, n, k, groups, reinterpret_cast<hipStream_t>(stream));
}

int uniql_w4a16_quantize(const void* W, int64_t ldw, const void* given_scales, void* B, void* S, int out_features,
                         int in_features, int n_pad, int k_pad, void* stream) {
    if (!W || !B || !S) return UNIQL_E_NULL;
    if (out_features <= 0 || in_features <= 0 || ldw < in_features) return UNIQL_E_SHAPE;
    if (k_pad != (in_features + 127) / 128 * 128 || n_pad < out_features || n_pad % 128 != 0) return UNIQL_E_SHAPE;
    if (in_features <= 128) return UNIQL_E_UNSUPPORTED;
    if ((int64_t)(k_pad / 16) * 2 * n_pad > 0x7fffffffLL * 256) return UNIQL_E_SHAPE;
    return quantize_launch(W, ldw, given_scales, B, S, out_features, in_features, n_pad, k_pad,
                           reinterpret_cast<hipStream_t>(stream));
}

int uniql_w4a16_pack(const uint8_t* codes, const void* scales, void* B, void* S, int n, int k, int n_pad,
                     void* stream) {
    if (!codes || !scales || !B || !S) return UNIQL_E_NULL;
    if (n <= 0 || k <= 0 || k % 128 != 0 || n_pad < n || n_pad % 128 != 0) return UNIQL_E_SHAPE;
    if ((int64_t)(k / 16) * 2 * n_pad > 0x7fffffffLL * 256) return UNIQL_E_SHAPE;
    return pack_launch(codes, scales, B, S, n, k, n_pad, k, reinterpret_cast<hipStream_t>(stream));
}

int uniql_w4a16_cut_columns(const void* B, const void* S, int n, int k, int k_real, const int* runs, int n_runs, int n_scaled,
                            void* B_out, void* S_out, int n_pad, void* stream) {
    const int rc = check_linear_shape(1, n, k, k / 128);
    if (rc != UNIQL_OK) return rc;
    if (!B || !S || !runs || !B_out || !S_out) return UNIQL_E_NULL;
    if (n_runs < 1 || n_runs > 5 || k_real < 0 || k_real > k) return UNIQL_E_SHAPE;
    int64_t total = 0;
    for (int i = 0; i < n_runs; ++i) {
        const int64_t base = runs[6 * i], units = runs[6 * i + 1], full = runs[6 * i + 2], kept = runs[6 * i + 3];
        const int64_t split = runs[6 * i + 4], skip = runs[6 * i + 5];
        if (base < 0 || units < 0 || full < 0 || kept < 0 || split < 0 || split > kept) return UNIQL_E_SHAPE;
        if (units * kept == 0) continue;
        const int64_t last_unit = base + (units - 1) * full;
        if (last_unit + split > n) return UNIQL_E_SHAPE;
        if (split < kept && (base + split + skip < 0 || last_unit + kept + skip > n)) return UNIQL_E_SHAPE;
        total += units * kept;
    }
    if (total <= 0 || n_pad <= 0 || n_pad < total || n_pad % 128 != 0 || n_scaled < 0) return UNIQL_E_SHAPE;
    if (!aligned16(B) || !aligned16(B_out)) return UNIQL_E_ALIGN;
    return cut_columns_launch(B, S, n, k, k_real, runs, n_runs, n_scaled, B_out, S_out, n_pad,
                              reinterpret_cast<hipStream_t>(stream));
}

int uniql_w4a16_cut_rows(const void* B, const void* S, int n, int k, int groups, int units, int full, int kept, int n_real,
                         void* B_out, void* S_out, int n_pad, void* stream) {
    const int rc = check_linear_shape(1, n, k, groups);
    if (rc != UNIQL_OK) return rc;
    if (!B || !S || !B_out || !S_out) return UNIQL_E_NULL;
    if (units < 1 || full < 0 || kept < 1 || (int64_t)(units - 1) * full + kept > k) return UNIQL_E_SHAPE;
    if (n_real < 1 || n_real > n || n_pad < n_real || n_pad % 128 != 0) return UNIQL_E_SHAPE;
    if ((int64_t)units * kept <= 128) return UNIQL_E_UNSUPPORTED;
    if ((int64_t)units * kept > 0x7fffffffLL - 128) return UNIQL_E_SHAPE;
    if (!aligned16(B) || !aligned16(B_out) || !aligned16(S_out)) return UNIQL_E_ALIGN;
    return cut_rows_launch(B, S, n, groups, units, full, kept, n_real, B_out, S_out, n_pad,
                           reinterpret_cast<hipStream_t>(stream));
}

int uniql_w4_embedding_lookup(const int64_t* ids, int64_t ntokens, const void* weight, const void* scales,
                              void* out, int64_t vocab, int dim, void* stream) {
    if (ntokens < 0 || vocab <= 0 || dim <= 0 || dim % 8 != 0) return UNIQL_E_SHAPE;
    if (ntokens == 0) return UNIQL_OK;
    if (!ids || !weight || !scales || !out) return UNIQL_E_NULL;
    if (!aligned16(out) || (reinterpret_cast<uintptr_t>(weight) & 3u)) return UNIQL_E_ALIGN;
    return embedding_launch(ids, ntokens, weight, scales, out, vocab, dim, reinterpret_cast<hipStream_t>(stream));
}

int uniql_w4_embedding_quantize(const void* W, int64_t ldw, void* packed, void* scales, int64_t vocab, int dim,
                                void* stream) {
    if (vocab < 0 || dim <= 0 || dim % 8 != 0 || ldw < dim || ldw % 8 != 0) return UNIQL_E_SHAPE;
    if (vocab == 0) return UNIQL_OK;
    if (!W || !packed || !scales) return UNIQL_E_NULL;
    if (!aligned16(W) || (reinterpret_cast<uintptr_t>(packed) & 3u)) return UNIQL_E_ALIGN;
    return embedding_quantize_launch(W, ldw, packed, scales, vocab, dim, reinterpret_cast<hipStream_t>(stream));
}

int uniql_rope_indices(void* q, int64_t q_row_stride, void* k, int64_t k_row_stride, const void* cos,
                       const void* sin, int64_t cos_row_stride, const void* indices, int index_bytes, int64_t rows,
                       int seq_len, int cos_batch, int n_q_heads, int n_kv_heads, int head_dim, int cos_dim,
                       void* stream) {
    if (rows < 0 || seq_len < 0 || n_q_heads <= 0 || n_kv_heads <= 0 || head_dim <= 0 || cos_dim <= 0)
        return UNIQL_E_SHAPE;
    if (seq_len == 0) return rows == 0 ? UNIQL_OK : UNIQL_E_SHAPE;  // no tokens: nothing to rotate
    if (head_dim % 2 != 0 || n_q_heads % n_kv_heads != 0) return UNIQL_E_SHAPE;
    if (index_bytes != 1 && index_bytes != 4 && index_bytes != 8) return UNIQL_E_UNSUPPORTED;
    if (index_bytes == 1 && cos_dim > 256) return UNIQL_E_SHAPE;
    if (cos_batch != 1 && (cos_batch <= 0 || rows != (int64_t)cos_batch * seq_len)) return UNIQL_E_SHAPE;
    if (cos_batch == 1 && rows % seq_len != 0) return UNIQL_E_SHAPE;
    if (q_row_stride < (int64_t)n_q_heads * head_dim || k_row_stride < (int64_t)n_kv_heads * head_dim ||
        cos_row_stride < cos_dim)
        return UNIQL_E_SHAPE;
    if (rows == 0) return UNIQL_OK;
    if (!q || !k || !cos || !sin || !indices) return UNIQL_E_NULL;
    return rope_indices_launch(q, q_row_stride, k, k_row_stride, cos, sin, cos_row_stride, indices, index_bytes,
                               rows, seq_len, cos_batch, n_q_heads, n_kv_heads, head_dim, cos_dim,
                               reinterpret_cast<hipStream_t>(stream));
}

int uniql_fwht(const void* x, void* y, int64_t rows, int dim, int block, float scale, int dtype, void* stream) {
    if (dtype != UNIQL_DT_F16 && dtype != UNIQL_DT_BF16 && dtype != UNIQL_DT_F32) return UNIQL_E_UNSUPPORTED;
    if (rows < 0 || dim <= 0 || !is_pow2(block) || block < 2 || block > 32768 || dim % block != 0)
        return UNIQL_E_SHAPE;
    if (rows == 0) return UNIQL_OK;
    if (!x || !y) return UNIQL_E_NULL;
    if (block == 128 && dtype == UNIQL_DT_F16 && (!aligned16(x) || !aligned16(y))) return UNIQL_E_ALIGN;
    return fwht_launch(x, y, rows, dim, block, scale, dtype, reinterpret_cast<hipStream_t>(stream));
}

int uniql_fwht_composite(const void* x, void* y, int64_t rows, int dim, int base, float scale, int dtype, void* stream) {
    if (dtype != UNIQL_DT_F16 && dtype != UNIQL_DT_BF16 && dtype != UNIQL_DT_F32) return UNIQL_E_UNSUPPORTED;
    if (base != 12 && base != 20 && base != 28 && base != 40) return UNIQL_E_UNSUPPORTED;
    if (rows < 0 || dim <= 0 || dim % base != 0 || !is_pow2(dim / base) || dim > 40960) return UNIQL_E_SHAPE;
    if (rows == 0) return UNIQL_OK;
    if (!x || !y) return UNIQL_E_NULL;
    return fwht_composite_launch(x, y, rows, dim, base, scale, dtype, reinterpret_cast<hipStream_t>(stream));
}

int uniql_fwht_columns(const void* x, void* y, int rows, int cols, float scale, int dtype, void* stream) {
    if (dtype != UNIQL_DT_F16 && dtype != UNIQL_DT_BF16 && dtype != UNIQL_DT_F32) return UNIQL_E_UNSUPPORTED;
    if (rows != 1024 && rows != 2048 && rows != 4096) return UNIQL_E_UNSUPPORTED;
    if (cols <= 0 || cols % 8 != 0) return UNIQL_E_SHAPE;
    if (!x || !y) return UNIQL_E_NULL;
    if (!aligned16(x) || !aligned16(y)) return UNIQL_E_ALIGN;
    return fwht_columns_launch(x, y, rows, cols, scale, dtype, reinterpret_cast<hipStream_t>(stream));
}

}  // extern "C"
