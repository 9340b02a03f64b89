// Walsh-Hadamard transform of fp16 / bf16 / fp32 rows: y = T((x . H_block) * scale), H the
// Sylvester (natural-order) matrix, applied to consecutive `block`-wide pieces.
// Butterflies run in fp32, lowest index bit first, one rounding to T at the end.
#include <algorithm>
#include <atomic>

#include "common.hpp"
#include "fwht_device.hpp"
#include "hadamard_base.hpp"

namespace uniql {

// ---- values in memory <-> fp32 ----------------------------------------------------------------
// Eight consecutive values as raw 16-byte words (fp32: two of them), so that a load can be issued long before the
// conversion; results are rounded once (see scaled_to_half: multiply and rounding stay separate).
template <typename T>
struct RowIo;
template <>
struct RowIo<half_t> {
    struct Raw { u32x4 a; };
    static __device__ __forceinline__ Raw load(const half_t* p) { return Raw{*reinterpret_cast<const u32x4*>(p)}; }
    static __device__ __forceinline__ Raw load(__amdgpu_buffer_rsrc_t rsrc, unsigned bytes) {
        return Raw{__builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, bytes, 0, 0))};
    }
    static __device__ __forceinline__ void settle(Raw& r) { asm volatile("" : "+v"(r.a)); }
    static __device__ __forceinline__ void unpack(const Raw& r, float (&f)[8]) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const h2 hv = bits_to_h2(r.a[p]);
            f[2 * p] = (float)hv.x;
            f[2 * p + 1] = (float)hv.y;
        }
    }
    static __device__ __forceinline__ uint32_t pair(float a, float b, float scale) {
        h2 r;
        r.x = scaled_to_half(a, scale);
        r.y = scaled_to_half(b, scale);
        return h2_to_bits(r);
    }
    static __device__ __forceinline__ void store2(half_t* p, float a, float b, float scale) {
        *reinterpret_cast<uint32_t*>(p) = pair(a, b, scale);
    }
    static __device__ __forceinline__ void store4(half_t* p, f4 f, float scale) {
        *reinterpret_cast<uint2*>(p) = make_uint2(pair(f[0], f[1], scale), pair(f[2], f[3], scale));
    }
    static __device__ __forceinline__ void store8(half_t* p, const float (&f)[8], float scale) {
        *reinterpret_cast<u32x4*>(p) =
            u32x4{pair(f[0], f[1], scale), pair(f[2], f[3], scale), pair(f[4], f[5], scale), pair(f[6], f[7], scale)};
    }
};
template <>
struct RowIo<__bf16> {
    struct Raw { u32x4 a; };
    static __device__ __forceinline__ Raw load(const __bf16* p) { return Raw{*reinterpret_cast<const u32x4*>(p)}; }
    static __device__ __forceinline__ Raw load(__amdgpu_buffer_rsrc_t rsrc, unsigned bytes) {
        return Raw{__builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, bytes, 0, 0))};
    }
    static __device__ __forceinline__ void settle(Raw& r) { asm volatile("" : "+v"(r.a)); }
    static __device__ __forceinline__ void unpack(const Raw& r, float (&f)[8]) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            f[2 * p] = __uint_as_float(r.a[p] << 16);
            f[2 * p + 1] = __uint_as_float(r.a[p] & 0xffff0000u);
        }
    }
    static __device__ __forceinline__ uint32_t pair(float a, float b, float scale) {
        float p = a * scale, q = b * scale;
        asm volatile("" : "+v"(p), "+v"(q));
        const __bf16 lo = (__bf16)p, hi = (__bf16)q;
        return (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
    }
    static __device__ __forceinline__ void store2(__bf16* p, float a, float b, float scale) {
        *reinterpret_cast<uint32_t*>(p) = pair(a, b, scale);
    }
    static __device__ __forceinline__ void store4(__bf16* p, f4 f, float scale) {
        *reinterpret_cast<uint2*>(p) = make_uint2(pair(f[0], f[1], scale), pair(f[2], f[3], scale));
    }
    static __device__ __forceinline__ void store8(__bf16* p, const float (&f)[8], float scale) {
        *reinterpret_cast<u32x4*>(p) =
            u32x4{pair(f[0], f[1], scale), pair(f[2], f[3], scale), pair(f[4], f[5], scale), pair(f[6], f[7], scale)};
    }
};
template <>
struct RowIo<float> {
    struct Raw { f4 a, b; };
    static __device__ __forceinline__ Raw load(const float* p) {
        return Raw{*reinterpret_cast<const f4*>(p), *reinterpret_cast<const f4*>(p + 4)};
    }
    static __device__ __forceinline__ Raw load(__amdgpu_buffer_rsrc_t rsrc, unsigned bytes) {
        return Raw{__builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, bytes, 0, 0)),
                   __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, bytes + 16, 0, 0))};
    }
    static __device__ __forceinline__ void settle(Raw& r) { asm volatile("" : "+v"(r.a), "+v"(r.b)); }
    static __device__ __forceinline__ void unpack(const Raw& r, float (&f)[8]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[i] = r.a[i];
            f[4 + i] = r.b[i];
        }
    }
    static __device__ __forceinline__ void store2(float* p, float a, float b, float scale) {
        *reinterpret_cast<float2*>(p) = make_float2(a * scale, b * scale);
    }
    static __device__ __forceinline__ void store4(float* p, f4 f, float scale) { *reinterpret_cast<f4*>(p) = f * scale; }
    static __device__ __forceinline__ void store8(float* p, const float (&f)[8], float scale) {
        *reinterpret_cast<f4*>(p) = f4{f[0] * scale, f[1] * scale, f[2] * scale, f[3] * scale};
        *reinterpret_cast<f4*>(p + 4) = f4{f[4] * scale, f[5] * scale, f[6] * scale, f[7] * scale};
    }
};

// index bits 0..2 of eight consecutive values
__device__ __forceinline__ void wht8(float (&f)[8]) {
#pragma unroll
    for (int h = 1; h < 8; h <<= 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if ((i & h) == 0) {
                const float p = f[i], q = f[i + h];
                f[i] = p + q;
                f[i + h] = p - q;
            }
        }
    }
}

// ---- block == 128: one 16-lane group per piece, all in registers ------------------
template <typename T>
__global__ __launch_bounds__(256) void fwht128_kernel(const T* __restrict__ x, T* __restrict__ y, int64_t pieces, float scale) {
    const int64_t piece = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    const int seg = threadIdx.x & 15;
    // every lane of a 16-lane group shares `piece`, so the exchange below never
    // crosses into a group that has left
    if (piece >= pieces) return;
    float f[8];
    RowIo<T>::unpack(RowIo<T>::load(x + (piece * 16 + seg) * 8), f);
    wht128_row16(f, seg);
    RowIo<T>::store8(y + (piece * 16 + seg) * 8, f, scale);
}

// ---- general power of two: one workgroup per piece, fp32 image in LDS --------------
// A pass handles CNT consecutive index bits starting at bit `lo`: each task gathers
// 2^CNT values whose indices differ only in those bits, runs CNT butterfly stages in
// registers and scatters them back.
template <int CNT>
__device__ __forceinline__ void fwht_pass(float* buf, int L, int lo, int tid, int nthreads) {
    constexpr int E = 1 << CNT;
    const int tasks = L >> CNT;
    const int lowmask = (1 << lo) - 1;
    for (int t = tid; t < tasks; t += nthreads) {
        const int base = ((t >> lo) << (lo + CNT)) | (t & lowmask);
        float v[E];
#pragma unroll
        for (int i = 0; i < E; ++i) v[i] = buf[base + (i << lo)];
#pragma unroll
        for (int h = 1; h < E; h <<= 1) {
#pragma unroll
            for (int i = 0; i < E; ++i) {
                if ((i & h) == 0) {
                    const float p = v[i], q = v[i + h];
                    v[i] = p + q;
                    v[i + h] = p - q;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < E; ++i) buf[base + (i << lo)] = v[i];
    }
}

template <typename T>
__global__ __launch_bounds__(256) void fwht_lds_kernel(const T* __restrict__ x, T* __restrict__ y, int L,
                                                      int log2L, float scale) {
    extern __shared__ __attribute__((aligned(16))) float fbuf[];
    const int tid = threadIdx.x;
    const T* xp = x + (size_t)blockIdx.x * L;
    T* yp = y + (size_t)blockIdx.x * L;
    for (int i = tid; i < L; i += 256) fbuf[i] = (float)xp[i];
    __syncthreads();
    int lo = 0;
    while (lo < log2L) {
        const int left = log2L - lo;
        if (left >= 3) {
            fwht_pass<3>(fbuf, L, lo, tid, 256);
            lo += 3;
        } else if (left == 2) {
            fwht_pass<2>(fbuf, L, lo, tid, 256);
            lo += 2;
        } else {
            fwht_pass<1>(fbuf, L, lo, tid, 256);
            lo += 1;
        }
        __syncthreads();
    }
    for (int i = tid; i < L; i += 256) {
        float p = fbuf[i] * scale;
        asm volatile("" : "+v"(p));  // see scaled_to_half: keep multiply and rounding separate
        yp[i] = (T)p;
    }
}

// ---- 256 and 512: vector loads, index bits 0..2 in registers, LDS passes of
// up to four bits, vector stores ----------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void fwht_vec_kernel(const T* __restrict__ x, T* __restrict__ y, int L, int log2L, float scale) {
    extern __shared__ __attribute__((aligned(16))) float fbuf[];
    const int tid = threadIdx.x, nthreads = blockDim.x;
    const int chunks = L >> 3;
    const T* xp = x + (size_t)blockIdx.x * L;
    T* yp = y + (size_t)blockIdx.x * L;
    for (int c = tid; c < chunks; c += nthreads) {
        float f[8];
        RowIo<T>::unpack(RowIo<T>::load(xp + 8 * c), f);
        wht8(f);
        float* dst = fbuf + fwht_pad(8 * c);
        *reinterpret_cast<f4*>(dst) = f4{f[0], f[1], f[2], f[3]};
        *reinterpret_cast<f4*>(dst + 4) = f4{f[4], f[5], f[6], f[7]};
    }
    __syncthreads();
    fwht_passes_from_bit3(fbuf, 1, 0, L, log2L, tid, nthreads);
    for (int c = tid; c < chunks; c += nthreads) {
        const float* src = fbuf + fwht_pad(8 * c);
        const f4 a = *reinterpret_cast<const f4*>(src), b = *reinterpret_cast<const f4*>(src + 4);
        const float f[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        RowIo<T>::store8(yp + 8 * c, f, scale);
    }
}

// Barriers that order LDS alone: loads from and stores to memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
__device__ __forceinline__ void lds_wave_fence() {  // a wave's LDS operations complete in issue order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Eight floats of padding per 64: the 64 lanes of either pass touch every bank once.
__device__ __forceinline__ int fwht_pad8of64(int idx) { return idx + ((idx >> 6) << 3); }

// Index bits 3..5 of 512 values that lie eight to a lane, in an LDS pass of two fenced steps: on entry f holds values 8 piece ..
// (bits 0..2 done, every piece on one lane), behind it f[e] is value lane + 64 e.  buf: 576 floats of the wave's own.
__device__ __forceinline__ void wht512_put(float* buf, int piece, const float (&f)[8]) {
    float* d = buf + fwht_pad8of64(8 * piece);
    *reinterpret_cast<f4*>(d) = f4{f[0], f[1], f[2], f[3]};
    *reinterpret_cast<f4*>(d + 4) = f4{f[4], f[5], f[6], f[7]};
}
__device__ __forceinline__ void wht512_middle(float* buf, int lane, float (&f)[8]) {
    float* d = buf + 72 * (lane >> 3) + (lane & 7);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = d[8 * e];
    wht8(f);
#pragma unroll
    for (int e = 0; e < 8; ++e) d[8 * e] = f[e];
}
__device__ __forceinline__ void wht512_get(const float* buf, int lane, float (&f)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = buf[lane + 72 * e];
}
__device__ __forceinline__ void wht512_pass3(float* buf, int piece, int lane, float (&f)[8]) {
    wht512_put(buf, piece, f);
    lds_wave_fence();
    wht512_middle(buf, lane, f);
    lds_wave_fence();
    wht512_get(buf, lane, f);
}
// Bits 6.. of f[e] as far as a chunk of P values has them.
__device__ __forceinline__ void wht512_upper(float (&f)[8], int P) {
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        if ((64 << b) >= P) break;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if ((e & (1 << b)) == 0) {
                const float p = f[e], q = f[e + (1 << b)];
                f[e] = p + q;
                f[e + (1 << b)] = p - q;
            }
    }
}

// Long rows, 1024 to 32768 values.  A wave takes one, two or four neighbouring blocks of 512 values: 16-byte loads and index
// bits 0..2 in registers, bits 3..5 and 6..8 in LDS passes of its own, bits 9 and 10 in registers again, no workgroup
// barrier; then, behind one, the one to four bits that lie across the waves: a thread reads two or four neighbouring values at
// the waves' strides, transforms, scales, rounds and stores them.  Bits in ascending order like everywhere else: the same
// bits.  The workgroups stay and request their next row ahead of the last step.
// What bounds it: memory (16384 rows of 4096: 5.9 TB/s), and for few rows the latency of load, passes and store.  fp16, cold,
// against one workgroup a row with a workgroup barrier behind every pass: one row of 4096 4.6 -> 2.8 us, of 16384 7.7 -> 4.4;
// 1024 rows of 1024 3.4 -> 3.2, of 4096 7.3 -> 5.9, of 8192 11.0 -> 9.7, of 16384 23.2 -> 16.5, of 32768 45 -> 31; 4096 rows
// of 4096 18.4 -> 15.5, of 16384 72 -> 50.
template <int LOG2L>
struct RowShape {
    static constexpr int kBlocks = LOG2L <= 11 ? 1 : LOG2L == 12 ? 2 : 4;               // of 512 values, a wave
    static constexpr int kWaves = (1 << LOG2L) / (512 * kBlocks);
    static constexpr size_t kBytes = (size_t)(1 << LOG2L) / 8 * 9 * sizeof(float);
};

template <typename T, int LOG2L>
__global__ __launch_bounds__(64 * RowShape<LOG2L>::kWaves, 4) void fwht_rows_kernel(const T* __restrict__ x, T* __restrict__ y, int rows, float scale) {
    extern __shared__ __attribute__((aligned(16))) float fbuf[];
    constexpr int L = 1 << LOG2L, NB = RowShape<LOG2L>::kBlocks, W = RowShape<LOG2L>::kWaves, kSpan = 512 * NB;
    constexpr int V = LOG2L == 11 || W == 16 ? 2 : 4;  // neighbouring values of a thread in the last step
    typedef float fv __attribute__((ext_vector_type(V)));
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    typename RowIo<T>::Raw v[NB];
    auto request = [&](int row) __attribute__((always_inline)) {  // a row that does not exist: beyond the descriptor
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<T*>(x + (size_t)(row < rows ? row : 0) * L), 0, row < rows ? (unsigned)(L * sizeof(T)) : 0u, 0x00020000);
#pragma unroll
        for (int i = 0; i < NB; ++i) v[i] = RowIo<T>::load(rsrc, (unsigned)((kSpan * w + 512 * i + 8 * lane) * sizeof(T)));
    };
    float* const mine = fbuf + 576 * NB * w;
    int row = blockIdx.x;
    request(row);
    while (true) {
        float f[NB][8];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            RowIo<T>::unpack(v[i], f[i]);
            wht8(f[i]);
            wht512_put(mine + 576 * i, lane, f[i]);
        }
        lds_wave_fence();
#pragma unroll
        for (int i = 0; i < NB; ++i) wht512_middle(mine + 576 * i, lane, f[i]);
        lds_wave_fence();
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            wht512_get(mine + 576 * i, lane, f[i]);
            wht512_upper(f[i], 512);
        }
#pragma unroll
        for (int h = 1; h < NB; h <<= 1)
#pragma unroll
            for (int i = 0; i < NB; ++i)
                if ((i & h) == 0)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float p = f[i][e], q = f[i + h][e];
                        f[i][e] = p + q;
                        f[i + h][e] = p - q;
                    }
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) mine[576 * i + lane + 72 * e] = f[i][e];
        const int next = row + gridDim.x;
        request(next);
        lds_barrier();
        T* const yp = y + (size_t)row * L;
#pragma unroll
        for (int t = 0; t < kSpan / (V * 64 * W); ++t) {
            const int col = V * ((int)threadIdx.x + 64 * W * t);
            fv g[W];
#pragma unroll
            for (int j = 0; j < W; ++j) g[j] = *reinterpret_cast<const fv*>(fbuf + 576 * NB * j + fwht_pad8of64(col));
#pragma unroll
            for (int h = 1; h < W; h <<= 1)
#pragma unroll
                for (int j = 0; j < W; ++j)
                    if ((j & h) == 0) {
                        const fv p = g[j], q = g[j + h];
                        g[j] = p + q;
                        g[j + h] = p - q;
                    }
            // the next row has arrived by now; waited for behind the stores, it would be waited for with them
#pragma unroll
            for (int i = 0; i < NB; ++i) RowIo<T>::settle(v[i]);
#pragma unroll
            for (int j = 0; j < W; ++j) {
                if constexpr (V == 4) RowIo<T>::store4(yp + kSpan * j + col, g[j], scale);
                else RowIo<T>::store2(yp + kSpan * j + col, g[j][0], g[j][1], scale);
            }
        }
        if (next >= rows) break;
        row = next;
        lds_barrier();  // the next row overwrites what other waves may still be reading
    }
}

// more than 64 KiB of LDS, for calls that launch one kernel: set on its first launch on a device
template <typename K>
static bool allow_lds(K kern, size_t bytes, std::atomic<unsigned long long>& done) {
    if (bytes <= 64 * 1024) return true;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    const unsigned long long bit = dev < 64 ? 1ull << dev : 0ull;
    if (done.load(std::memory_order_acquire) & bit) return true;
    if (!allow_lds(kern, 160 * 1024)) return false;
    done.fetch_or(bit, std::memory_order_release);
    return true;
}

template <typename T, int LOG2L>
static bool fwht_rows_allow_lds() {
    static std::atomic<unsigned long long> done{0};
    return allow_lds(&fwht_rows_kernel<T, LOG2L>, RowShape<LOG2L>::kBytes, done);
}
// the rotations in front of a layer's product
bool fwht_allow_lds() { return fwht_rows_allow_lds<half_t, 14>() && fwht_rows_allow_lds<half_t, 15>(); }

template <typename T, int LOG2L>
static int fwht_rows_go(const void* x, void* y, int64_t rows, float scale, hipStream_t stream) {
    using S = RowShape<LOG2L>;
    if (!fwht_rows_allow_lds<T, LOG2L>()) return UNIQL_E_LAUNCH;
    // The workgroups that the chip holds at once, by registers.  fp32 rows of 4096 and more each get their own: memory is
    // busy without the request ahead, and rows in launch order use it better (16384 rows of 8192: 199 us, 207 with
    // workgroups that stay; fp16 102 either way).
    const int64_t resident = 256 * ((LOG2L <= 12 && sizeof(T) == 2 ? 32 : 16) / S::kWaves);
    const int64_t grid = sizeof(T) == 4 && LOG2L >= 12 ? rows : std::min(rows, resident);
    hipLaunchKernelGGL((fwht_rows_kernel<T, LOG2L>), dim3((unsigned)grid), dim3(64 * S::kWaves), S::kBytes, stream,
                       reinterpret_cast<const T*>(x), reinterpret_cast<T*>(y), (int)rows, scale);
    return UNIQL_OK;
}

template <typename T>
static int fwht_vec_launch(const void* x, void* y, int64_t pieces, int block, float scale, hipStream_t stream) {
    int log2L = 0;
    while ((1 << log2L) < block) ++log2L;
    const size_t shmem = (size_t)(block + (block >> 7) * 8) * sizeof(float);
    switch (log2L) {
        case 10: return fwht_rows_go<T, 10>(x, y, pieces, scale, stream);
        case 11: return fwht_rows_go<T, 11>(x, y, pieces, scale, stream);
        case 12: return fwht_rows_go<T, 12>(x, y, pieces, scale, stream);
        case 13: return fwht_rows_go<T, 13>(x, y, pieces, scale, stream);
        case 14: return fwht_rows_go<T, 14>(x, y, pieces, scale, stream);
        case 15: return fwht_rows_go<T, 15>(x, y, pieces, scale, stream);
        default: break;
    }
    hipLaunchKernelGGL(fwht_vec_kernel<T>, dim3((unsigned)pieces), dim3(block / 8), shmem, stream,
                       reinterpret_cast<const T*>(x), reinterpret_cast<T*>(y), block, log2L, scale);
    return UNIQL_OK;
}

// ---- down the columns of a row-major matrix: y = T((H_L . x) * scale), L = 1024, 2048 or 4096 rows ------------
// The output side of a weight rotation without the two transposed copies around the row transform.  A workgroup
// takes 4096 WAVES / L neighbouring columns over all rows, 64 values a thread, and reads and writes a value once:
//   load    a thread reads eight consecutive rows x eight columns (16 bytes of fp16 per row), neighbouring lanes the
//           neighbouring columns of a row: index bits 0..2;
//   wave    the next bits lie inside a wave: column by column through a few KB of LDS, no workgroup barrier;
//   last    the remaining bits lie across the waves: half of the values at a time through LDS, scaled, rounded, stored.
// Same butterfly order as the row transform: the same values as transposing twice.  Neighbouring tiles share cache lines: the
// tiles of one XCD (workgroups i, i + 8, i + 16, ...) are neighbours, and run at the same time, so a line is fetched and
// written back once per second-level cache.
// What bounds it: the second-level cache's requests, one for every 16 to 64 bytes of a row that a tile is wide (4096 x 14336
// fp16 as 8 columns a tile: 14.7 M of them, 55 us of the caches' request rate), and load, passes and store following each
// other inside a workgroup; so tiles are wide, and
// two workgroups share a compute unit where a tile has eight waves.  fp16, cold, against one workgroup of 136 KB and 4-byte
// stores: 4096 x 14336 125 -> 101 us, 4096 x 4096 29 -> 25, 1024 x 14336 20.5 -> 17.1.
// Three heights: the power-of-two output widths of the projections it rotates; others go through the copies.
template <int LOG2L, int WAVES>
struct ColumnTile {
    static constexpr int kColumns = (4096 * WAVES) >> LOG2L;
    static constexpr int CB = (WAVES == 16 ? 4 : WAVES == 8 ? 3 : 2) + 9 - LOG2L;  // log2 of the chunks of eight columns
    static constexpr int kRowsInWave = 512 >> CB;
    // the last exchange, half of a wave's values: 64 << kRowBits rows x kHalfChunks chunks
    static constexpr int kRowBits = CB < 2 ? 2 - CB : 0, kHalfChunks = CB < 2 ? 1 << CB : 4;
    static constexpr int kStride = WAVES * 8 * kHalfChunks + 4;  // floats per row
    static constexpr size_t kPasses = WAVES * 4 * 576 * sizeof(float), kLast = (size_t)(64 << kRowBits) * kStride * sizeof(float);
    static constexpr size_t kBytes = kPasses > kLast ? kPasses : kLast;
};

template <typename T, int LOG2L, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 4) void fwht_columns_kernel(const T* __restrict__ x, T* __restrict__ y, int cols, int tiles, float scale) {
    extern __shared__ __attribute__((aligned(16))) float fbuf[];
    using Tile = ColumnTile<LOG2L, WAVES>;
    constexpr int CB = Tile::CB, RIW = Tile::kRowsInWave, RB = Tile::kRowBits, HC = Tile::kHalfChunks;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per_xcd = (tiles + 7) >> 3;
    const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tile >= tiles) return;  // uniform
    const int col0 = tile * Tile::kColumns;
    const int chunk = lane & ((1 << CB) - 1), rows8 = lane >> CB;
    float f[8][8];  // [row, later what the wave's passes leave][column]
    {
        typename RowIo<T>::Raw raw[8];
        // (cols is a multiple of eight: a chunk exists or it does not, and then stands in for the tile's first)
        const int col = col0 + 8 * chunk < cols ? col0 + 8 * chunk : col0;
        const T* src = x + (size_t)(RIW * w + 8 * rows8) * cols + col;
#pragma unroll
        for (int i = 0; i < 8; ++i) raw[i] = RowIo<T>::load(src + (size_t)i * cols);
#pragma unroll
        for (int i = 0; i < 8; ++i) RowIo<T>::unpack(raw[i], f[i]);
    }
    // A wave's values of column e of every chunk: chunk by chunk RIW rows, 512 in all.
    float* own = fbuf + w * (4 * 576);
    const int piece = (chunk << (6 - CB)) | rows8;
#pragma unroll
    for (int e0 = 0; e0 < 8; e0 += 4) {
#pragma unroll
        for (int e = e0; e < e0 + 4; ++e) {
            float g[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) g[i] = f[i][e];
            wht8(g);
            wht512_pass3(own + (e - e0) * 576, piece, lane, g);
            wht512_upper(g, RIW);
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i][e] = g[i];
        }
        lds_wave_fence();
    }
    // f[k][e]: value lane + 64 k.  The halves: rows with bit 6 clear and set, or, where k counts eight chunks, four of them each.
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        lds_barrier();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float (&r)[8] = f[CB < 3 ? 2 * q + half : 4 * half + q];
            float* dst = fbuf + (lane + 64 * (q & ((1 << RB) - 1))) * Tile::kStride + (w * HC + (q >> RB)) * 8;
            *reinterpret_cast<f4*>(dst) = f4{r[0], r[1], r[2], r[3]};
            *reinterpret_cast<f4*>(dst + 4) = f4{r[4], r[5], r[6], r[7]};
        }
        lds_barrier();
        // an item: a row, four columns; 512 of them in a half (sixteen waves: the halves go to one half of the threads each)
        for (int item = WAVES == 16 ? tid - 512 * half : tid; item >= 0 && item < 512; item += 64 * WAVES) {
            const int quad = item & (2 * HC - 1), at = item / (2 * HC);
            const int c = 4 * quad + (CB < 3 ? 0 : 32 * half);
            if (col0 + c >= cols) continue;
            f4 v[WAVES];
#pragma unroll
            for (int r = 0; r < WAVES; ++r) v[r] = *reinterpret_cast<const f4*>(fbuf + at * Tile::kStride + r * 8 * HC + 4 * quad);
#pragma unroll
            for (int h = 1; h < WAVES; h <<= 1)
#pragma unroll
                for (int r = 0; r < WAVES; ++r)
                    if ((r & h) == 0) {
                        const f4 p = v[r], q = v[r + h];
                        v[r] = p + q;
                        v[r + h] = p - q;
                    }
            const int row = CB < 3 ? (at & 63) + 64 * half + 128 * (at >> 6) : at;
            T* out = y + (size_t)row * cols + col0 + c;
#pragma unroll
            for (int r = 0; r < WAVES; ++r) RowIo<T>::store4(out + (size_t)(RIW * r) * cols, v[r], scale);
        }
    }
}

// The same over 4096 rows for 16-bit values, two chunks of eight columns a workgroup, one after the other.  Eight columns are
// 16 bytes of a row, and the caches' requests for those were what bound the tiles above; here neighbouring lanes read and
// write neighbouring chunks of a row, 32 bytes a request, and swap halves: a wave then holds one chunk of its 512 rows in
// fp32, as above, and the other as it was read, later the first one's results, rounded.  That is all the registers of two
// workgroups a compute unit, hence the empty asm statements (values packed, and columns finished, where they are written) and
// the scheduling barriers: without them 40 to 70 registers spill.
// What bounds it now: load, passes and stores follow each other in all workgroups at once.  fp16, cold, us with eight columns and
// with sixteen: 4096 x 4096 35.7 -> 28.9, x 8192 82.4 -> 54.8, x 11008 98 -> 64, x 14336 103.5 -> 82.0.
__device__ __forceinline__ void swap_neighbours(bool odd, uint32_t& a, uint32_t& b) {  // an even lane's b for the next lane's a
    const uint32_t mine = odd ? a : b;
    const uint32_t other = (uint32_t)__builtin_amdgcn_mov_dpp((int)mine, 0xB1, 0xF, 0xF, true);  // lane ^ 1
    a = odd ? other : a;
    b = odd ? b : other;
}

template <typename T>
__global__ __launch_bounds__(512, 4) void fwht_column_pairs_kernel(const T* __restrict__ x, T* __restrict__ y, int cols, int tiles, float scale) {
    extern __shared__ __attribute__((aligned(16))) float fbuf[];
    using Tile = ColumnTile<12, 8>;
    constexpr int kFlight = 2;  // columns of a wave in LDS together
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per_xcd = (tiles + 7) >> 3;
    const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tile >= tiles) return;  // uniform
    const int col0 = tile * 16;
    const bool odd = lane & 1, second = col0 + 8 < cols;  // cols is a multiple of eight
    u32x4 chunk[2][8];  // [.. of eight columns][row 8 lane + ..]
    {
        const char* src = reinterpret_cast<const char*>(x + (size_t)(512 * w) * cols + col0);
        const uint32_t mine = 16u * ((uint32_t)(lane & ~1) * (uint32_t)cols + (odd && second ? 1u : 0u));  // bytes
#pragma unroll
        for (int i = 0; i < 16; ++i) chunk[i >> 3][i & 7] = *reinterpret_cast<const u32x4*>(src + (size_t)i * cols * sizeof(T) + mine);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t a = chunk[0][i][j], b = chunk[1][i][j];
            swap_neighbours(odd, a, b);
            chunk[0][i][j] = a;
            chunk[1][i][j] = b;
        }
    __builtin_amdgcn_sched_barrier(0);
    float* own = fbuf + w * (kFlight * 576);
    const int quad = tid & 1, at = tid >> 1;
    const uint32_t out = quad == 1 && !second ? 0xfffffff0u : 2u * (((uint32_t)(at & 63) + 128 * (uint32_t)(at >> 6)) * (uint32_t)cols + 8 * (uint32_t)quad);  // bytes
    uint32_t kept[2][8][2];  // the first chunk's results: [half][wave]
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        float f[8][8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            asm volatile("" : "+v"(chunk[c][i]));
            RowIo<T>::unpack(typename RowIo<T>::Raw{chunk[c][i]}, f[i]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (c == 1) lds_barrier();  // others may still be reading the first chunk's last half
#pragma unroll
        for (int e0 = 0; e0 < 8; e0 += kFlight) {
#pragma unroll
            for (int e = e0; e < e0 + kFlight; ++e) {
                float g[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) g[i] = f[i][e];
                wht8(g);
                wht512_pass3(own + (e - e0) * 576, lane, lane, g);
                wht512_upper(g, 512);
#pragma unroll
                for (int i = 0; i < 8; ++i) f[i][e] = g[i];
                asm volatile("" : "+v"(f[0][e]), "+v"(f[1][e]), "+v"(f[2][e]), "+v"(f[3][e]), "+v"(f[4][e]), "+v"(f[5][e]), "+v"(f[6][e]), "+v"(f[7][e]));
            }
            lds_wave_fence();
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            __builtin_amdgcn_sched_barrier(0);
            lds_barrier();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float (&r)[8] = f[2 * q + half];
                float* dst = fbuf + (lane + 64 * q) * Tile::kStride + w * 8;
                *reinterpret_cast<f4*>(dst) = f4{r[0], r[1], r[2], r[3]};
                *reinterpret_cast<f4*>(dst + 4) = f4{r[4], r[5], r[6], r[7]};
            }
            lds_barrier();
            f4 v[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) v[r] = *reinterpret_cast<const f4*>(fbuf + at * Tile::kStride + r * 8 + 4 * quad);
#pragma unroll
            for (int h = 1; h < 8; h <<= 1)
#pragma unroll
                for (int r = 0; r < 8; ++r)
                    if ((r & h) == 0) {
                        const f4 p = v[r], q = v[r + h];
                        v[r] = p + q;
                        v[r + h] = p - q;
                    }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                uint32_t lo = RowIo<T>::pair(v[r][0], v[r][1], scale), hi = RowIo<T>::pair(v[r][2], v[r][3], scale);
                if (c == 0) {
                    asm volatile("" : "+v"(lo), "+v"(hi));  // in 32 registers
                    kept[half][r][0] = lo;
                    kept[half][r][1] = hi;
                } else {
                    // an even thread has columns 0 .. 3 of both chunks, the next one 4 .. 7
                    swap_neighbours(odd, kept[half][r][0], lo);
                    swap_neighbours(odd, kept[half][r][1], hi);
                    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(y + (size_t)(512 * r + 64 * half) * cols + col0, 0, 0x7fffffff, 0x00020000);
                    __builtin_amdgcn_raw_buffer_store_b128(u32x4{kept[half][r][0], kept[half][r][1], lo, hi}, rows, out, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
}

template <typename T, int LOG2L, int WAVES>
static int fwht_columns_tiles(const void* x, void* y, int cols, float scale, hipStream_t stream) {
    using Tile = ColumnTile<LOG2L, WAVES>;
    static std::atomic<unsigned long long> done{0};
    if (!allow_lds(&fwht_columns_kernel<T, LOG2L, WAVES>, Tile::kBytes, done)) return UNIQL_E_LAUNCH;
    const int tiles = (cols + Tile::kColumns - 1) / Tile::kColumns;
    hipLaunchKernelGGL((fwht_columns_kernel<T, LOG2L, WAVES>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(64 * WAVES), Tile::kBytes, stream,
                       reinterpret_cast<const T*>(x), reinterpret_cast<T*>(y), cols, tiles, scale);
    return hipGetLastError() == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
}
template <typename T>
static int fwht_column_pairs(const void* x, void* y, int cols, float scale, hipStream_t stream) {
    static std::atomic<unsigned long long> done{0};
    constexpr size_t bytes = ColumnTile<12, 8>::kBytes;
    if (!allow_lds(&fwht_column_pairs_kernel<T>, bytes, done)) return UNIQL_E_LAUNCH;
    const int tiles = (cols + 15) / 16;
    hipLaunchKernelGGL(fwht_column_pairs_kernel<T>, dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(512), bytes, stream,
                       reinterpret_cast<const T*>(x), reinterpret_cast<T*>(y), cols, tiles, scale);
    return hipGetLastError() == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
}
template <typename T, int LOG2L>
static int fwht_columns_go(const void* x, void* y, int cols, float scale, hipStream_t stream) {
    // 16-bit values of 4096 rows in tiles of sixteen columns where those are faster from memory: us with eight columns and with
    // sixteen.  Not below 2560 columns, where they leave more than three in eight compute units idle (2048: 19.3 and 25.3; 2304: 23.7 and
    // 24.5; 2560: 28.2 and 27.4; 2816: 29.3 and 26.4; 3328: 30.1 and 26.6; 4096: 35.2 and 30.6), and not from 273 to 384 tiles, where a few
    // compute units get a second one (4352: 36.4 and 35.9; 4608: 41.7 and 42.9; 5120: 42.2 and 46.8; 6144: 48.8 and 51.0; 6152: 44.2 and
    // 38.4).  Further on the workgroups of a compute unit are out of step, and one tile more than there are places for costs nothing
    // that shows (8192, 512 tiles: 76.0 and 57.2; 8200: 54.9 and 55.5; 8448: 64.1 and 51.5; 9216: 68.3 and 58.4; 12296: 83.8 and 74.3; 16392:
    // 117.6 and 112.7).  A matrix that is in the caches with its result is a little faster in eight columns up to 4352 (2560: 21.5 and
    // 23.1; 3072: 21.8 and 23.3; 3328: 22.5 and 22.4; 4096: 24.2 and 24.6), not further on (7168: 38.4 and 33.4; 8192: 49.7 and 34.2).
    if constexpr (LOG2L == 12 && sizeof(T) == 2)
        if (cols >= 2560 && cols < (1 << 21) && !(cols > 4352 && cols <= 6144)) return fwht_column_pairs<T>(x, y, cols, scale, stream);
    // Else the widest tiles of which every compute unit gets one: eight waves, two workgroups a compute unit; sixteen for fp32
    // over 4096 rows, where eight columns are a full sector and only one workgroup's stores fit beside the other's loads
    // (4096 x 14336: 150 us against 165; fp16 102 either way); four for few columns of 1024 rows (x 4096: 8.5 us against 9.3).
    if (LOG2L == 12 && sizeof(T) == 4 && cols >= 256 * ColumnTile<LOG2L, 16>::kColumns) return fwht_columns_tiles<T, LOG2L, LOG2L == 12 && sizeof(T) == 4 ? 16 : 8>(x, y, cols, scale, stream);
    if (LOG2L == 10 && cols < 256 * ColumnTile<LOG2L, 8>::kColumns) return fwht_columns_tiles<T, LOG2L, LOG2L == 10 ? 4 : 8>(x, y, cols, scale, stream);
    return fwht_columns_tiles<T, LOG2L, 8>(x, y, cols, scale, stream);
}
template <typename T>
static int fwht_columns_rows(const void* x, void* y, int rows, int cols, float scale, hipStream_t stream) {
    switch (rows) {
        case 1024: return fwht_columns_go<T, 10>(x, y, cols, scale, stream);
        case 2048: return fwht_columns_go<T, 11>(x, y, cols, scale, stream);
        case 4096: return fwht_columns_go<T, 12>(x, y, cols, scale, stream);
        default: return UNIQL_E_UNSUPPORTED;
    }
}
int fwht_columns_launch(const void* x, void* y, int rows, int cols, float scale, int dtype, hipStream_t stream) {
    if (dtype == UNIQL_DT_F16) return fwht_columns_rows<half_t>(x, y, rows, cols, scale, stream);
    if (dtype == UNIQL_DT_BF16) return fwht_columns_rows<__bf16>(x, y, rows, cols, scale, stream);
    return fwht_columns_rows<float>(x, y, rows, cols, scale, stream);
}

// ---- composite widths: dim = BASE * P with P a power of two -----------------------------------
// The row is BASE chunks of P values: every chunk gets the P-point transform (LDS passes over
// the whole row touch only index bits below log2 P, so the chunks stay apart), then the BASE x BASE
// matrix combines the chunks: y[c P + i] = sum_c' z[c' P + i] H[c'][c], added in ascending c' in
// fp32; one rounding at the end.
template <typename T, int BASE>
__global__ __launch_bounds__(256) void fwht_composite_kernel(const T* __restrict__ x, T* __restrict__ y, int P,
                                                            int log2P, float scale) {
    extern __shared__ __attribute__((aligned(16))) float fbuf[];
    const uint64_t* table = BASE == 12 ? kHadamard12 : BASE == 20 ? kHadamard20 : BASE == 28 ? kHadamard28 : kHadamard40;
    const int tid = threadIdx.x;
    const int L = BASE * P;
    const T* xp = x + (size_t)blockIdx.x * L;
    T* yp = y + (size_t)blockIdx.x * L;
    for (int i = tid; i < L; i += 256) fbuf[i] = (float)xp[i];
    __syncthreads();
    int lo = 0;
    while (lo < log2P) {
        const int left = log2P - lo;
        if (left >= 3) {
            fwht_pass<3>(fbuf, L, lo, tid, 256);
            lo += 3;
        } else if (left == 2) {
            fwht_pass<2>(fbuf, L, lo, tid, 256);
            lo += 2;
        } else {
            fwht_pass<1>(fbuf, L, lo, tid, 256);
            lo += 1;
        }
        __syncthreads();
    }
    for (int i = tid; i < P; i += 256) {
        float z[BASE];
#pragma unroll
        for (int c = 0; c < BASE; ++c) z[c] = fbuf[c * P + i];
#pragma unroll
        for (int c = 0; c < BASE; ++c) {
            const uint64_t minus = table[c];
            float sum = 0.f;
#pragma unroll
            for (int cp = 0; cp < BASE; ++cp) sum += ((minus >> cp) & 1ull) ? -z[cp] : z[cp];
            float p = sum * scale;
            asm volatile("" : "+v"(p));  // see scaled_to_half: keep multiply and rounding separate
            yp[c * P + i] = (T)p;
        }
    }
}

// The same for P >= 128.  A wave transforms blocks of 512 consecutive values (whole chunks, or a half or quarter of one) by
// itself: 16-byte loads and index bits 0..2 in registers, bits 3..5 and 6..8 in two LDS passes without a workgroup barrier;
// chunks of more than 512 values have one or two bits left for the workgroup.  Then the base matrix across the chunks with
// its signs as constants, on pairs of neighbouring columns; the terms are added in ascending order, starting from zero, as
// fwht_composite_kernel does: the same bits.  Outputs whose first signs agree share the sums of those terms: with the outputs
// in the order of their signs, quarter by quarter, 644 additions a column in place of 784 (28), 1135 of 1600 (40), 335 of 400
// (20), 124 of 144 (12).
// What bounds it: the additions (a SIMD takes one of a wave in 2.4 clocks; the matrix unit's fp32 forms, tried, hold the
// vector unit up for as long as the additions take) and eight passes of the row through LDS, each about as long as the memory
// time, and at most two rows of 14336 in a compute unit's LDS to overlap them.  So the workgroups stay, and request their next
// row before they transform the current one.  fp16, one row a workgroup with a barrier behind every pass -> workgroups that
// stay -> shared sums: 1024 rows of 14336 20.9 -> 18.7 -> 18.2 us, 4096 rows 72 -> 66.3 -> 63.9; 4096 rows of 5120 (40 x 128)
// 30.7 -> 26.3 by the shared sums, of fp32 34.8 -> 32.6; one row of 14336 6.9 -> 6.2.
template <int BASE>
struct BaseTable;
template <> struct BaseTable<12> { static constexpr const uint64_t (&mask)[12] = kHadamard12; };
template <> struct BaseTable<20> { static constexpr const uint64_t (&mask)[20] = kHadamard20; };
template <> struct BaseTable<28> { static constexpr const uint64_t (&mask)[28] = kHadamard28; };
template <> struct BaseTable<40> { static constexpr const uint64_t (&mask)[40] = kHadamard40; };

// The outputs ordered by the signs of their terms, the first term's first: those whose sums begin alike are neighbours.
template <int BASE>
struct BaseOrder {
    int output[BASE];
    constexpr BaseOrder() : output() {
        for (int i = 0; i < BASE; ++i) {
            int at = i;
            for (; at > 0 && before(i, output[at - 1]); --at) output[at] = output[at - 1];
            output[at] = i;
        }
    }
    static constexpr bool minus(int c, int term) { return (BaseTable<BASE>::mask[c] >> term) & 1ull; }
    static constexpr bool before(int a, int b) {
        for (int t = 0; t < BASE; ++t)
            if (minus(a, t) != minus(b, t)) return minus(b, t);
        return false;
    }
    // of outputs lo .. hi - 1 in this order, which agree in the terms in front of `term`: the first that subtracts it
    constexpr int split(int lo, int hi, int term) const {
        while (lo < hi && !minus(output[lo], term)) ++lo;
        return lo;
    }
};
template <int BASE>
inline constexpr BaseOrder<BASE> kBaseOrder{};

// Outputs LO .. HI - 1 of that order, which agree in their first TERM terms: a, b are the sums of those.
template <typename T, int BASE, int LO, int HI, int TERM = 0>
__device__ __forceinline__ void base_outputs(const float2 (&z)[BASE], T* yp, int P, float scale, float a = 0.f, float b = 0.f) {
    if constexpr (TERM == BASE) {
        static_assert(HI - LO == 1);
        RowIo<T>::store2(yp + kBaseOrder<BASE>.output[LO] * P, a, b, scale);
    } else {
        constexpr int mid = kBaseOrder<BASE>.split(LO, HI, TERM);
        if constexpr (LO < mid) base_outputs<T, BASE, LO, mid, TERM + 1>(z, yp, P, scale, a + z[TERM].x, b + z[TERM].y);
        if constexpr (mid < HI) base_outputs<T, BASE, mid, HI, TERM + 1>(z, yp, P, scale, a - z[TERM].x, b - z[TERM].y);
    }
}

template <typename T, int BASE>
__global__ __launch_bounds__(512, BASE == 40 ? 3 : 4) void fwht_composite_vec_kernel(const T* __restrict__ x, T* __restrict__ y, int rows, int P, int log2P,
                                                                   float scale) {
    extern __shared__ __attribute__((aligned(16))) float fbuf[];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), W = blockDim.x >> 6;
    const int L = BASE * P, blocks = L >> 9;  // BASE is a multiple of four, P of 128
    constexpr int kAhead = sizeof(T) == 4 ? 2 : 4;  // blocks of a wave requested together
    typename RowIo<T>::Raw v[kAhead];
    // Always kAhead loads; blocks and rows that do not exist lie beyond the descriptor.
    auto request = [&](int row, int first) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<T*>(x + (size_t)(row < rows ? row : 0) * L), 0, row < rows ? (unsigned)(L * sizeof(T)) : 0u, 0x00020000);
#pragma unroll
        for (int i = 0; i < kAhead; ++i) v[i] = RowIo<T>::load(rsrc, (unsigned)((512 * (first + W * i) + 8 * lane) * sizeof(T)));
    };
    auto transform = [&](int first) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            const int block = first + W * i;
            if (block >= blocks) break;  // uniform
            float* buf = fbuf + 576 * block;
            float f[8];
            RowIo<T>::unpack(v[i], f);
            wht8(f);
            wht512_pass3(buf, lane, lane, f);
            wht512_upper(f, P);
#pragma unroll
            for (int e = 0; e < 8; ++e) buf[lane + 72 * e] = f[e];
        }
    };
    // quarters of the outputs of 128 columns, in order, an equal share to every wave
    const int tasks = P >> 5, t0 = w * tasks / W, t1 = (w + 1) * tasks / W;
    int row = blockIdx.x;
    request(row, w);
    while (true) {
        transform(w);
        for (int first = w + W * kAhead; first < blocks; first += W * kAhead) {
            request(row, first);
            transform(first);
        }
        const int next = row + gridDim.x;
        request(next, w);
        lds_barrier();
        for (int bit = 9; bit < log2P; ++bit) {
#pragma unroll 4
            for (int t = threadIdx.x; t < L >> 1; t += blockDim.x) {
                const int at = ((t >> bit) << (bit + 1)) | (t & ((1 << bit) - 1));
                float *p = fbuf + fwht_pad8of64(at), *q = p + (9 << (bit - 3));
                const float a = *p, b = *q;
                *p = a + b;
                *q = a - b;
            }
            lds_barrier();
        }
        for (int set = t0 >> 2; 4 * set < t1; ++set) {
            float2 z[BASE];
            const float* src = fbuf + 144 * set + fwht_pad8of64(2 * lane);
#pragma unroll
            for (int c = 0; c < BASE; ++c) z[c] = *reinterpret_cast<const float2*>(src + c * (P + (P >> 3)));
            // the next row has arrived by now; waited for behind the stores, it would be waited for with them
#pragma unroll
            for (int i = 0; i < kAhead; ++i) RowIo<T>::settle(v[i]);
            T* yp = y + (size_t)row * L + 128 * set + 2 * lane;
            auto mine = [&](int quarter) { return 4 * set + quarter >= t0 && 4 * set + quarter < t1; };  // uniform
            if (mine(0)) base_outputs<T, BASE, 0, BASE / 4>(z, yp, P, scale);
            if (mine(1)) base_outputs<T, BASE, BASE / 4, BASE / 2>(z, yp, P, scale);
            if (mine(2)) base_outputs<T, BASE, BASE / 2, BASE * 3 / 4>(z, yp, P, scale);
            if (mine(3)) base_outputs<T, BASE, BASE * 3 / 4, BASE>(z, yp, P, scale);
        }
        if (next >= rows) break;
        row = next;
        lds_barrier();  // the next row overwrites what other waves may still be reading
    }
}

// The vector kernels move 16 bytes at a time; rows that start elsewhere (a contiguous view with an offset) take the kernels
// that move single values.  Both give the same bits.
static bool rows_aligned(const void* x, const void* y) {
    return ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15u) == 0;
}

template <typename T, int BASE>
static int fwht_composite_go(const void* x, void* y, int64_t rows, int P, float scale, hipStream_t stream) {
    int log2P = 0;
    while ((1 << log2P) < P) ++log2P;
    const int L = BASE * P;
    const size_t image = (size_t)(L + (L >> 3)) * sizeof(float);
    if (P >= 128 && image <= 160 * 1024 && rows_aligned(x, y)) {
        static std::atomic<unsigned long long> done{0};
        if (!allow_lds(&fwht_composite_vec_kernel<T, BASE>, image, done)) return UNIQL_E_LAUNCH;
        // few waves where a row gives them little to do: several small workgroups instead (10240 = 40 x 256 at 4096 rows
        // 56 us with four waves, 71 with eight)
        const int waves = BASE == 12 ? (P == 128 ? 2 : P <= 512 ? 4 : 8) : P == 128 || (BASE == 40 && P == 256) ? 4 : 8;
        // the workgroups that the chip holds at once: registers for sixteen waves a compute unit, LDS
        const int64_t resident = 256 * std::min<int64_t>((BASE == 12 ? 20 : BASE == 40 ? 12 : 16) / waves, (int64_t)(160 * 1024 / image));
        hipLaunchKernelGGL((fwht_composite_vec_kernel<T, BASE>), dim3((unsigned)std::min(rows, resident)), dim3(64 * waves), image, stream,
                           reinterpret_cast<const T*>(x), reinterpret_cast<T*>(y), (int)rows, P, log2P, scale);
        return hipGetLastError() == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
    }
    const size_t shmem = (size_t)L * sizeof(float);
    static std::atomic<unsigned long long> done{0};
    if (!allow_lds(&fwht_composite_kernel<T, BASE>, shmem, done)) return UNIQL_E_LAUNCH;
    hipLaunchKernelGGL((fwht_composite_kernel<T, BASE>), dim3((unsigned)rows), dim3(256), shmem, stream,
                       reinterpret_cast<const T*>(x), reinterpret_cast<T*>(y), P, log2P, scale);
    return hipGetLastError() == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
}

template <typename T>
static int fwht_composite_base(const void* x, void* y, int64_t rows, int base, int P, float scale, hipStream_t stream) {
    switch (base) {
        case 12: return fwht_composite_go<T, 12>(x, y, rows, P, scale, stream);
        case 20: return fwht_composite_go<T, 20>(x, y, rows, P, scale, stream);
        case 28: return fwht_composite_go<T, 28>(x, y, rows, P, scale, stream);
        case 40: return fwht_composite_go<T, 40>(x, y, rows, P, scale, stream);
        default: return UNIQL_E_UNSUPPORTED;
    }
}

int fwht_composite_launch(const void* x, void* y, int64_t rows, int dim, int base, float scale, int dtype,
                          hipStream_t stream) {
    if (rows == 0) return UNIQL_OK;
    if (rows > 0x7fffffffLL) return UNIQL_E_SHAPE;
    const int P = dim / base;
    if (dtype == UNIQL_DT_F16) return fwht_composite_base<half_t>(x, y, rows, base, P, scale, stream);
    if (dtype == UNIQL_DT_BF16) return fwht_composite_base<__bf16>(x, y, rows, base, P, scale, stream);
    return fwht_composite_base<float>(x, y, rows, base, P, scale, stream);
}

template <typename T>
static int fwht_typed_launch(const void* x, void* y, int64_t pieces, int block, float scale, hipStream_t stream) {
    const bool vec = rows_aligned(x, y);
    if (block == 128 && vec) {
        const int64_t grid = (pieces + 15) / 16;
        if (grid > 0x7fffffffLL) return UNIQL_E_SHAPE;
        hipLaunchKernelGGL(fwht128_kernel<T>, dim3((unsigned)grid), dim3(256), 0, stream, reinterpret_cast<const T*>(x),
                           reinterpret_cast<T*>(y), pieces, scale);
        return UNIQL_OK;
    }
    if (pieces > 0x7fffffffLL) return UNIQL_E_SHAPE;
    if (block >= 256 && vec) return fwht_vec_launch<T>(x, y, pieces, block, scale, stream);
    int log2L = 0;
    while ((1 << log2L) < block) ++log2L;
    static std::atomic<unsigned long long> done{0};
    if (!allow_lds(&fwht_lds_kernel<T>, (size_t)block * sizeof(float), done)) return UNIQL_E_LAUNCH;
    hipLaunchKernelGGL((fwht_lds_kernel<T>), dim3((unsigned)pieces), dim3(256), (size_t)block * sizeof(float), stream,
                       reinterpret_cast<const T*>(x), reinterpret_cast<T*>(y), block, log2L, scale);
    return UNIQL_OK;
}

int fwht_launch(const void* x, void* y, int64_t rows, int dim, int block, float scale, int dtype,
                hipStream_t stream) {
    const int64_t pieces = rows * (dim / block);
    if (pieces == 0) return UNIQL_OK;
    const int rc = dtype == UNIQL_DT_F16    ? fwht_typed_launch<half_t>(x, y, pieces, block, scale, stream)
                   : dtype == UNIQL_DT_BF16 ? fwht_typed_launch<__bf16>(x, y, pieces, block, scale, stream)
                                            : fwht_typed_launch<float>(x, y, pieces, block, scale, stream);
    if (rc != UNIQL_OK) return rc;
    return hipGetLastError() == hipSuccess ? UNIQL_OK : UNIQL_E_LAUNCH;
}

}  // namespace uniql
