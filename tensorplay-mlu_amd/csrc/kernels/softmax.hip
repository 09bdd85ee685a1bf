// Fused softmax / log_softmax forward and backward for gfx950 (the
// reference's cnnlSoftmaxForward / cnnlSoftmaxBackward,
// tensorplay_mlu/csrc/ReduceKernels.cpp:171-199).
//
// Rows along the last axis (inner == 1) are held in registers: each row is
// read from HBM once and written once.  A configuration (WAVES, EPT) gives a
// row WAVES wavefronts and each thread EPT elements (EPT / N 16-byte
// packets), so rows up to 64 * WAVES * EPT elements stay on chip; up to 4
// waves per row, a 256-thread block holds 4 / WAVES rows, so several blocks
// share a CU.  The row max and the exponential sum combine across lanes with
// shuffles and across waves in LDS.  Rows past what 16 waves hold that way
// (large vocabularies) stay in the registers of a 512-thread block, two
// blocks a CU; still longer ones take a block-per-row kernel that keeps a
// running (max, sum) per thread over the row, then re-reads it to write the
// result.  Each of these kernels has an ANY form for rows that start at any
// element (a length that is not a whole number of packets, as 50257): its
// packets are unaligned 16-byte accesses, and the row's last D % N elements
// go one to a thread.  Softmax over a leading axis (inner > 1) walks the
// reduced axis with the contiguous inner axis across threads.
//
// The per-element arithmetic is kept short because for 16-bit storage it,
// not HBM, would set the pace: exponentials are 2^(d log2 e) on v_exp_f32
// with d = x - max formed first, the softmax quotient is one reciprocal per
// row, and results are packed with the hardware round-to-nearest-even
// conversions.

#include <cmath>
#include <type_traits>

#include "device_common.h"
#include "../allocator.h"
#include "../runtime.h"
#include "tp_amd_kernels.h"

namespace tp_amd {

namespace {

constexpr int kBlock = 256;
constexpr float kLog2e = 1.44269504088896340736f;

// e^d on v_exp_f32 (the softmax arguments d = x - max are <= 0, where its
// error stays within a few float32 ulps), as (2^(a/2))^2 with a = d log2 e:
// the instruction returns 0 for results below 2^-126, where the halves are
// still normal and their product underflows gradually, so an entry 88-103
// below its row's maximum keeps its subnormal value (bfloat16 has them).
__device__ __forceinline__ float exp_fast(float d) {
    const float h = __builtin_amdgcn_exp2f(d * (0.5f * kLog2e));
    return h * h;
}

__device__ __forceinline__ float wave_max(float v) {
    return wave_allreduce(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_sum(float v) {
    return wave_allreduce(v, [](float a, float b) { return a + b; });
}

// Layout of a (WAVES, EPT) configuration: WAVES <= 4 packs 4 / WAVES rows
// into a 256-thread block; more waves make one row per block.
template <int WAVES>
constexpr int block_threads() {
    return WAVES >= 4 ? WAVES * kWave : kBlock;
}
template <int WAVES>
constexpr int rows_per_block() {
    return WAVES >= 4 ? 1 : 4 / WAVES;
}

// Reduce ``v`` over the WAVES waves of this thread's row.  ``scratch`` holds
// one float per wave of the block.  Every wave of the block must call it.
template <int WAVES, bool MAX>
__device__ __forceinline__ float row_reduce(float v, float* scratch) {
    v = MAX ? wave_max(v) : wave_sum(v);
    if constexpr (WAVES > 1) {
        const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
        const int first = (wave / WAVES) * WAVES;
        __syncthreads();  // scratch may still be read from the previous use
        if (lane == 0) scratch[wave] = v;
        __syncthreads();
        const float t = lane < WAVES ? scratch[first + lane] : (MAX ? -INFINITY : 0.0f);
        v = MAX ? wave_max(t) : wave_sum(t);
    }
    return v;
}

template <typename T, int WAVES, int EPT, bool ANY>
__global__ __launch_bounds__(block_threads<WAVES>()) void softmax_rows_kernel(
    const typename Elem<T>::storage* x, typename Elem<T>::storage* y, int64_t rows, int64_t D,
    bool log) {
    constexpr int N = Packet<T>::N;
    constexpr int VPT = EPT / N;
    static_assert(VPT * N == EPT, "EPT must be a whole number of packets");
    constexpr int kThreads = WAVES * kWave;
    __shared__ float scratch[block_threads<WAVES>() / kWave];
    const int64_t row = static_cast<int64_t>(blockIdx.x) * rows_per_block<WAVES>() +
                        threadIdx.x / kThreads;
    const int tid = threadIdx.x % kThreads;
    const bool active = row < rows;  // uniform per wave
    const int64_t npk = D / N;
    const typename Elem<T>::storage* xr = x + (active ? row : 0) * D;
    float v[VPT][N];
    float m = -INFINITY;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int64_t q = tid + static_cast<int64_t>(k) * kThreads;
        if (active && q < npk) {
            unpack<T>(load_raw_stream<ANY>(xr + q * N), v[k]);
#pragma unroll
            for (int j = 0; j < N; ++j) m = fmaxf(m, v[k][j]);
        } else {
#pragma unroll
            for (int j = 0; j < N; ++j) v[k][j] = -INFINITY;
        }
    }
    const bool tail = ANY && active && tid < D - npk * N;  // one of the row's last D % N elements
    float t = -INFINITY;
    if (tail) {
        t = Elem<T>::load(xr[npk * N + tid]);
        m = fmaxf(m, t);
    }
    m = row_reduce<WAVES, true>(m, scratch);
    // A row of -inf (or an inactive one) would give inf - inf; exp(-inf - 0)
    // keeps it at 0 instead.
    const float shift = m == -INFINITY ? 0.0f : m;
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < VPT; ++k)
#pragma unroll
        for (int j = 0; j < N; ++j) {
            v[k][j] -= shift;
            const float e = exp_fast(v[k][j]);
            s += e;
            if (!log) v[k][j] = e;
        }
    if constexpr (ANY) {
        t -= shift;
        const float e = exp_fast(t);
        s += e;
        if (!log) t = e;
    }
    s = row_reduce<WAVES, false>(s, scratch);
    if (!active) return;
    const float lse = logf(s);
    const float inv = 1.0f / s;
    typename Elem<T>::storage* yr = y + row * D;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int64_t q = tid + static_cast<int64_t>(k) * kThreads;
        if (q < npk) {
            float o[N];
#pragma unroll
            for (int j = 0; j < N; ++j) o[j] = log ? v[k][j] - lse : v[k][j] * inv;
            store_raw_stream<ANY>(yr + q * N, pack<T>(o));
        }
    }
    if (tail) yr[npk * N + tid] = Elem<T>::store(log ? t - lse : t * inv);
}

// Rows that need a whole 16-wave block: one such block fills a CU, so a
// block per row would leave the CU idle while each row's loads are in
// flight.  Instead a grid of one block per CU walks the rows, and the loads
// of its next row are issued before the current row is reduced and written
// (two register sets, alternating).  Rows are addressed through buffer
// resources (a row and the whole grid under 4 GiB of offsets per row): no
// branch surrounds a load or store, so the compiler waits for a prefetched
// row without also waiting for the stores issued after it.
template <typename T, int VPT>
struct RowBuffer {
    uint4 raw[VPT];
    float tail;  // ANY: this thread's element of the row's last D % N
};

// Row `row` (zeros past the last row or the row's last packet).
template <typename T, int VPT, bool ANY>
__device__ __forceinline__ void fetch_row(RowBuffer<T, VPT>& b, const typename Elem<T>::storage* x,
                                          int64_t row, int64_t rows, int64_t D, int tid) {
    constexpr int N = Packet<T>::N;
    const bool ok = row < rows;
    const uint32_t packets = static_cast<uint32_t>(D / N * 16);
    const Rsrc r = buffer_over(x + (ok ? row : 0) * D, ok ? packets : 0u);
#pragma unroll
    for (int k = 0; k < VPT; ++k) b.raw[k] = buffer_load16(r, static_cast<uint32_t>(tid + k * 16 * kWave) * 16u);
    if constexpr (ANY) {
        constexpr uint32_t S = sizeof(typename Elem<T>::storage);
        const Rsrc whole = buffer_over(x + (ok ? row : 0) * D, ok ? static_cast<uint32_t>(D) * S : 0u);
        b.tail = buffer_load_elem<T>(whole, packets + static_cast<uint32_t>(tid) * S);
    }
}

__device__ __forceinline__ uint32_t& word(uint4& v, int i) {
    return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
}

// float32 rows work in place in the packet registers (a second float copy
// of the row would not fit beside the prefetched next row).
template <int VPT, bool ANY>
__device__ __forceinline__ void finish_row_f32(RowBuffer<float, VPT>& b, float* yr, int64_t npk, int rem,
                                               int tid, bool log, float* scratch) {
    float m = ANY && tid < rem ? b.tail : -INFINITY;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const bool in = tid + k * 16 * kWave < npk;
#pragma unroll
        for (int j = 0; j < 4; ++j) m = fmaxf(m, in ? __uint_as_float(word(b.raw[k], j)) : -INFINITY);
    }
    m = row_reduce<16, true>(m, scratch);
    const float shift = m == -INFINITY ? 0.0f : m;
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const bool in = tid + k * 16 * kWave < npk;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float d = __uint_as_float(word(b.raw[k], j)) - shift;
            const float e = exp_fast(d);
            s += in ? e : 0.0f;
            word(b.raw[k], j) = __float_as_uint(log ? d : e);
        }
    }
    float t = 0.0f;
    if (ANY && tid < rem) {
        t = b.tail - shift;
        const float e = exp_fast(t);
        s += e;
        if (!log) t = e;
    }
    s = row_reduce<16, false>(s, scratch);
    const float lse = logf(s);
    const float inv = 1.0f / s;
    if (ANY && tid < rem) yr[npk * 4 + tid] = log ? t - lse : t * inv;
    const Rsrc out = buffer_over(yr, static_cast<uint32_t>(npk * 16));
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        uint4 o = b.raw[k];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float v = __uint_as_float(word(o, j));
            word(o, j) = __float_as_uint(log ? v - lse : v * inv);
        }
        buffer_store16(out, static_cast<uint32_t>(tid + k * 16 * kWave) * 16u, o);
    }
}

template <typename T, int VPT, bool ANY>
__device__ __forceinline__ void finish_row(RowBuffer<T, VPT>& b,
                                           typename Elem<T>::storage* yr, int64_t npk, int rem, int tid,
                                           bool log, float* scratch) {
    if constexpr (sizeof(typename Elem<T>::storage) == 4) {
        finish_row_f32<VPT, ANY>(b, yr, npk, rem, tid, log, scratch);
        return;
    }
    constexpr int N = Packet<T>::N;
    float v[VPT][N];
    float m = ANY && tid < rem ? b.tail : -INFINITY;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const bool in = tid + k * 16 * kWave < npk;
        unpack<T>(b.raw[k], v[k]);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            v[k][j] = in ? v[k][j] : -INFINITY;
            m = fmaxf(m, v[k][j]);
        }
    }
    m = row_reduce<16, true>(m, scratch);
    const float shift = m == -INFINITY ? 0.0f : m;
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < VPT; ++k)
#pragma unroll
        for (int j = 0; j < N; ++j) {
            v[k][j] -= shift;
            const float e = exp_fast(v[k][j]);
            s += e;
            if (!log) v[k][j] = e;
        }
    float t = 0.0f;
    if (ANY && tid < rem) {
        t = b.tail - shift;
        const float e = exp_fast(t);
        s += e;
        if (!log) t = e;
    }
    s = row_reduce<16, false>(s, scratch);
    const float lse = logf(s);
    const float inv = 1.0f / s;
    if (ANY && tid < rem) yr[npk * N + tid] = Elem<T>::store(log ? t - lse : t * inv);
    const Rsrc out = buffer_over(yr, static_cast<uint32_t>(npk * 16));
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        float o[N];
#pragma unroll
        for (int j = 0; j < N; ++j) o[j] = log ? v[k][j] - lse : v[k][j] * inv;
        buffer_store16(out, static_cast<uint32_t>(tid + k * 16 * kWave) * 16u, pack<T>(o));
    }
}

template <typename T, int VPT, bool ANY>
__global__ __launch_bounds__(16 * kWave) void softmax_rows_stream_kernel(
    const typename Elem<T>::storage* x, typename Elem<T>::storage* y, int64_t rows, int64_t D,
    bool log) {
    constexpr int N = Packet<T>::N;
    __shared__ float scratch[16];
    const int tid = threadIdx.x;
    const int64_t npk = D / N;
    const int rem = static_cast<int>(D - npk * N);
    const int64_t step = gridDim.x;
    RowBuffer<T, VPT> a, b;
    int64_t row = blockIdx.x;
    fetch_row<T, VPT, ANY>(a, x, row, rows, D, tid);
    drain();
    // Uniform per block: every thread walks the same rows.
    for (; row < rows; row += 2 * step) {
        fetch_row<T, VPT, ANY>(b, x, row + step, rows, D, tid);
        finish_row<T, VPT, ANY>(a, y + row * D, npk, rem, tid, log, scratch);
        if (row + step >= rows) break;
        fetch_row<T, VPT, ANY>(a, x, row + 2 * step, rows, D, tid);
        finish_row<T, VPT, ANY>(b, y + (row + step) * D, npk, rem, tid, log, scratch);
    }
}

// The backward keeps the two rows as raw packets (16-bit storage takes half
// the registers of unpacked floats) and converts them on use.
template <typename T, int WAVES, int EPT, bool ANY>
__global__ __launch_bounds__(block_threads<WAVES>()) void softmax_backward_rows_kernel(
    const typename Elem<T>::storage* y, const typename Elem<T>::storage* dy,
    typename Elem<T>::storage* dx, int64_t rows, int64_t D, bool log) {
    constexpr int N = Packet<T>::N;
    constexpr int VPT = EPT / N;
    static_assert(VPT * N == EPT, "EPT must be a whole number of packets");
    constexpr int kThreads = WAVES * kWave;
    __shared__ float scratch[block_threads<WAVES>() / kWave];
    const int64_t row = static_cast<int64_t>(blockIdx.x) * rows_per_block<WAVES>() +
                        threadIdx.x / kThreads;
    const int tid = threadIdx.x % kThreads;
    const bool active = row < rows;
    const int64_t npk = D / N;
    const int64_t base = (active ? row : 0) * D;
    uint4 ry[VPT], rg[VPT];
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int64_t q = tid + static_cast<int64_t>(k) * kThreads;
        if (active && q < npk) {
            ry[k] = load_raw_stream<ANY>(y + base + q * N);
            rg[k] = load_raw_stream<ANY>(dy + base + q * N);
        } else {
            ry[k] = rg[k] = make_uint4(0, 0, 0, 0);  // zeros add nothing to the sum
        }
    }
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        float a[N], g[N];
        unpack<T>(ry[k], a);
        unpack<T>(rg[k], g);
#pragma unroll
        for (int j = 0; j < N; ++j) s += log ? g[j] : g[j] * a[j];
    }
    const bool tail = ANY && active && tid < D - npk * N;  // one of the row's last D % N elements
    float ta = 0.0f, tg = 0.0f;
    if (tail) {
        ta = Elem<T>::load(y[base + npk * N + tid]);
        tg = Elem<T>::load(dy[base + npk * N + tid]);
        s += log ? tg : tg * ta;
    }
    s = row_reduce<WAVES, false>(s, scratch);
    if (!active) return;
    if (tail) dx[base + npk * N + tid] = Elem<T>::store(log ? tg - exp_fast(ta) * s : ta * (tg - s));
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int64_t q = tid + static_cast<int64_t>(k) * kThreads;
        if (q < npk) {
            float a[N], g[N], o[N];
            unpack<T>(ry[k], a);
            unpack<T>(rg[k], g);
#pragma unroll
            for (int j = 0; j < N; ++j) {
                o[j] = log ? g[j] - exp_fast(a[j]) * s : a[j] * (g[j] - s);
            }
            store_raw_stream<ANY>(dx + base + q * N, pack<T>(o));
        }
    }
}

// The backward of rows that need a whole 16-wave block, the forward's
// stream scheme for two inputs: one block per CU walks the rows with the
// next row's y and dy loaded before this row's reduction (two register sets
// of raw packets), all through buffer resources.  Packets past the row's
// end load as zeros and add nothing to the row sum.
template <typename T, int VPT>
struct GradRows {
    uint4 y[VPT], g[VPT];
    float ty, tg;  // ANY: this thread's elements of the rows' last D % N
};

template <typename T, int VPT, bool ANY>
__global__ __launch_bounds__(16 * kWave) void softmax_backward_stream_kernel(
    const typename Elem<T>::storage* y, const typename Elem<T>::storage* dy,
    typename Elem<T>::storage* dx, int64_t rows, int64_t D, bool log) {
    constexpr int N = Packet<T>::N;
    __shared__ float scratch[16];
    const int tid = threadIdx.x;
    constexpr uint32_t S = sizeof(typename Elem<T>::storage);
    const uint32_t row_bytes = static_cast<uint32_t>(D / N * 16);  // whole packets
    const uint32_t rem = static_cast<uint32_t>(D % N);
    const int64_t step = gridDim.x;
    auto fetch = [&](GradRows<T, VPT>& b, int64_t row) {
        const bool ok = row < rows;
        const int64_t at = (ok ? row : 0) * D;
        const Rsrc ry = buffer_over(y + at, ok ? row_bytes : 0u);
        const Rsrc rg = buffer_over(dy + at, ok ? row_bytes : 0u);
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            const uint32_t off = static_cast<uint32_t>(tid + k * 16 * kWave) * 16u;
            b.y[k] = buffer_load16(ry, off);
            b.g[k] = buffer_load16(rg, off);
        }
        if constexpr (ANY) {
            const uint32_t off = row_bytes + static_cast<uint32_t>(tid) * S;
            b.ty = buffer_load_elem<T>(buffer_over(y + at, ok ? row_bytes + rem * S : 0u), off);
            b.tg = buffer_load_elem<T>(buffer_over(dy + at, ok ? row_bytes + rem * S : 0u), off);
        }
    };
    auto finish = [&](const GradRows<T, VPT>& b, int64_t row) {
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            float a[N], g[N];
            unpack<T>(b.y[k], a);
            unpack<T>(b.g[k], g);
#pragma unroll
            for (int j = 0; j < N; ++j) s += log ? g[j] : g[j] * a[j];
        }
        if constexpr (ANY) s += log ? b.tg : b.tg * b.ty;  // zeros past the row
        s = row_reduce<16, false>(s, scratch);
        if (ANY && static_cast<uint32_t>(tid) < rem) {
            dx[row * D + D / N * N + tid] = Elem<T>::store(log ? b.tg - exp_fast(b.ty) * s : b.ty * (b.tg - s));
        }
        const Rsrc out = buffer_over(dx + row * D, row_bytes);
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            float a[N], g[N], o[N];
            unpack<T>(b.y[k], a);
            unpack<T>(b.g[k], g);
#pragma unroll
            for (int j = 0; j < N; ++j) o[j] = log ? g[j] - exp_fast(a[j]) * s : a[j] * (g[j] - s);
            buffer_store16(out, static_cast<uint32_t>(tid + k * 16 * kWave) * 16u, pack<T>(o));
        }
    };
    GradRows<T, VPT> a, b;
    int64_t row = blockIdx.x;
    fetch(a, row);
    drain();
    for (; row < rows; row += 2 * step) {
        fetch(b, row + step);
        finish(a, row);
        if (row + step >= rows) break;
        fetch(a, row + 2 * step);
        finish(b, row + step);
    }
}

// The larger of a and b, NaN if either is (fmaxf returns the other operand
// for a NaN, which would let a thread whose only numbers are NaN and -inf
// look empty and be skipped).
__device__ __forceinline__ float max_keep_nan(float a, float b) { return (a > b || a != a) ? a : b; }

// (m, s) <- (m, s) merged with (m2, s2), each s a sum of exp(v - m).  A NaN
// maximum makes the merged sum NaN, so the line's outputs become NaN.
__device__ __forceinline__ void lse_merge(float& m, float& s, float m2, float s2) {
    const float mn = max_keep_nan(m, m2);
    if (mn == -INFINITY) return;
    s = (m == -INFINITY ? 0.0f : s * exp_fast(m - mn)) + (m2 == -INFINITY ? 0.0f : s2 * exp_fast(m2 - mn));
    m = mn;
}

__device__ __forceinline__ void block_merge(float& m, float& s) {
    __shared__ float sm[kBlock / kWave], ss[kBlock / kWave];
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        const float m2 = wave_shfl_xor(m, o), s2 = wave_shfl_xor(s, o);
        lse_merge(m, s, m2, s2);
    }
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (lane == 0) {
        sm[wave] = m;
        ss[wave] = s;
    }
    __syncthreads();
    m = sm[0];
    s = ss[0];
#pragma unroll
    for (int w = 1; w < kBlock / kWave; ++w) lse_merge(m, s, sm[w], ss[w]);
}

// Rows too long to hold: a 256-thread block per row.  Pass 1 keeps a running
// (max, sum) per thread, UNROLL packets in flight; pass 2 re-reads the row
// and writes the result.
template <typename T, int UNROLL, bool ANY>
__global__ __launch_bounds__(kBlock) void softmax_rows_long_kernel(
    const typename Elem<T>::storage* x, typename Elem<T>::storage* y, int64_t D, bool log) {
    constexpr int N = Packet<T>::N;
    const int64_t npk = D / N;
    const typename Elem<T>::storage* xr = x + static_cast<int64_t>(blockIdx.x) * D;
    float m = -INFINITY, s = 0.0f;
    for (int64_t q0 = threadIdx.x; q0 < npk; q0 += static_cast<int64_t>(kBlock) * UNROLL) {
        uint4 raw[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int64_t q = q0 + static_cast<int64_t>(u) * kBlock;
            raw[u] = q < npk ? load_raw<ANY>(xr + q * N)
                             : make_uint4(0xff800000u, 0xff800000u, 0xff800000u, 0xff800000u);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int64_t q = q0 + static_cast<int64_t>(u) * kBlock;
            if (q >= npk) continue;
            float v[N];
            unpack<T>(raw[u], v);
            float pm = v[0];
#pragma unroll
            for (int j = 1; j < N; ++j) pm = fmaxf(pm, v[j]);
            // With nothing but -inf (or NaN) so far, exponentials relative
            // to 0: 0 of -inf, and NaN stays.
            const float mn = fmaxf(m, pm), shift = mn == -INFINITY ? 0.0f : mn;
            float t = 0.0f;
#pragma unroll
            for (int j = 0; j < N; ++j) t += exp_fast(v[j] - shift);
            s = s * exp_fast(m - shift) + t;
            m = mn;
        }
    }
    const bool tail = ANY && threadIdx.x < D - npk * N;  // one of the row's last D % N elements
    const float tv = tail ? Elem<T>::load(xr[npk * N + threadIdx.x]) : -INFINITY;
    if (ANY && tv != -INFINITY) {
        const float mn = fmaxf(m, tv);
        s = s * exp_fast(m - mn) + exp_fast(tv - mn);
        m = mn;
    }
    // fmaxf lets a NaN go, and each exponential of one is NaN: the sum keeps
    // it, and the merge takes it from the maximum (NaN kept by the maximum
    // of every packet: 8-18 % of the kernel).
    if (s != s) m = s;
    block_merge(m, s);
    const float shift = m == -INFINITY ? 0.0f : m;
    const float lse = logf(s);
    const float inv = 1.0f / s;
    typename Elem<T>::storage* yr = y + static_cast<int64_t>(blockIdx.x) * D;
    if (tail) {
        const float d = tv - shift;
        yr[npk * N + threadIdx.x] = Elem<T>::store(log ? d - lse : exp_fast(d) * inv);
    }
    for (int64_t q = threadIdx.x; q < npk; q += kBlock) {
        float v[N], o[N];
        unpack<T>(load_raw<ANY>(xr + q * N), v);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const float d = v[j] - shift;
            o[j] = log ? d - lse : exp_fast(d) * inv;
        }
        store_raw_stream<ANY>(yr + q * N, pack<T>(o));
    }
}

template <typename T, int UNROLL, bool ANY>
__global__ __launch_bounds__(kBlock) void softmax_backward_rows_long_kernel(
    const typename Elem<T>::storage* y, const typename Elem<T>::storage* dy,
    typename Elem<T>::storage* dx, int64_t D, bool log) {
    constexpr int N = Packet<T>::N;
    __shared__ float scratch[kBlock / kWave];
    const int64_t npk = D / N;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * D;
    float s = 0.0f;
    for (int64_t q0 = threadIdx.x; q0 < npk; q0 += static_cast<int64_t>(kBlock) * UNROLL) {
        uint4 ra[UNROLL], rg[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            const int64_t q = q0 + static_cast<int64_t>(u) * kBlock;
            const bool in = q < npk;
            ra[u] = in ? load_raw<ANY>(y + base + q * N) : make_uint4(0, 0, 0, 0);
            rg[u] = in ? load_raw<ANY>(dy + base + q * N) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            float a[N], g[N];
            unpack<T>(ra[u], a);
            unpack<T>(rg[u], g);
#pragma unroll
            for (int j = 0; j < N; ++j) s += log ? g[j] : g[j] * a[j];
        }
    }
    const bool tail = ANY && threadIdx.x < D - npk * N;  // one of the row's last D % N elements
    float ta = 0.0f, tg = 0.0f;
    if (tail) {
        ta = Elem<T>::load(y[base + npk * N + threadIdx.x]);
        tg = Elem<T>::load(dy[base + npk * N + threadIdx.x]);
        s += log ? tg : tg * ta;
    }
    s = row_reduce<kBlock / kWave, false>(s, scratch);
    if (tail) {
        dx[base + npk * N + threadIdx.x] = Elem<T>::store(log ? tg - exp_fast(ta) * s : ta * (tg - s));
    }
    for (int64_t q = threadIdx.x; q < npk; q += kBlock) {
        float a[N], g[N], o[N];
        unpack<T>(load_raw<ANY>(y + base + q * N), a);
        unpack<T>(load_raw<ANY>(dy + base + q * N), g);
#pragma unroll
        for (int j = 0; j < N; ++j) o[j] = log ? g[j] - exp_fast(a[j]) * s : a[j] * (g[j] - s);
        store_raw_stream<ANY>(dx + base + q * N, pack<T>(o));
    }
}

// Rows past what 16 waves hold beside a prefetched next row (a vocabulary of
// 50257, or float32 rows of more than 32768): a 512-thread block holds the
// raw row in up to 25 packets a thread, and two blocks share a CU, so one
// loads or stores while the other reduces.  Read once and written once; the
// two-pass kernel above reads such a row twice from HBM (the rows in flight
// pass the L2).  Measured, log_softmax of 2048 x 50257: bfloat16 259 ->
// 95 us, float32 318 -> 167 us.
constexpr int kWideThreads = 512;
constexpr int kWideWaves = kWideThreads / kWave;

// Before a pass takes a held packet: the compiler neither keeps an earlier
// pass's unpacked floats (twice the registers of 16-bit storage) nor starts
// on the next packet before this one's work is done, so the row and one
// packet's temporaries fit the 128 registers two blocks a CU allow.
__device__ __forceinline__ void take_packet(uint4& raw) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+v"(raw.x), "+v"(raw.y), "+v"(raw.z), "+v"(raw.w));
}

template <typename T, int VPT>
__global__ __launch_bounds__(kWideThreads, 4) void softmax_rows_wide_kernel(
    const typename Elem<T>::storage* x, typename Elem<T>::storage* y, int64_t D, bool log) {
    constexpr int N = Packet<T>::N;
    __shared__ float scratch[kWideWaves];
    const int tid = threadIdx.x;
    const int npk = static_cast<int>(D / N), rem = static_cast<int>(D - static_cast<int64_t>(npk) * N);
    const int64_t at = static_cast<int64_t>(blockIdx.x) * D;
    const Rsrc in_row = buffer_over(x + at, static_cast<uint32_t>(npk) * 16u);
    uint4 raw[VPT];
#pragma unroll
    for (int k = 0; k < VPT; ++k)
        raw[k] = buffer_load16(in_row, static_cast<uint32_t>(tid + k * kWideThreads) * 16u);
    float t = -INFINITY;
    if (tid < rem) t = Elem<T>::load(x[at + static_cast<int64_t>(npk) * N + tid]);
    float m = t;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const bool in = tid + k * kWideThreads < npk;
        float v[N];
        take_packet(raw[k]);
        unpack<T>(raw[k], v);
#pragma unroll
        for (int j = 0; j < N; ++j) m = fmaxf(m, in ? v[j] : -INFINITY);
    }
    m = row_reduce<kWideWaves, true>(m, scratch);
    const float shift = m == -INFINITY ? 0.0f : m;
    float s = 0.0f;
    // The row stays raw; its exponentials are formed again for the output.
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const bool in = tid + k * kWideThreads < npk;
        float v[N];
        take_packet(raw[k]);
        unpack<T>(raw[k], v);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const float e = exp_fast(v[j] - shift);
            s += in ? e : 0.0f;
        }
    }
    t -= shift;
    {
        const float e = exp_fast(t);
        s += e;
        if (!log) t = e;
    }
    s = row_reduce<kWideWaves, false>(s, scratch);
    const float lse = logf(s);
    const float inv = 1.0f / s;
    if (tid < rem) y[at + static_cast<int64_t>(npk) * N + tid] = Elem<T>::store(log ? t - lse : t * inv);
    const Rsrc out = buffer_over(y + at, static_cast<uint32_t>(npk) * 16u);
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        float v[N], o[N];
        take_packet(raw[k]);
        unpack<T>(raw[k], v);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const float d = v[j] - shift;
            o[j] = log ? d - lse : exp_fast(d) * inv;
        }
        buffer_store16(out, static_cast<uint32_t>(tid + k * kWideThreads) * 16u, pack<T>(o));
    }
}

// The same for the backward: dy's row is held, y's streams past it (once for
// log_softmax, whose sum needs dy alone; a second time for softmax).
// Measured, the log_softmax backward of 2048 x 50257: bfloat16 225 -> 132
// us, float32 389 -> 250 us.
template <typename T, int VPT>
__global__ __launch_bounds__(kWideThreads, 4) void softmax_backward_rows_wide_kernel(
    const typename Elem<T>::storage* y, const typename Elem<T>::storage* dy,
    typename Elem<T>::storage* dx, int64_t D, bool log) {
    constexpr int N = Packet<T>::N;
    __shared__ float scratch[kWideWaves];
    const int tid = threadIdx.x;
    const int npk = static_cast<int>(D / N), rem = static_cast<int>(D - static_cast<int64_t>(npk) * N);
    const int64_t at = static_cast<int64_t>(blockIdx.x) * D;
    const uint32_t bytes = static_cast<uint32_t>(npk) * 16u;
    const Rsrc rg = buffer_over(dy + at, bytes), ry = buffer_over(y + at, bytes);
    uint4 raw[VPT];
#pragma unroll
    for (int k = 0; k < VPT; ++k)
        raw[k] = buffer_load16(rg, static_cast<uint32_t>(tid + k * kWideThreads) * 16u);
    float ta = 0.0f, tg = 0.0f;
    if (tid < rem) {
        ta = Elem<T>::load(y[at + static_cast<int64_t>(npk) * N + tid]);
        tg = Elem<T>::load(dy[at + static_cast<int64_t>(npk) * N + tid]);
    }
    // packets past the row's end are zeros and add nothing
    float s = log ? tg : tg * ta;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        float g[N];
        take_packet(raw[k]);
        unpack<T>(raw[k], g);
        if (log) {
#pragma unroll
            for (int j = 0; j < N; ++j) s += g[j];
        } else {
            float a[N];
            unpack<T>(buffer_load16_cached(ry, static_cast<uint32_t>(tid + k * kWideThreads) * 16u), a);
#pragma unroll
            for (int j = 0; j < N; ++j) s += g[j] * a[j];
        }
    }
    s = row_reduce<kWideWaves, false>(s, scratch);
    if (tid < rem) {
        dx[at + static_cast<int64_t>(npk) * N + tid] =
            Elem<T>::store(log ? tg - exp_fast(ta) * s : ta * (tg - s));
    }
    const Rsrc out = buffer_over(dx + at, bytes);
    constexpr int kAhead = VPT > 19 && sizeof(typename Elem<T>::storage) == 4 ? 2 : 4;  // packets of y in flight
    uint4 next[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
        next[k] = buffer_load16(ry, static_cast<uint32_t>(tid + k * kWideThreads) * 16u);
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const uint32_t off = static_cast<uint32_t>(tid + k * kWideThreads) * 16u;
        float a[N], g[N], o[N];
        take_packet(raw[k]);
        unpack<T>(next[k % kAhead], a);
        unpack<T>(raw[k], g);
#pragma unroll
        for (int j = 0; j < N; ++j) o[j] = log ? g[j] - exp_fast(a[j]) * s : a[j] * (g[j] - s);
        buffer_store16(out, off, pack<T>(o));
        if (k + kAhead < VPT)
            next[k % kAhead] = buffer_load16(ry, static_cast<uint32_t>(tid + (k + kAhead) * kWideThreads) * 16u);
    }
}

// ---- softmax over a dimension that is not the last ---------------------------
//
// [outer, D, inner] with inner > 1: a block takes 64 consecutive columns of
// one outer index (one a lane, so a wave reads 64 neighbours of a row) and
// one slice of D; its four waves take the slice's rows in turn, eight rows
// loaded together a lane (rows past the slice are clamped and masked, so
// the loads carry no branch).  Per column, the forward keeps a running
// (max, sum of exp) and the backward a running sum; the waves' partials
// fold through LDS in wave order.  With enough column tiles to fill the GPU
// there is one slice and one launch (MODE kColFused); otherwise a first
// launch writes each slice's partials (kColStats) and a second folds them in
// slice order and writes the output (kColWrite).  The earlier kernel gave
// each column to one thread, which walked D alone: 2.4 ms for a dim-0
// softmax of [4096, 4096].
constexpr int kColWaves = 4;
constexpr int kColWidth = kWave;  // columns of a block
constexpr int kColBatch = 8;      // rows loaded together a lane
constexpr int kColFused = 0, kColStats = 1, kColWrite = 2;

struct ColBlock {
    int64_t o, c0, d0, d1, sl;
};

// Block b: column tile b % tiles, slice (b / tiles) % slices, outer index
// b / (tiles * slices).
__device__ __forceinline__ ColBlock col_block(int64_t tiles, int64_t slices, int64_t D, int64_t dslice) {
    ColBlock cb;
    int64_t b = blockIdx.x;
    cb.c0 = (b % tiles) * kColWidth;
    b /= tiles;
    cb.sl = b % slices;
    cb.o = b / slices;
    cb.d0 = cb.sl * dslice;
    cb.d1 = cb.d0 + dslice < D ? cb.d0 + dslice : D;
    return cb;
}

template <typename T, int MODE>
__global__ __launch_bounds__(kColWaves * kWave) void softmax_cols_kernel(
    const typename Elem<T>::storage* x, typename Elem<T>::storage* y, float* pm, float* ps, int64_t outer,
    int64_t D, int64_t inner, int64_t tiles, int64_t slices, int64_t dslice, bool log) {
    __shared__ float sm[kColWaves][kColWidth], ss[kColWaves][kColWidth];
    const ColBlock cb = col_block(tiles, slices, D, dslice);
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    const int64_t c = cb.c0 + lane;
    const bool live = c < inner;
    const int64_t base = cb.o * D * inner + (live ? c : inner - 1);
    const typename Elem<T>::storage* col = x + base;
    float m = -INFINITY, s = 0.0f;
    if constexpr (MODE != kColWrite) {
        for (int64_t d = cb.d0 + w; d < cb.d1; d += kColWaves * kColBatch) {
            float v[kColBatch];
#pragma unroll
            for (int j = 0; j < kColBatch; ++j) {
                const int64_t dj = d + j * kColWaves;
                v[j] = Elem<T>::load(col[(dj < cb.d1 ? dj : cb.d1 - 1) * inner]);
            }
            float bm = -INFINITY;
#pragma unroll
            for (int j = 0; j < kColBatch; ++j) {
                if (d + j * kColWaves >= cb.d1) v[j] = -INFINITY;
                bm = max_keep_nan(bm, v[j]);
            }
            if (bm == -INFINITY) continue;  // only -inf and masked rows: nothing to add
            float bs = 0.0f;
#pragma unroll
            for (int j = 0; j < kColBatch; ++j) bs += exp_fast(v[j] - bm);
            lse_merge(m, s, bm, bs);
        }
        sm[w][lane] = m;
        ss[w][lane] = s;
        __syncthreads();
        m = sm[0][lane];
        s = ss[0][lane];
#pragma unroll
        for (int k = 1; k < kColWaves; ++k) lse_merge(m, s, sm[k][lane], ss[k][lane]);
        if constexpr (MODE == kColStats) {
            if (w == 0 && live) {
                const int64_t at = (cb.sl * outer + cb.o) * inner + c;
                pm[at] = m;
                ps[at] = s;
            }
            return;
        }
    } else {
        const int64_t cc = live ? c : inner - 1;
        for (int64_t k = 0; k < slices; ++k) {
            const int64_t at = (k * outer + cb.o) * inner + cc;
            lse_merge(m, s, pm[at], ps[at]);
        }
    }
    // A column of -inf (or an empty one) would give inf - inf; exp(-inf - 0)
    // keeps it at 0 instead.
    const float shift = m == -INFINITY ? 0.0f : m;
    const float lse = logf(s);
    const float inv = 1.0f / s;
    typename Elem<T>::storage* out = y + base;
    for (int64_t d = cb.d0 + w; d < cb.d1; d += kColWaves * kColBatch) {
        float v[kColBatch];
#pragma unroll
        for (int j = 0; j < kColBatch; ++j) {
            const int64_t dj = d + j * kColWaves;
            v[j] = Elem<T>::load(col[(dj < cb.d1 ? dj : cb.d1 - 1) * inner]) - shift;
        }
#pragma unroll
        for (int j = 0; j < kColBatch; ++j) {
            const int64_t dj = d + j * kColWaves;
            if (live && dj < cb.d1) out[dj * inner] = Elem<T>::store(log ? v[j] - lse : exp_fast(v[j]) * inv);
        }
    }
}

// The backward: per column s = sum over D of dy (log) or dy * y, then
// dx = dy - exp(y) s (log) or y (dy - s).
template <typename T, int MODE>
__global__ __launch_bounds__(kColWaves * kWave) void softmax_backward_cols_kernel(
    const typename Elem<T>::storage* y, const typename Elem<T>::storage* dy, typename Elem<T>::storage* dx,
    float* ps, int64_t outer, int64_t D, int64_t inner, int64_t tiles, int64_t slices, int64_t dslice, bool log) {
    __shared__ float ss[kColWaves][kColWidth];
    const ColBlock cb = col_block(tiles, slices, D, dslice);
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    const int64_t c = cb.c0 + lane;
    const bool live = c < inner;
    const int64_t base = cb.o * D * inner + (live ? c : inner - 1);
    const typename Elem<T>::storage* ycol = y + base;
    const typename Elem<T>::storage* gcol = dy + base;
    float s = 0.0f;
    if constexpr (MODE != kColWrite) {
        for (int64_t d = cb.d0 + w; d < cb.d1; d += kColWaves * kColBatch) {
            float a[kColBatch], g[kColBatch];
#pragma unroll
            for (int j = 0; j < kColBatch; ++j) {
                const int64_t dj = d + j * kColWaves;
                const int64_t at = (dj < cb.d1 ? dj : cb.d1 - 1) * inner;
                a[j] = Elem<T>::load(ycol[at]);
                g[j] = Elem<T>::load(gcol[at]);
            }
#pragma unroll
            for (int j = 0; j < kColBatch; ++j) {
                if (d + j * kColWaves < cb.d1) s += log ? g[j] : g[j] * a[j];
            }
        }
        ss[w][lane] = s;
        __syncthreads();
        s = ss[0][lane];
#pragma unroll
        for (int k = 1; k < kColWaves; ++k) s += ss[k][lane];
        if constexpr (MODE == kColStats) {
            if (w == 0 && live) ps[(cb.sl * outer + cb.o) * inner + c] = s;
            return;
        }
    } else {
        const int64_t cc = live ? c : inner - 1;
        for (int64_t k = 0; k < slices; ++k) s += ps[(k * outer + cb.o) * inner + cc];
    }
    typename Elem<T>::storage* out = dx + base;
    for (int64_t d = cb.d0 + w; d < cb.d1; d += kColWaves * kColBatch) {
        float a[kColBatch], g[kColBatch];
#pragma unroll
        for (int j = 0; j < kColBatch; ++j) {
            const int64_t dj = d + j * kColWaves;
            const int64_t at = (dj < cb.d1 ? dj : cb.d1 - 1) * inner;
            a[j] = Elem<T>::load(ycol[at]);
            g[j] = Elem<T>::load(gcol[at]);
        }
#pragma unroll
        for (int j = 0; j < kColBatch; ++j) {
            const int64_t dj = d + j * kColWaves;
            if (live && dj < cb.d1) {
                out[dj * inner] = Elem<T>::store(log ? g[j] - exp_fast(a[j]) * s : a[j] * (g[j] - s));
            }
        }
    }
}

// Tiles, slices and rows a slice for the column kernels: enough blocks for
// two a CU, slices of at least 64 rows.
struct ColPlan {
    int64_t tiles, slices, dslice, blocks;
};

ColPlan col_plan(int64_t outer, int64_t D, int64_t inner, int device) {
    ColPlan p;
    p.tiles = (inner + kColWidth - 1) / kColWidth;
    const int64_t base = outer * p.tiles;
    const int64_t want = 2 * static_cast<int64_t>(cu_count(device));
    int64_t slices = (want + base - 1) / base;
    const int64_t most = (D + 63) / 64;
    if (slices > most) slices = most;
    if (slices < 1) slices = 1;
    p.dslice = (D + slices - 1) / slices;
    p.slices = (D + p.dslice - 1) / p.dslice;
    p.blocks = base * p.slices;
    return p;
}

// ---- configuration choice ---------------------------------------------------

// A register-resident layout; waves == 0 means the long-row kernel.
struct RowConfig {
    int waves, ept;
};

template <typename T, int W, int E, bool ANY>
void launch_forward_rows(int device, const void* x, void* y, int64_t rows, int64_t D, bool log) {
    using S = typename Elem<T>::storage;
    const int64_t blocks = (rows + rows_per_block<W>() - 1) / rows_per_block<W>();
    softmax_rows_kernel<T, W, E, ANY><<<blocks, block_threads<W>(), 0, stream(device)>>>(
        static_cast<const S*>(x), static_cast<S*>(y), rows, D, log);
}

template <typename T, int W, int E, bool ANY>
void launch_backward_rows(int device, const void* y, const void* dy, void* dx, int64_t rows,
                          int64_t D, bool log) {
    using S = typename Elem<T>::storage;
    const int64_t blocks = (rows + rows_per_block<W>() - 1) / rows_per_block<W>();
    softmax_backward_rows_kernel<T, W, E, ANY><<<blocks, block_threads<W>(), 0, stream(device)>>>(
        static_cast<const S*>(y), static_cast<const S*>(dy), static_cast<S*>(dx), rows, D, log);
}

// The layouts compiled, as (waves per row, packets per thread): the
// measured best on MI355X puts about two 16-byte packets in each thread and
// grows the number of waves with the row, up to 16 (a 1024-thread block);
// longer rows then take more packets per thread, up to 32 float32 values.
#define TP_AMD_SOFTMAX_CONFIGS(X) \
    X(1, 1) X(1, 2) X(2, 2) X(4, 2) X(8, 2) X(16, 2) X(16, 4) X(16, 8)

template <typename T, bool ANY>
bool launch_forward_config(RowConfig c, int device, const void* x, void* y, int64_t rows,
                           int64_t D, bool log) {
    constexpr int N = Packet<T>::N;
#define TP_AMD_FWD(W, V)                                                             \
    if constexpr (V * N <= 32) {                                                     \
        if (c.waves == W && c.ept == V * N) {                                        \
            launch_forward_rows<T, W, V * N, ANY>(device, x, y, rows, D, log);       \
            return true;                                                             \
        }                                                                            \
    }
    TP_AMD_SOFTMAX_CONFIGS(TP_AMD_FWD)
#undef TP_AMD_FWD
    return false;
}

template <typename T, bool ANY>
bool launch_backward_config(RowConfig c, int device, const void* y, const void* dy, void* dx,
                            int64_t rows, int64_t D, bool log) {
    constexpr int N = Packet<T>::N;
#define TP_AMD_BWD(W, V)                                                             \
    if constexpr (V * N <= 32) {                                                     \
        if (c.waves == W && c.ept == V * N) {                                        \
            launch_backward_rows<T, W, V * N, ANY>(device, y, dy, dx, rows, D, log); \
            return true;                                                             \
        }                                                                            \
    }
    TP_AMD_SOFTMAX_CONFIGS(TP_AMD_BWD)
#undef TP_AMD_BWD
    return false;
}

// The compiled layout for a row of D elements (waves == 0: none holds it).
template <typename T>
RowConfig choose_config(int64_t D) {
    constexpr int N = Packet<T>::N;
    constexpr int kPairs[][2] = {{1, 1}, {1, 2}, {2, 2}, {4, 2}, {8, 2}, {16, 2}, {16, 4}, {16, 8}};
    const int64_t npk = (D + N - 1) / N;
    for (const auto& c : kPairs) {
        if (c[1] * N > 32) break;
        if (static_cast<int64_t>(c[0]) * kWave * c[1] >= npk) return RowConfig{c[0], c[1] * N};
    }
    return RowConfig{0, 0};
}

// Packets a thread of the 512-thread kernels holds for a row of D elements:
// the smallest compiled count, 0 when none holds the row.
template <typename T>
int wide_packets(int64_t D) {
    for (const int v : {13, 19, 25}) {
        if (D / Packet<T>::N <= int64_t{v} * kWideThreads) return v;
    }
    return 0;
}

// Softmax over rows.  The kernel by the row's length: registers of 1 to 16
// waves, then the 16-wave walk with a prefetched next row, then the
// 512-thread blocks, then two passes.
template <typename T, bool ANY>
void launch_forward(int device, bool log, int64_t rows, int64_t D, const typename Elem<T>::storage* x,
                    typename Elem<T>::storage* y) {
    constexpr int N = Packet<T>::N;
    hipStream_t st = stream(device);
    const RowConfig c = choose_config<T>(D);
    if (c.waves == 16) {
        // Rows that need a whole block: one block per CU walks them.
        const int64_t grid = rows < cu_count(device) ? rows : cu_count(device);
        const int vpt = c.ept / N;
        if (vpt <= 2) {
            softmax_rows_stream_kernel<T, 2, ANY><<<grid, 16 * kWave, 0, st>>>(x, y, rows, D, log);
        } else if (vpt <= 4) {
            softmax_rows_stream_kernel<T, 4, ANY><<<grid, 16 * kWave, 0, st>>>(x, y, rows, D, log);
        } else if constexpr (N == 4) {
            softmax_rows_stream_kernel<T, 8, ANY><<<grid, 16 * kWave, 0, st>>>(x, y, rows, D, log);
        }
        return;
    }
    if (c.waves > 0) {
        launch_forward_config<T, ANY>(c, device, x, y, rows, D, log);
        return;
    }
    switch (wide_packets<T>(D)) {
        case 13: softmax_rows_wide_kernel<T, 13><<<rows, kWideThreads, 0, st>>>(x, y, D, log); break;
        case 19: softmax_rows_wide_kernel<T, 19><<<rows, kWideThreads, 0, st>>>(x, y, D, log); break;
        case 25: softmax_rows_wide_kernel<T, 25><<<rows, kWideThreads, 0, st>>>(x, y, D, log); break;
        default: softmax_rows_long_kernel<T, 4, ANY><<<rows, kBlock, 0, st>>>(x, y, D, log);
    }
}

template <typename T, bool ANY>
void launch_backward(int device, bool log, int64_t rows, int64_t D, const typename Elem<T>::storage* y,
                     const typename Elem<T>::storage* dy, typename Elem<T>::storage* dx) {
    constexpr int N = Packet<T>::N;
    hipStream_t st = stream(device);
    const RowConfig c = choose_config<T>(D);
    if (c.waves == 16 && c.ept / N <= 4) {
        // Rows that need a whole block: one block per CU walks them.
        const int64_t grid = rows < cu_count(device) ? rows : cu_count(device);
        if (c.ept / N <= 2) {
            softmax_backward_stream_kernel<T, 2, ANY><<<grid, 16 * kWave, 0, st>>>(y, dy, dx, rows, D, log);
        } else {
            softmax_backward_stream_kernel<T, 4, ANY><<<grid, 16 * kWave, 0, st>>>(y, dy, dx, rows, D, log);
        }
        return;
    }
    if (c.waves > 0) {
        launch_backward_config<T, ANY>(c, device, y, dy, dx, rows, D, log);
        return;
    }
    switch (wide_packets<T>(D)) {
        case 13: softmax_backward_rows_wide_kernel<T, 13><<<rows, kWideThreads, 0, st>>>(y, dy, dx, D, log); break;
        case 19: softmax_backward_rows_wide_kernel<T, 19><<<rows, kWideThreads, 0, st>>>(y, dy, dx, D, log); break;
        case 25: softmax_backward_rows_wide_kernel<T, 25><<<rows, kWideThreads, 0, st>>>(y, dy, dx, D, log); break;
        default: softmax_backward_rows_long_kernel<T, 2, ANY><<<rows, kBlock, 0, st>>>(y, dy, dx, D, log);
    }
}

template <typename T>
void softmax_typed(int device, bool log, int64_t outer, int64_t D, int64_t inner, const void* x,
                   void* y) {
    using S = typename Elem<T>::storage;
    constexpr int N = Packet<T>::N;
    hipStream_t st = stream(device);
    if (inner == 1) {
        if (D % N == 0 && aligned16(x) && aligned16(y)) {
            launch_forward<T, false>(device, log, outer, D, static_cast<const S*>(x), static_cast<S*>(y));
        } else {
            launch_forward<T, true>(device, log, outer, D, static_cast<const S*>(x), static_cast<S*>(y));
        }
    } else {
        const ColPlan cp = col_plan(outer, D, inner, device);
        TP_AMD_CHECK(cp.blocks < (int64_t{1} << 31), "softmax: ", cp.blocks, " blocks exceed the grid");
        const unsigned blocks = static_cast<unsigned>(cp.blocks);
        if (cp.slices == 1) {
            softmax_cols_kernel<T, kColFused><<<blocks, kColWaves * kWave, 0, st>>>(
                static_cast<const S*>(x), static_cast<S*>(y), nullptr, nullptr, outer, D, inner, cp.tiles, 1, cp.dslice,
                log);
        } else {
            const size_t parts = static_cast<size_t>(cp.slices * outer * inner);
            Workspace ws(2 * parts * sizeof(float), device);
            float* pm = static_cast<float*>(ws.get());
            float* ps = pm + parts;
            softmax_cols_kernel<T, kColStats><<<blocks, kColWaves * kWave, 0, st>>>(
                static_cast<const S*>(x), nullptr, pm, ps, outer, D, inner, cp.tiles, cp.slices, cp.dslice, log);
            softmax_cols_kernel<T, kColWrite><<<blocks, kColWaves * kWave, 0, st>>>(
                static_cast<const S*>(x), static_cast<S*>(y), pm, ps, outer, D, inner, cp.tiles, cp.slices, cp.dslice,
                log);
        }
    }
    TP_AMD_HIP_CHECK(hipGetLastError());
}

template <typename T>
void softmax_backward_typed(int device, bool log, int64_t outer, int64_t D, int64_t inner,
                            const void* y, const void* dy, void* dx) {
    using S = typename Elem<T>::storage;
    constexpr int N = Packet<T>::N;
    hipStream_t st = stream(device);
    if (inner == 1) {
        if (D % N == 0 && aligned16(y) && aligned16(dy) && aligned16(dx)) {
            launch_backward<T, false>(device, log, outer, D, static_cast<const S*>(y),
                                      static_cast<const S*>(dy), static_cast<S*>(dx));
        } else {
            launch_backward<T, true>(device, log, outer, D, static_cast<const S*>(y),
                                     static_cast<const S*>(dy), static_cast<S*>(dx));
        }
    } else {
        const ColPlan cp = col_plan(outer, D, inner, device);
        TP_AMD_CHECK(cp.blocks < (int64_t{1} << 31), "softmax backward: ", cp.blocks, " blocks exceed the grid");
        const unsigned blocks = static_cast<unsigned>(cp.blocks);
        if (cp.slices == 1) {
            softmax_backward_cols_kernel<T, kColFused><<<blocks, kColWaves * kWave, 0, st>>>(
                static_cast<const S*>(y), static_cast<const S*>(dy), static_cast<S*>(dx), nullptr, outer, D, inner,
                cp.tiles, 1, cp.dslice, log);
        } else {
            Workspace ws(static_cast<size_t>(cp.slices * outer * inner) * sizeof(float), device);
            float* ps = static_cast<float*>(ws.get());
            softmax_backward_cols_kernel<T, kColStats><<<blocks, kColWaves * kWave, 0, st>>>(
                static_cast<const S*>(y), static_cast<const S*>(dy), nullptr, ps, outer, D, inner, cp.tiles,
                cp.slices, cp.dslice, log);
            softmax_backward_cols_kernel<T, kColWrite><<<blocks, kColWaves * kWave, 0, st>>>(
                static_cast<const S*>(y), static_cast<const S*>(dy), static_cast<S*>(dx), ps, outer, D, inner,
                cp.tiles, cp.slices, cp.dslice, log);
        }
    }
    TP_AMD_HIP_CHECK(hipGetLastError());
}

}  // namespace

}  // namespace tp_amd

using namespace tp_amd;

extern "C" {

int tp_amd_launch_softmax(int device, int log, int dtype, int64_t outer, int64_t dim,
                          int64_t inner, const void* x, void* y) {
    return guarded([&] {
        TP_AMD_CHECK(outer >= 0 && dim >= 0 && inner >= 0, "negative softmax extent");
        if (outer == 0 || dim == 0 || inner == 0) return;
        TP_AMD_CHECK(outer <= 0x7fffffff, "softmax: too many rows");
        const OnDevice scope(device);
        const int index = scope.index();
        switch (dtype) {
            case TP_AMD_FLOAT32: softmax_typed<float>(index, log != 0, outer, dim, inner, x, y); break;
            case TP_AMD_BFLOAT16: softmax_typed<bf16_t>(index, log != 0, outer, dim, inner, x, y); break;
            case TP_AMD_FLOAT16: softmax_typed<f16_t>(index, log != 0, outer, dim, inner, x, y); break;
            default:
                TP_AMD_CHECK(false, "softmax takes float32, float16 or bfloat16, got ",
                             dtype_name(dtype));
        }
    });
}

int tp_amd_launch_softmax_backward(int device, int log, int dtype, int64_t outer, int64_t dim,
                                   int64_t inner, const void* y, const void* dy, void* dx) {
    return guarded([&] {
        TP_AMD_CHECK(outer >= 0 && dim >= 0 && inner >= 0, "negative softmax extent");
        if (outer == 0 || dim == 0 || inner == 0) return;
        TP_AMD_CHECK(outer <= 0x7fffffff, "softmax: too many rows");
        const OnDevice scope(device);
        const int index = scope.index();
        switch (dtype) {
            case TP_AMD_FLOAT32:
                softmax_backward_typed<float>(index, log != 0, outer, dim, inner, y, dy, dx);
                break;
            case TP_AMD_BFLOAT16:
                softmax_backward_typed<bf16_t>(index, log != 0, outer, dim, inner, y, dy, dx);
                break;
            case TP_AMD_FLOAT16:
                softmax_backward_typed<f16_t>(index, log != 0, outer, dim, inner, y, dy, dx);
                break;
            default:
                TP_AMD_CHECK(false, "softmax takes float32, float16 or bfloat16, got ",
                             dtype_name(dtype));
        }
    });
}

}  // extern "C"
