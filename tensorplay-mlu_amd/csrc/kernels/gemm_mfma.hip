// Matrix-core GEMM for gfx950 (CDNA4), and the dispatch between it and the
// general kernel (gemm.hip).
//
// C[b] = alpha * op(A[b]) op(B[b]) + beta * Cin[b] with float32
// accumulation on MFMA:
//   * bfloat16 / float16: v_mfma_f32_32x32x16_{bf16,f16} -- each lane feeds
//     8 consecutive k of one row of A and of one column of B;
//   * float32: v_mfma_f32_32x32x2_f32 -- each lane feeds one k; a 16-byte
//     LDS read gives a lane 4 consecutive k that feed 4 back-to-back MFMAs
//     (lane half h supplies k = 4h + j to MFMA j, for A and B alike, so the
//     pairing of A and B elements is exact whatever order the sum takes).
// Kernels, tried in this order:
//   * 16-bit operands, K of 64 or 128, M and N multiples of 256, at least
//     one 256 x 256 tile per CU: `smallk` below -- all of K loaded at once,
//     one barrier, the stores of one 32 x 32 tile overlapping the MFMAs of
//     the next (attention-sized bmm).
//   * 16-bit operands, M and N multiples of 256, K of 128, at least one
//     256 x 256 tile per CU: `big` below -- four waves of 128 x 128 (eight
//     of 128 x 64 when K <= 256), operand
//     tiles loaded straight into LDS by buffer loads and read back with
//     ds_read_b128 (K-major operands) or ds_read_b64_tr_b16 (transposed
//     views, read in place); no bounds checks anywhere in the K loop.
//   * everything else: the tile kernel, gemm_tile_kernel, at a tile shape
//     and a split over K that plan_tiles picks.
// The last two load operand tiles straight into LDS, 128 bytes of K a step,
// read an operand where it lies in either orientation, and keep the next K
// tiles' loads in flight while they multiply.  All kernels number their
// tiles so each of the 8 XCDs walks a contiguous range in groups of 8 tile
// rows, keeping an XCD's A and B panels hot in its own L2.

#include <type_traits>
#include <utility>

#include "device_common.h"
#include "gemm.h"
#include "../allocator.h"
#include "../common.h"
#include "../runtime.h"
#include "tp_amd_kernels.h"

namespace tp_amd {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <typename T>
struct Mfma;

template <>
struct Mfma<bf16_t> {
    static constexpr int V = 8;     // elements per 16-byte vector
    static constexpr int BK = 64;   // K per LDS tile
    __device__ __forceinline__ static f32x16 mma(const uint4& a, const uint4& b, f32x16 c) {
        bf16x8 av, bv;
        __builtin_memcpy(&av, &a, 16);
        __builtin_memcpy(&bv, &b, 16);
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, c, 0, 0, 0);
    }
    static constexpr int kPerTile = 1;  // MFMAs a 32 x 32 tile takes per fragment
    // The tiles' MFMAs of substep s, on the s-th of CH accumulators each.
    template <int TM, int TN, int CH>
    __device__ __forceinline__ static void tiles(const uint4 (&a)[TM], const uint4 (&b)[TN], f32x16 (&c)[CH][TM][TN],
                                                 int s) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) c[s % CH][i][j] = mma(a[i], b[j], c[s % CH][i][j]);
    }
};

template <>
struct Mfma<f16_t> {
    static constexpr int V = 8;
    static constexpr int BK = 64;
    __device__ __forceinline__ static f32x16 mma(const uint4& a, const uint4& b, f32x16 c) {
        f16x8 av, bv;
        __builtin_memcpy(&av, &a, 16);
        __builtin_memcpy(&bv, &b, 16);
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, c, 0, 0, 0);
    }
    static constexpr int kPerTile = 1;
    template <int TM, int TN, int CH>
    __device__ __forceinline__ static void tiles(const uint4 (&a)[TM], const uint4 (&b)[TN], f32x16 (&c)[CH][TM][TN],
                                                 int s) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) c[s % CH][i][j] = mma(a[i], b[j], c[s % CH][i][j]);
    }
};

template <>
struct Mfma<float> {
    static constexpr int V = 4;
    static constexpr int BK = 32;
    static constexpr int kPerTile = 4;
    // The four k of a fragment in order, a pass over the tiles for each, the
    // k-th on the k-th of CH accumulators: consecutive MFMAs do not wait on
    // one accumulator.
    template <int TM, int TN, int CH>
    __device__ __forceinline__ static void tiles(const uint4 (&a)[TM], const uint4 (&b)[TN], f32x16 (&c)[CH][TM][TN],
                                                 int) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const uint32_t u = k == 0 ? a[i].x : k == 1 ? a[i].y : k == 2 ? a[i].z : a[i].w;
                    const uint32_t v = k == 0 ? b[j].x : k == 1 ? b[j].y : k == 2 ? b[j].z : b[j].w;
                    f32x16& acc = c[k % CH][i][j];
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(u), __uint_as_float(v), acc, 0, 0, 0);
                }
    }
};

constexpr int kGroupM = 8;

// Stores of C bypass the caches' normal retention (non-temporal): a large
// product's output then does not evict the A and B panels later tiles read
// (bf16 linear 8192 x 4096 x 11008: 704-713 -> 656-670 us).
template <typename S>
__device__ __forceinline__ void put_c(S* dst, S v) {
    __builtin_nontemporal_store(v, dst);
}

// XCD-aware, L2-grouped tile order: blocks are dealt round-robin over the 8
// XCDs, and each XCD walks a contiguous range of tiles (the first total % 8
// one tile more) in groups of kGroupM tile rows.
__device__ __forceinline__ void tile_coords(int bid, int grid_m, int grid_n, int& pm, int& pn) {
    const int total = grid_m * grid_n;
    const int xcd = bid % 8, q = total / 8, rest = total % 8;
    const int pid = xcd * q + (xcd < rest ? xcd : rest) + bid / 8;
    const int in_group = kGroupM * grid_n;
    const int group = pid / in_group;
    const int first_m = group * kGroupM;
    const int size_m = grid_m - first_m < kGroupM ? grid_m - first_m : kGroupM;
    pm = first_m + (pid % in_group) % size_m;
    pn = (pid % in_group) / size_m;
}

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef short short4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), static_cast<short>(0), bytes,
                                             0x00020000);
}

// K-major: rows r and r + 8 (one 16-lane group) differ in the low bit of the
// slot; rows of one parity (the same half of a 256-byte bank line) take 8
// distinct slots.
__device__ __forceinline__ int kswz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// MF MFMAs with RD LDS reads and LD loads spread evenly between them.
template <int MF, int RD, int LD, int Q>
__device__ __forceinline__ void interleave_slot() {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    constexpr int r = RD * (Q + 1) / MF - RD * Q / MF;
    constexpr int l = LD * (Q + 1) / MF - LD * Q / MF;
    if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);
    if constexpr (l > 0) __builtin_amdgcn_sched_group_barrier(0x020, l, 0);
}
template <int MF, int RD, int LD, int... Q>
__device__ __forceinline__ void interleave_slots(std::integer_sequence<int, Q...>) {
    (interleave_slot<MF, RD, LD, Q>(), ...);
}
template <int MF, int RD, int LD>
__device__ __forceinline__ void interleave() {
    interleave_slots<MF, RD, LD>(std::make_integer_sequence<int, MF>{});
}

// One operand's panel of the tile kernel: R rows (M or N) by BK, 128 bytes of
// K, loaded straight into LDS by W waves (buffer loads of 16 bytes a lane,
// no registers in between) and read as NT 32-wide tiles a wave.  The buffer
// resource covers exactly what the block may read, and a load past it writes
// zeros, so ragged edges cost no branch:
//   * K-major (element (r, k) at X[r ld + k]): LDS rows of 128 bytes, the
//     16-byte chunk c of row r at slot c ^ kswz(r); chunks at or past K are
//     sent out of range lane by lane (they would read the next row).
//   * M/N-major (element (k, r) at X[k ld + r]): LDS rows (k) of R elements
//     as they lie.  16-bit ones are read by ds_read_b64_tr_b16, whose 32
//     lanes a clock take 64 bytes of four consecutive k: slots
//     c ^ (2 (k & 3) ^ 8 (k & 1)) put those on four quarters of the banks
//     (R of 128 and 256; rows of 64 take half a bank line each, and k and
//     k + 2 swap halves).  float32 ones are read as four single floats a
//     lane, the lane halves 4 rows of k apart: slots c ^ 8 ((k >> 2) & 1)
//     put the halves on opposite 32 banks.  Rows at or past K read zeros;
//     columns past R's edge read the next row's elements and only reach
//     outputs that are not stored.
// Operands are read where they lie, at any element: the loads need no
// alignment, but the resource's bound drops each of a load's four dwords that
// is not wholly inside it.  Without ODD, operands are whole dwords and whole
// packets of K, and that bound is exact.  With ODD the resource starts at the
// dword of the first element and ends at that of the last (an aligned dword
// never leaves the last element's page), and `finish_last` mends the last K
// tile in LDS: it zeroes what a packet or dword across K let in, and puts in
// the last element where that is the low half of a load's dword and so was
// dropped.
// One resource reaches 4 GiB.  With FAR (and ODD's rules) each row of a load
// has its own, so rows may be any distance apart, at the price of a load
// instruction a row.
enum class Rows { kWhole, kOdd, kFar };

template <typename T, bool KMAJOR, int R, int W, int NT, Rows ROWS>
struct Panel {
    static constexpr bool ODD = ROWS != Rows::kWhole, FAR = ROWS == Rows::kFar;
    using S = typename Elem<T>::storage;
    static constexpr int E = sizeof(S), V = 16 / E, BK = Mfma<T>::BK;
    static_assert(BK * E == 128, "a K tile is 128 bytes a row");
    static constexpr int kIssue = R / 8 / W;        // load instructions per wave per K tile
    static constexpr int kRowBytes = R * E;         // M/N-major LDS row
    static constexpr int kPerLoad = 1024 / kRowBytes;  // its rows per load instruction
    static constexpr int kFrags = KMAJOR ? 4 : NT;
    static_assert(kIssue * 8 * W == R, "the waves share a panel's loads evenly");
    // the slot of a lane's chunk must not depend on which of its loads it is
    static_assert(KMAJOR || E == 2 ? W % 2 == 0 : (W * kPerLoad) % 8 == 0, "swizzle period");
    // DS read instructions of one fragment set (two b64 or two paired b32
    // reads a tile when M/N-major)
    static constexpr int kReads = NT * (KMAJOR ? 1 : 2);

    const char* base;
    int64_t ld_bytes, bytes;  // bytes: readable from base (M/N-major: from k = 0)
    uint32_t voff, kleft;     // kleft: K-major, elements of K from this lane's chunk of K tile 0 on
    uint32_t coff, lead;      // FAR: the lane's offset in its row, bytes from base to the first element
    bool past_k, lost;        // the last K tile holds elements past K, lacks the last element
    uint32_t frag[kFrags];

    static __device__ __forceinline__ int slot_of(int c, int k) {
        if constexpr (R == 32) return c;
        else if constexpr (E == 4) return c ^ (8 * ((k >> 2) & 1));
        else if constexpr (R >= 128) return c ^ ((2 * (k & 3)) ^ (8 * (k & 1)));
        else return c ^ (4 * ((k >> 1) & 1));
    }

    __device__ __forceinline__ void init(const S* X, int64_t ld, int64_t r0, int64_t rows, int64_t K, int wave,
                                         int lane, int wbase) {
        const int l32 = lane % 32, half = lane / 32;
        ld_bytes = ld * E;
        if constexpr (KMAJOR) {
            const int64_t mine = rows - r0 < R ? rows - r0 : R;
            base = reinterpret_cast<const char*>(X) + r0 * ld_bytes;
            bytes = (mine - 1) * ld_bytes + K * E;
            past_k = ODD && K % V != 0;
            lost = ODD && E == 2 && K % 2 != 0;
            const int row = lane >> 3, chunk = (lane & 7) ^ kswz(8 * wave + row);
            voff = static_cast<uint32_t>((8 * wave + row) * ld_bytes + chunk * 16);
            coff = static_cast<uint32_t>(chunk * 16);
            kleft = static_cast<uint32_t>(K > chunk * V ? K - chunk * V : 0);
#pragma unroll
            for (int s = 0; s < 4; ++s) frag[s] = (wbase + l32) * 128 + (((2 * s + half) ^ kswz(l32)) << 4);
        } else {
            constexpr int kSlots = kRowBytes / 16;
            base = reinterpret_cast<const char*>(X + r0);
            bytes = (K - 1) * ld_bytes + (rows - r0) * E;
            past_k = ODD && E == 2 && K % BK != 0 && ((reinterpret_cast<uintptr_t>(base) + bytes) & 2) != 0;
            lost = ODD && E == 2 && (rows - r0) % 2 != 0 && rows - r0 <= R;
            const int k = wave * kPerLoad + lane / kSlots;
            voff = static_cast<uint32_t>(k * ld_bytes + slot_of(lane % kSlots, k) * 16);
            coff = static_cast<uint32_t>(slot_of(lane % kSlots, k) * 16);
            kleft = 0;
            if constexpr (E == 2) {
                // transposed reads: lane p of 16-lane group g addresses row
                // 8 half + p / 4 and column 16 (g & 1) + 4 (p % 4)
                const int g = lane / 16, pl = lane % 16;
                const int krow = 8 * half + pl / 4;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int col = wbase + t * 32 + 16 * (g & 1) + 4 * (pl % 4);
                    frag[t] = krow * kRowBytes + (slot_of(col / 8, krow) << 4) + (col % 8) * 2;
                }
            } else {
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int col = wbase + t * 32 + l32;
                    frag[t] = 4 * half * kRowBytes + (slot_of(col / 4, 4 * half) << 4) + (col % 4) * 4;
                }
            }
        }
        if constexpr (!ODD) return;
        // an odd count that ends on a dword began in the middle of one
        lost = lost && ((reinterpret_cast<uintptr_t>(base) + bytes) & 2) == 0;
        lead = reinterpret_cast<uintptr_t>(base) & 3;
        base -= lead;
        voff += lead;
        bytes = (bytes + lead + 3) / 4 * 4;
    }

    // Mends the last K tile; `left` = K's elements in it (1 .. BK), `extent`
    // = the panel's rows.
    __device__ __forceinline__ void finish_last(char* tile, int left, int64_t extent) const {
        const int r = threadIdx.x;
        if constexpr (KMAJOR) {
            if (past_k && r < R) {
                S* chunk = reinterpret_cast<S*>(tile + r * 128 + (((left / V) ^ kswz(r)) << 4));
                for (int e = left % V; e < V; ++e) chunk[e] = S{};
                if (lost && r == extent - 1) {
                    chunk[left % V - 1] = *reinterpret_cast<const S*>(base + bytes - E);
                }
            }
        } else {
            if (past_k && r < R) reinterpret_cast<S*>(tile + left * kRowBytes)[r] = S{};
            if (lost && r == extent - 1) {
                S* chunk = reinterpret_cast<S*>(tile + (left - 1) * kRowBytes + (slot_of(r / V, left - 1) << 4));
                chunk[r % V] = *reinterpret_cast<const S*>(base + bytes - E);
            }
        }
    }

    // Loads of K tile kt into `tile` (this wave's share); past the last K
    // tile every load is out of range.
    __device__ __forceinline__ void issue(int kt, char* tile, int wave) const {
        if constexpr (FAR) {
            issue_rows(kt, tile, wave);
            return;
        }
        uint32_t off;
        const char* from;
        int64_t left;
        if constexpr (KMAJOR) {
            from = base;
            left = bytes;
            const uint32_t k0 = static_cast<uint32_t>(kt) * BK;
            off = k0 < kleft ? voff + k0 * E : kOutOfRange;
        } else {
            const int64_t skip = static_cast<int64_t>(kt) * BK * ld_bytes;
            from = base + skip;
            left = bytes - skip;
            if (left < 0) left = 0;
            off = voff;
        }
        const uint32_t records = left < int64_t{kOutOfRange} ? static_cast<uint32_t>(left) : kOutOfRange;
        const __amdgpu_buffer_rsrc_t res = rsrc(from, records);
        const uint32_t step = static_cast<uint32_t>((KMAJOR ? 8 * W : W * kPerLoad) * ld_bytes);
#pragma unroll
        for (int i = 0; i < kIssue; ++i) {
            // an out-of-range lane stays so: its offset only needs not to wrap
            const uint32_t at = KMAJOR ? (off == kOutOfRange ? kOutOfRange : off + i * step) : off + i * step;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(res, (lds_ptr)(tile + (i * W + wave) * 1024), 16, at, 0, 0, 0);
        }
    }

    // The same with FAR: row by row, the lanes of one row a load.
    __device__ __forceinline__ void issue_rows(int kt, char* tile, int wave) const {
        constexpr int kRows = KMAJOR ? 8 : kPerLoad;
        const int row = threadIdx.x % kWave / (kWave / kRows);
        const int64_t k0 = static_cast<int64_t>(kt) * BK;
        const int64_t skip = lead + k0 * (KMAJOR ? E : ld_bytes);
        const bool in = !KMAJOR || k0 < kleft;
#pragma unroll
        for (int i = 0; i < kIssue; ++i) {
#pragma unroll 1
            for (int r = 0; r < kRows; ++r) {
                const int64_t at = skip + static_cast<int64_t>((i * W + wave) * kRows + r) * ld_bytes;
                const int64_t start = at & ~int64_t{3};
                const int64_t left = bytes > start ? bytes - start : 0;
                const uint32_t records = left < int64_t{kOutOfRange} ? static_cast<uint32_t>(left) : kOutOfRange;
                const __amdgpu_buffer_rsrc_t res = rsrc(base + start, records);
                const uint32_t off = in ? coff + static_cast<uint32_t>(at & 3) : kOutOfRange;
                if (row == r) {
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(res, (lds_ptr)(tile + (i * W + wave) * 1024), 16, off, 0, 0, 0);
                }
            }
        }
    }

    // The fragment of substep s for the wave's 32-wide tile t: 16 bytes of K
    // a lane.
    __device__ __forceinline__ uint4 read(const char* tile, int t, int s) const {
        if constexpr (KMAJOR) {
            return *reinterpret_cast<const uint4*>(tile + t * 32 * 128 + frag[s]);
        } else if constexpr (E == 2) {
            const char* q = tile + frag[t] + s * 16 * kRowBytes;
            const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(q));
            const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) short4_t*)(q + 4 * kRowBytes));
            uint4 v;
            __builtin_memcpy(&v, &lo, 8);
            __builtin_memcpy(reinterpret_cast<char*>(&v) + 8, &hi, 8);
            return v;
        } else {
            const char* q = tile + frag[t] + s * 8 * kRowBytes;
            uint4 v;
            v.x = *reinterpret_cast<const uint32_t*>(q);
            v.y = *reinterpret_cast<const uint32_t*>(q + kRowBytes);
            v.z = *reinterpret_cast<const uint32_t*>(q + 2 * kRowBytes);
            v.w = *reinterpret_cast<const uint32_t*>(q + 3 * kRowBytes);
            return v;
        }
    }
};

// F32OUT: C is float32 (split-K partials of a 16-bit product), written as
// alpha acc with no Cin.
//
// Four waves (2 x 2), a K step a 128-byte slab of K, STAGES LDS stages.  A
// step runs its four substeps' MFMAs with the next substep's fragment reads
// between them, and in the first the loads of the K tile STAGES - 1 ahead.
// After the third it waits until the next K tile's loads have landed (later
// tiles' stay in flight), passes the one barrier and reads the next step's
// first fragments under the last substep's MFMAs.  With two stages A of the
// tile after next goes out there too, into the stage just left.  Nothing but MFMAs stands
// between two barriers but the wait itself: the kernel this replaced staged
// tiles through registers and LDS stores, and its waves met at the end of
// each step with the matrix pipe idle (float32 4096^3 85 % busy).
// BLOCKS is how many blocks a CU holds (LDS and registers).
// ODD (see Panel) is a variant of its own: its test for the last K tile in
// the loop costs the others 3-8 % (float32 256 x 1024 x 4096 25.3 -> 27.4 us).
template <typename T, bool A_KMAJOR, bool B_KMAJOR, int BM, int BN, int STAGES, int BLOCKS, bool F32OUT, Rows ROWS>
__global__ __launch_bounds__(4 * kWave, BLOCKS) void gemm_tile_kernel(GemmArgs p) {
    using S = typename Elem<T>::storage;
    constexpr int WM = BM >= 64 ? 2 : 1, WN = 4 / WM, W = WM * WN;
    constexpr int BK = Mfma<T>::BK;
    constexpr int kWaveM = BM / WM, kWaveN = BN / WN;
    constexpr int TM = kWaveM / 32, TN = kWaveN / 32;
    using PA = Panel<T, A_KMAJOR, BM, W, TM, ROWS>;
    using PB = Panel<T, B_KMAJOR, BN, W, TN, ROWS>;
    constexpr bool ODD = PA::ODD;
    constexpr int ATILE = BM * 128, STAGE = (BM + BN) * 128;
    // An object a stage, so the compiler can tell the ones being filled from
    // the one being read and leaves the loads in flight.
    static_assert(STAGES >= 2 && STAGES <= 4, "LDS stages");
    __shared__ __attribute__((aligned(1024))) char lds0[STAGE];
    __shared__ __attribute__((aligned(1024))) char lds1[STAGE];
    __shared__ __attribute__((aligned(1024))) char lds2[STAGES > 2 ? STAGE : 16];
    __shared__ __attribute__((aligned(1024))) char lds3[STAGES > 3 ? STAGE : 16];
    auto stage_at = [&](auto i) -> char* {
        constexpr int I = decltype(i)::value % STAGES;
        if constexpr (I == 0) return lds0;
        else if constexpr (I == 1) return lds1;
        else if constexpr (I == 2) return lds2;
        else return lds3;
    };

    const int grid_m = static_cast<int>((p.m + BM - 1) / BM);
    const int grid_n = static_cast<int>((p.n + BN - 1) / BN);
    int pm, pn;
    tile_coords(blockIdx.x, grid_m, grid_n, pm, pn);
    const int64_t m0 = static_cast<int64_t>(pm) * BM, n0 = static_cast<int64_t>(pn) * BN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int wm = wave / WN, wn = wave % WN;
    const int half = lane / 32, l32 = lane % 32;

    // One batch entry per blockIdx.z (the host launches batches of at most
    // 65535).
    {
        const int64_t bi = blockIdx.z;
        // Split-K partials: batch entry bi is the slice k = bi k .. of the
        // product's k_total, the last one shorter when k does not divide it.
        const int64_t kk = F32OUT && p.k_total - bi * p.k < p.k ? p.k_total - bi * p.k : p.k;
        const int nk = static_cast<int>((kk + BK - 1) / BK);
        PA oa;
        PB ob;
        oa.init(static_cast<const S*>(p.a) + bi * p.stride_a, p.lda, m0, p.m, kk, wave, lane, wm * kWaveM);
        ob.init(static_cast<const S*>(p.b) + bi * p.stride_b, p.ldb, n0, p.n, kk, wave, lane, wn * kWaveN);
        // A wave of one or two 32 x 32 tiles sums each in four or two
        // interleaved accumulators, added at the end: its MFMAs do not queue
        // on one, and the sum's rounding error is that of a chain a fourth
        // or half as long.
        constexpr int CH = TM * TN == 1 ? 4 : TM * TN == 2 ? 2 : 1;
        f32x16 sums[CH][TM][TN];
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) sums[c][i][j][e] = 0.0f;

        uint4 af[2][TM], bf[2][TN];
        auto fetch = [&](const char* stage, int s, int buf) {
#pragma unroll
            for (int i = 0; i < TM; ++i) af[buf][i] = oa.read(stage, i, s);
#pragma unroll
            for (int j = 0; j < TN; ++j) bf[buf][j] = ob.read(stage + ATILE, j, s);
        };
        auto mma = [&](int s) { Mfma<T>::template tiles<TM, TN, CH>(af[s & 1], bf[s & 1], sums, s); };
        constexpr int kMf = TM * TN * Mfma<T>::kPerTile;
        constexpr int kReads = PA::kReads + PB::kReads;
        // The loads a wave may leave in flight when it passes the barrier of a
        // step: those of the K tiles after the next.
        constexpr int kAhead = (STAGES - 2) * (PA::kIssue + PB::kIssue);
        constexpr int kWait = (kAhead & 15) | (7 << 4) | ((kAhead >> 4) << 14);  // vmcnt(kAhead) lgkmcnt(0)
        auto meet = [&]() {
            __builtin_amdgcn_s_waitcnt(kWait);
            // A bare barrier: the fence of __syncthreads() would wait for
            // every load.
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        const bool mend = ODD && (oa.past_k || oa.lost || ob.past_k || ob.lost);
        auto finish = [&](char* last) {
            if constexpr (!ODD) return;
            const int left = static_cast<int>(kk - static_cast<int64_t>(nk - 1) * BK);
            oa.finish_last(last, left, p.m - m0 < BM ? p.m - m0 : BM);
            ob.finish_last(last + ATILE, left, p.n - n0 < BN ? p.n - n0 : BN);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the stores are in LDS
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        auto body = [&](auto at, int kt) {
            constexpr int I = decltype(at)::value;
            char* cur = stage_at(std::integral_constant<int, I>{});
            char* next = stage_at(std::integral_constant<int, I + 1>{});
            char* fill = stage_at(std::integral_constant<int, I + STAGES - 1>{});
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                fetch(cur, s + 1, (s + 1) & 1);
                if (s == 0) {
                    if (STAGES > 2) oa.issue(kt + STAGES - 1, fill, wave);
                    ob.issue(kt + STAGES - 1, fill + ATILE, wave);
                }
                mma(s);
                if (s == 0) {
                    interleave<kMf, kReads, PB::kIssue + (STAGES > 2 ? PA::kIssue : 0)>();
                } else {
                    interleave<kMf, kReads, 0>();
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            meet();
            if (mend && kt + 2 == nk) finish(next);
            fetch(next, 0, 0);
            if (STAGES == 2) oa.issue(kt + 2, cur, wave);
            mma(3);
            interleave<kMf, kReads, STAGES == 2 ? PA::kIssue : 0>();
            __builtin_amdgcn_sched_barrier(0);
        };
        auto prologue = [&](auto i) {
            constexpr int I = decltype(i)::value;
            if constexpr (I < STAGES - 1) {
                oa.issue(I, stage_at(i), wave);
                ob.issue(I, stage_at(i) + ATILE, wave);
            } else if constexpr (STAGES == 2) {
                oa.issue(1, lds1, wave);
            }
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        using I3 = std::integral_constant<int, 3>;
        prologue(I0{});
        prologue(I1{});
        if constexpr (STAGES > 2) prologue(I2{});
        meet();
        if (mend && nk == 1) finish(lds0);
        fetch(lds0, 0, 0);
        for (int kt = 0; kt < nk; kt += STAGES) {
            body(I0{}, kt);
            if (kt + 1 >= nk) break;
            body(I1{}, kt + 1);
            if constexpr (STAGES > 2) {
                if (kt + 2 >= nk) break;
                body(I2{}, kt + 2);
            }
            if constexpr (STAGES > 3) {
                if (kt + 3 >= nk) break;
                body(I3{}, kt + 3);
            }
        }
        // the last steps' out-of-range loads still write LDS
        __builtin_amdgcn_s_waitcnt(0);
        f32x16 (&acc)[TM][TN] = sums[0];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (CH == 2) acc[i][j] += sums[1][i][j];
                if constexpr (CH == 4) acc[i][j] = (acc[i][j] + sums[1][i][j]) + (sums[2][i][j] + sums[3][i][j]);
            }

        // Epilogue: lane holds column l32 of each 32 x 32 tile, rows
        // 8 * (e / 4) + 4 * half + e % 4 for accumulator element e.
        if constexpr (F32OUT) {
            float* C = static_cast<float*>(p.c) + bi * p.stride_c;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int64_t col = n0 + wn * kWaveN + j * 32 + l32;
                    const int64_t rbase = m0 + wm * kWaveM + i * 32 + 4 * half;
                    if (col >= p.n) continue;
#pragma unroll
                    for (int g = 0; g < 4; ++g)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int64_t row = rbase + 8 * g + r;
                            if (row < p.m) C[row * p.ldc + col] = p.alpha * acc[i][j][4 * g + r];
                        }
                }
            return;
        }
        S* C = static_cast<S*>(p.c) + bi * p.stride_c;
        const S* Cin = static_cast<const S*>(p.cin);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int64_t col = n0 + wn * kWaveN + j * 32 + l32;
                const int64_t rbase = m0 + wm * kWaveM + i * 32 + 4 * half;
                if (col >= p.n) continue;
                S* cp = C + rbase * p.ldc + col;
                if (p.beta == 0.0f) {
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            if (rbase + 8 * g + r < p.m) {
                                put_c(&cp[r * p.ldc], Elem<T>::store(p.alpha * acc[i][j][4 * g + r]));
                            }
                        }
                        cp += 8 * p.ldc;
                    }
                } else if (p.cin_rs == 0) {
                    // A bias along N (addmm / linear): one value per column.
                    const float c = p.beta * Elem<T>::load(Cin[bi * p.cin_stride_b + col * p.cin_cs]);
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            if (rbase + 8 * g + r < p.m) {
                                put_c(&cp[r * p.ldc], Elem<T>::store(fmaf(p.alpha, acc[i][j][4 * g + r], c)));
                            }
                        }
                        cp += 8 * p.ldc;
                    }
                } else {
                    const S* ci = Cin + bi * p.cin_stride_b + rbase * p.cin_rs + col * p.cin_cs;
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            if (rbase + 8 * g + r < p.m) {
                                const float c = Elem<T>::load(ci[r * p.cin_rs]);
                                put_c(&cp[r * p.ldc],
                                      Elem<T>::store(fmaf(p.beta, c, p.alpha * acc[i][j][4 * g + r])));
                            }
                        }
                        cp += 8 * p.ldc;
                        ci += 8 * p.cin_rs;
                    }
                }
            }
    }
}

namespace big {

// 256 x 256 x 64 tiles over WM x WN waves (2 x 2 waves of 128 x 128, or
// 2 x 4 of 128 x 64), every tile full.
//
// Operand tiles move from memory straight into LDS with buffer loads (16
// bytes a lane, no registers in between).  Each operand tile is 32 KB in one
// of two layouts, swizzled for gfx950's LDS of 64 four-byte banks (256 bytes
// a clock); both read at zero SQ_LDS_BANK_CONFLICT in every layout, which is
// what settles a swizzle here (the reasoning below, 16 lanes of a
// ds_read_b128 and 32 of an 8-byte read a clock, explains these two but is
// not a complete model of the hardware):
//   * K-major operand: 256 rows (M or N) of 128 bytes, one row = the tile's
//     64 k; logical 16-byte chunk c of row r sits at slot c ^ kswz(r).  A
//     load instruction fills 8 rows; a fragment read (ds_read_b128: 32 rows,
//     one chunk) puts each 16-lane group's 16 rows on 64 distinct banks.
//   * M/N-major operand (a transposed view, read in place): 64 rows (k) of
//     512 bytes, chunk c of row k at slot c ^ nswz(k).  A load instruction
//     fills 2 rows.  Fragments come from ds_read_b64_tr_b16, which hands
//     each lane of a 16-lane group one column of a 4 x 16 block: two of them
//     give a lane its 8 consecutive k; the 4 rows x 64 bytes that 32 lanes
//     read fall on 64 distinct banks.
// Both swizzles also keep 8 lanes of a b128 read (16 of a b64 read) on 32
// distinct banks.
// The loads for K tile kt + 1 go out during the first half of step kt into
// the other LDS stage, spread between the MFMAs.
constexpr int BM = 256, BN = 256, BK = 64;
constexpr int TILE = 256 * 128;   // bytes per operand tile
constexpr int STAGE = 2 * TILE;   // bytes per LDS stage
// M/N-major: rows k..k+3 move a 4-chunk span (64 bytes) to four distinct
// quarters of a bank line, and a 2-chunk span to four distinct slots mod 8.
__device__ __forceinline__ int nswz(int k) { return (2 * (k & 3)) ^ (8 * (k & 1)); }

// One operand: the block's 256-wide panel of X (M or N from mn0), loaded by
// W waves, read as T 32-wide tiles per wave.
template <bool KMAJOR, int W, int T>
struct Operand {
    static constexpr int kIssue = 32 / W;  // load instructions per wave per K tile
    __amdgpu_buffer_rsrc_t res;
    uint32_t voff, sbase, sstep, kstep;
    int frag[4];       // per-lane fragment byte offsets (K-major: per substep; M/N-major: per tile)

    __device__ __forceinline__ void init(const void* X, int64_t ld, int64_t mn0, int64_t K, int wave,
                                         int lane, int wbase) {
        const int l32 = lane % 32, half = lane / 32;
        if constexpr (KMAJOR) {
            // element (r, k) at X[r * ld + k]; a load's lane L fills slot L % 8
            // of row L / 8 of its 8-row group
            res = rsrc(static_cast<const uint16_t*>(X) + mn0 * ld, static_cast<uint32_t>(256 * ld * 2));
            const int row = lane >> 3, chunk = (lane & 7) ^ kswz(8 * wave + row);
            voff = static_cast<uint32_t>((row * ld + chunk * 8) * 2);
            sbase = static_cast<uint32_t>(wave * 8 * ld * 2);
            sstep = static_cast<uint32_t>(W * 8 * ld * 2);
            kstep = BK * 2;
#pragma unroll
            for (int s = 0; s < 4; ++s)
                frag[s] = (wbase + l32) * 128 + (((2 * s + half) ^ kswz(l32)) << 4);
        } else {
            // element (k, r) at X[k * ld + r]; a load fills 2 rows of k
            res = rsrc(static_cast<const uint16_t*>(X) + mn0, static_cast<uint32_t>(K * ld * 2));
            const int row = lane >> 5;
            const int chunk = (lane & 31) ^ nswz(2 * (wave & 1) + row);
            voff = static_cast<uint32_t>((row * ld + chunk * 8) * 2);
            sbase = static_cast<uint32_t>(2 * wave * ld * 2);
            sstep = static_cast<uint32_t>(2 * W * ld * 2);
            kstep = static_cast<uint32_t>(BK * ld * 2);
            // Transposed reads: lane p of 16-lane group g addresses row
            // 8 * half + p / 4 (+ 16 s + 4 h) and column 16 (g & 1) + 4 (p % 4)
            // of the wave's 32-wide tile t.
            const int g = lane / 16, pl = lane % 16;
            const int krow = 8 * half + pl / 4;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const int col = wbase + t * 32 + 16 * (g & 1) + 4 * (pl % 4);
                frag[t] = krow * 512 + (((col / 8) ^ nswz(krow)) << 4) + (col % 8) * 2;
            }
        }
    }

    // Loads of K tile kt into `tile` (this wave's share of the 32 instructions).
    __device__ __forceinline__ void issue(int kt, char* tile, int wave) const {
        const uint32_t kb = static_cast<uint32_t>(kt) * kstep;
#pragma unroll
        for (int i = 0; i < kIssue; ++i) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(res, (lds_ptr)(tile + (i * W + wave) * 1024), 16, voff,
                                                     sbase + i * sstep + kb, 0, 0);
        }
    }

    // The 8 k of substep s for the wave's 32-wide tile t.
    __device__ __forceinline__ uint4 read(const char* tile, int t, int s) const {
        if constexpr (KMAJOR) {
            return *reinterpret_cast<const uint4*>(tile + t * 32 * 128 + frag[s]);
        } else {
            const char* q = tile + frag[t] + s * 16 * 512;
            const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(q));
            const short4_t hi =
                __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t*)(q + 4 * 512));
            uint4 v;
            __builtin_memcpy(&v, &lo, 8);
            __builtin_memcpy(reinterpret_cast<char*>(&v) + 8, &hi, 8);
            return v;
        }
    }
};

template <typename T, bool A_KMAJOR, bool B_KMAJOR, int WM, int WN>
__global__ __launch_bounds__(WM * WN * kWave, (WM * WN) / 4) void gemm_big_kernel(GemmArgs p) {
    using S = typename Elem<T>::storage;
    static_assert(sizeof(S) == 2, "16-bit operands");
    constexpr int W = WM * WN;
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
    // Two LDS objects rather than one array: the compiler can then tell that
    // the loads filling one stage do not touch the stage being read, and
    // leaves them in flight across the step.
    __shared__ __attribute__((aligned(1024))) char lds0[STAGE];
    __shared__ __attribute__((aligned(1024))) char lds1[STAGE];

    const int grid_m = static_cast<int>(p.m / BM), grid_n = static_cast<int>(p.n / BN);
    int pm, pn;
    tile_coords(blockIdx.x, grid_m, grid_n, pm, pn);
    const int64_t m0 = static_cast<int64_t>(pm) * BM, n0 = static_cast<int64_t>(pn) * BN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int wm = wave / WN, wn = wave % WN;
    const int l32 = lane % 32, half = lane / 32;
    const int nk = static_cast<int>(p.k / BK);
    const int64_t bi = blockIdx.z;

    Operand<A_KMAJOR, W, TM> oa;
    Operand<B_KMAJOR, W, TN> ob;
    oa.init(static_cast<const S*>(p.a) + bi * p.stride_a, p.lda, m0, p.k, wave, lane, wm * TM * 32);
    ob.init(static_cast<const S*>(p.b) + bi * p.stride_b, p.ldb, n0, p.k, wave, lane, wn * TN * 32);

    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    uint4 af[2][TM], bf[2][TN];
    auto fetch = [&](const char* stage, int s, int buf) {
#pragma unroll
        for (int i = 0; i < TM; ++i) af[buf][i] = oa.read(stage, i, s);
#pragma unroll
        for (int j = 0; j < TN; ++j) bf[buf][j] = ob.read(stage + TILE, j, s);
    };
    auto mma = [&](int buf) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = Mfma<T>::mma(af[buf][i], bf[buf][j], acc[i][j]);
    };
    // Per substep: TM x TN MFMAs, and a b128 fragment read per K-major tile
    // or two transposed b64 reads per M/N-major one.
    constexpr int kMf = TM * TN;
    constexpr int kReads = TM * (A_KMAJOR ? 1 : 2) + TN * (B_KMAJOR ? 1 : 2);
    // One K step out of `cur`, entered with substep 0's fragments in
    // flight.  Substeps 0-2 each run their MFMAs interleaved with the next
    // substep's fragment reads (and, in substep 0, this wave's loads of B
    // for the next K tile).  The step then waits for its loads and the
    // barrier, and starts reading the next step's first fragments before
    // running substep 3's MFMAs, whose operands are in registers.  After
    // that barrier no wave reads `cur` again, so substep 3 also issues the
    // loads of A for the K tile after next into it: A's loads get four
    // substeps to land and B's three, against three and two when both went
    // out in substeps 0 and 1 (bf16 linear 8192 x 4096 x 11008 733 -> 706 us
    // on average over three alternating runs, 4096^3 1-2 % faster, the same
    // bits).
    // do_issue: load B of K tile kt_next into `next`; issue_a: load A of
    // K tile kt_next + 1 into `cur` after the barrier.
    auto body = [&](char* cur, char* next, int kt_next, auto do_issue, auto has_next, auto issue_a) {
        constexpr bool kIssue = decltype(do_issue)::value;
        constexpr bool kIssueA = decltype(issue_a)::value;
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            fetch(cur, s + 1, (s + 1) & 1);
            if constexpr (kIssue) {
                if (s == 0) ob.issue(kt_next, next + TILE, wave);
            }
            mma(s & 1);
            if (kIssue && s == 0) {
                interleave<kMf, kReads, 32 / W>();
            } else {
                interleave<kMf, kReads, 0>();
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (decltype(has_next)::value) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            fetch(next, 0, 0);
            if constexpr (kIssueA) oa.issue(kt_next + 1, cur, wave);
            mma(1);
            interleave<kMf, kReads, kIssueA ? 32 / W : 0>();
        } else {
            mma(1);
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // K tile 0 whole, and A of K tile 1 (the host guarantees nk >= 2).
    oa.issue(0, lds0, wave);
    ob.issue(0, lds0 + TILE, wave);
    oa.issue(1, lds1, wave);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    fetch(lds0, 0, 0);
    // Steps in pairs (stage 0 then stage 1), so every access names its LDS
    // object statically; the host guarantees an even number of K tiles.
    // Inside the loop kt + 3 <= nk - 1, so A of K tile kt_next + 1 exists.
    for (int kt = 0; kt + 2 < nk; kt += 2) {
        body(lds0, lds1, kt + 1, std::true_type{}, std::true_type{}, std::true_type{});
        body(lds1, lds0, kt + 2, std::true_type{}, std::true_type{}, std::true_type{});
    }
    body(lds0, lds1, nk - 1, std::true_type{}, std::true_type{}, std::false_type{});
    body(lds1, lds0, 0, std::false_type{}, std::false_type{}, std::false_type{});

    // Epilogue: lane holds column l32 of each 32 x 32 tile, rows
    // 8 * (e / 4) + 4 * half + e % 4 for accumulator element e.
    S* C = static_cast<S*>(p.c) + bi * p.stride_c;
    const S* Cin = static_cast<const S*>(p.cin);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int64_t col = n0 + wn * TN * 32 + j * 32 + l32;
            const int64_t rbase = m0 + wm * TM * 32 + i * 32 + 4 * half;
            S* cp = C + rbase * p.ldc + col;
            if (p.beta == 0.0f) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) put_c(&cp[r * p.ldc], Elem<T>::store(p.alpha * acc[i][j][4 * g + r]));
                    cp += 8 * p.ldc;
                }
            } else if (p.cin_rs == 0) {
                const float c = p.beta * Elem<T>::load(Cin[bi * p.cin_stride_b + col * p.cin_cs]);
#pragma unroll
                for (int g = 0; g < 4; ++g) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) put_c(&cp[r * p.ldc], Elem<T>::store(fmaf(p.alpha, acc[i][j][4 * g + r], c)));
                    cp += 8 * p.ldc;
                }
            } else {
                const S* ci = Cin + bi * p.cin_stride_b + rbase * p.cin_rs + col * p.cin_cs;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float c = Elem<T>::load(ci[r * p.cin_rs]);
                        put_c(&cp[r * p.ldc], Elem<T>::store(fmaf(p.beta, c, p.alpha * acc[i][j][4 * g + r])));
                    }
                    cp += 8 * p.ldc;
                    ci += 8 * p.cin_rs;
                }
            }
        }
}

template <typename T>
bool eligible(const GemmArgs& p, int cus) {
    const bool a_kmajor = !p.trans_a, b_kmajor = p.trans_b;
    // A block addresses its panel through one buffer resource: 256 rows of
    // ld (K-major, needs ld >= K) or K rows of ld (M/N-major, needs
    // ld >= 256), under 4 GiB.
    auto panel_ok = [&](const void* x, int64_t ld, int64_t stride, bool kmajor) {
        const int64_t bytes = kmajor ? 256 * ld * 2 : p.k * ld * 2;
        return aligned16(x) && ld % 8 == 0 && stride % 8 == 0 && bytes < (int64_t(1) << 32) &&
               (kmajor ? ld >= p.k : ld >= 256);
    };
    return p.m % BM == 0 && p.n % BN == 0 && p.k % (2 * BK) == 0 &&
           panel_ok(p.a, p.lda, p.stride_a, a_kmajor) && panel_ok(p.b, p.ldb, p.stride_b, b_kmajor) &&
           (p.m / BM) * (p.n / BN) * p.batch >= cus && (p.m / BM) * (p.n / BN) < (int64_t(1) << 31);
}

template <typename T, int WM, int WN>
void launch_shape(const GemmArgs& whole, hipStream_t stream) {
    constexpr int64_t kMaxZ = 65535;
    using S = typename Elem<T>::storage;
    const bool a_kmajor = !whole.trans_a, b_kmajor = whole.trans_b;
    for (int64_t b0 = 0; b0 < whole.batch; b0 += kMaxZ) {
        GemmArgs p = whole;
        p.batch = whole.batch - b0 < kMaxZ ? whole.batch - b0 : kMaxZ;
        p.a = static_cast<const S*>(whole.a) + b0 * whole.stride_a;
        p.b = static_cast<const S*>(whole.b) + b0 * whole.stride_b;
        p.c = static_cast<S*>(whole.c) + b0 * whole.stride_c;
        if (whole.cin != nullptr) p.cin = static_cast<const S*>(whole.cin) + b0 * whole.cin_stride_b;
        const dim3 grid(static_cast<unsigned>((p.m / BM) * (p.n / BN)), 1u, static_cast<unsigned>(p.batch));
        constexpr int THREADS = WM * WN * kWave;
        if (a_kmajor && b_kmajor) {
            gemm_big_kernel<T, true, true, WM, WN><<<grid, THREADS, 0, stream>>>(p);
        } else if (a_kmajor) {
            gemm_big_kernel<T, true, false, WM, WN><<<grid, THREADS, 0, stream>>>(p);
        } else if (b_kmajor) {
            gemm_big_kernel<T, false, true, WM, WN><<<grid, THREADS, 0, stream>>>(p);
        } else {
            gemm_big_kernel<T, false, false, WM, WN><<<grid, THREADS, 0, stream>>>(p);
        }
        TP_AMD_HIP_CHECK(hipGetLastError());
    }
}

// Four waves of 128 x 128 for long K.  With K <= 256 (two to four K steps:
// bmm of attention-sized products) the prologue and the epilogue dominate,
// and eight waves of 128 x 64 -- two per SIMD -- overlap them: bf16
// 64 x 512 x 128 x 512 bmm 15.9 -> 13.5 us.  At 4096^3 the two shapes
// measure the same.
template <typename T>
void launch(const GemmArgs& p, hipStream_t stream) {
    if (p.k <= 256) {
        launch_shape<T, 2, 4>(p, stream);
    } else {
        launch_shape<T, 2, 2>(p, stream);
    }
}

}  // namespace big

// Short products (16-bit, K = 64 or 128: attention-sized bmm) are bound by
// storing C, not by the MFMAs: bf16 64 x 512 x 128 x 512 reads 16 MB and
// writes 32 MB.  Here all of K goes into LDS at once (one or two of the big
// kernel's stages, same layouts), one barrier, and each of the 8 waves then
// works through its 128 x 64 patch one 32 x 32 tile at a time -- the tile's
// MFMAs over all of K, then its stores -- so the stores of one tile drain
// while the MFMAs of the next run, instead of all of C going out after all
// the products.  The grid is one dimension over batch x tiles, numbered so a
// batch's tiles (which share A and B panels) stay on one XCD and its L2.
// Measured on the config-5a bmm against the big kernel on the same box:
// 12.5 against 15.6 us (rocprof), hipBLASLt 15.0 us.
namespace smallk {

constexpr int W = 8, WN = 4, TM = 4, TN = 2;

template <typename T, bool A_KMAJOR, bool B_KMAJOR>
__global__ __launch_bounds__(W * kWave, 1) void gemm_smallk_kernel(GemmArgs p) {
    using S = typename Elem<T>::storage;
    using big::BK;
    using big::STAGE;
    using big::TILE;
    __shared__ __attribute__((aligned(1024))) char lds0[STAGE];
    __shared__ __attribute__((aligned(1024))) char lds1[STAGE];
    const int grid_n = static_cast<int>(p.n / big::BN);
    const int tiles = static_cast<int>(p.m / big::BM) * grid_n;
    const int total = static_cast<int>(gridDim.x);
    const int pid = total % 8 == 0 ? (blockIdx.x % 8) * (total / 8) + blockIdx.x / 8 : blockIdx.x;
    const int64_t bi = pid / tiles;
    const int tile = pid % tiles;
    const int64_t m0 = static_cast<int64_t>(tile / grid_n) * big::BM;
    const int64_t n0 = static_cast<int64_t>(tile % grid_n) * big::BN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int wm = wave / WN, wn = wave % WN;
    const int l32 = lane % 32, half = lane / 32;
    const int nk = static_cast<int>(p.k / BK);
    big::Operand<A_KMAJOR, W, TM> oa;
    big::Operand<B_KMAJOR, W, TN> ob;
    oa.init(static_cast<const S*>(p.a) + bi * p.stride_a, p.lda, m0, p.k, wave, lane, wm * TM * 32);
    ob.init(static_cast<const S*>(p.b) + bi * p.stride_b, p.ldb, n0, p.k, wave, lane, wn * TN * 32);
    oa.issue(0, lds0, wave);
    ob.issue(0, lds0 + TILE, wave);
    if (nk > 1) {
        oa.issue(1, lds1, wave);
        ob.issue(1, lds1 + TILE, wave);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    S* C = static_cast<S*>(p.c) + bi * p.stride_c;
    const S* Cin = static_cast<const S*>(p.cin);
    // Tiles in a fixed order, fully unrolled, so every fragment offset is
    // static; the scheduling barrier keeps the next tile's reads out of this
    // one's stores (otherwise the registers run out and spill).
#pragma unroll
    for (int t = 0; t < TM * TN; ++t) {
        __builtin_amdgcn_sched_barrier(0);
        const int i = t % TM, j = t / TM;
        f32x16 acc;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
        for (int kt = 0; kt < nk; ++kt) {
            const char* st = kt == 0 ? lds0 : lds1;
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = Mfma<T>::mma(oa.read(st, i, s), ob.read(st + TILE, j, s), acc);
        }
        const int64_t col = n0 + wn * TN * 32 + j * 32 + l32;
        const int64_t rbase = m0 + wm * TM * 32 + i * 32 + 4 * half;
        S* cp = C + rbase * p.ldc + col;
        if (p.beta == 0.0f) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
#pragma unroll
                for (int r = 0; r < 4; ++r) put_c(&cp[r * p.ldc], Elem<T>::store(p.alpha * acc[4 * g + r]));
                cp += 8 * p.ldc;
            }
        } else if (p.cin_rs == 0) {
            const float c = p.beta * Elem<T>::load(Cin[bi * p.cin_stride_b + col * p.cin_cs]);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
#pragma unroll
                for (int r = 0; r < 4; ++r) put_c(&cp[r * p.ldc], Elem<T>::store(fmaf(p.alpha, acc[4 * g + r], c)));
                cp += 8 * p.ldc;
            }
        } else {
            const S* ci = Cin + bi * p.cin_stride_b + rbase * p.cin_rs + col * p.cin_cs;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float c = Elem<T>::load(ci[r * p.cin_rs]);
                    put_c(&cp[r * p.ldc], Elem<T>::store(fmaf(p.beta, c, p.alpha * acc[4 * g + r])));
                }
                cp += 8 * p.ldc;
                ci += 8 * p.cin_rs;
            }
        }
    }
}

// K of one or two 64-deep stages, full 256 x 256 tiles, the big kernel's
// panel rules, and enough tiles to give every CU one.
template <typename T>
bool eligible(const GemmArgs& p, int cus) {
    const bool a_kmajor = !p.trans_a, b_kmajor = p.trans_b;
    auto panel_ok = [&](const void* x, int64_t ld, int64_t stride, bool kmajor) {
        const int64_t bytes = kmajor ? 256 * ld * 2 : p.k * ld * 2;
        return aligned16(x) && ld % 8 == 0 && stride % 8 == 0 && bytes < (int64_t(1) << 32) &&
               (kmajor ? ld >= p.k : ld >= 256);
    };
    const int64_t tiles = (p.m / big::BM) * (p.n / big::BN) * p.batch;
    return (p.k == 64 || p.k == 128) && p.m % big::BM == 0 && p.n % big::BN == 0 &&
           panel_ok(p.a, p.lda, p.stride_a, a_kmajor) && panel_ok(p.b, p.ldb, p.stride_b, b_kmajor) &&
           tiles >= cus && tiles < (int64_t(1) << 31);
}

template <typename T>
void launch(const GemmArgs& p, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>((p.m / big::BM) * (p.n / big::BN) * p.batch));
    const bool a_kmajor = !p.trans_a, b_kmajor = p.trans_b;
    if (a_kmajor && b_kmajor) {
        gemm_smallk_kernel<T, true, true><<<grid, W * kWave, 0, stream>>>(p);
    } else if (a_kmajor) {
        gemm_smallk_kernel<T, true, false><<<grid, W * kWave, 0, stream>>>(p);
    } else if (b_kmajor) {
        gemm_smallk_kernel<T, false, true><<<grid, W * kWave, 0, stream>>>(p);
    } else {
        gemm_smallk_kernel<T, false, false><<<grid, W * kWave, 0, stream>>>(p);
    }
    TP_AMD_HIP_CHECK(hipGetLastError());
}

}  // namespace smallk

// Whether an operand's panel (a tile's rows of K, or a K tile of rows) lies
// under 4 GiB, the reach of one buffer resource.
template <typename T>
bool panel_near(int64_t ld, bool kmajor) {
    constexpr int64_t E = sizeof(typename Elem<T>::storage);
    const int64_t rows = kmajor ? 128 : Mfma<T>::BK;  // the tallest tile, or a K tile
    return ld < ((int64_t{1} << 32) - 4096) / (rows * E);
}

template <typename T>
bool rows_far(const GemmArgs& p) {
    return !panel_near<T>(p.lda, !p.trans_a) || !panel_near<T>(p.ldb, p.trans_b);
}

// The grid's limit, and the panels' 32-bit K (one product of a longer K is
// always split).
bool tiles_fit(const GemmArgs& p) {
    return (p.m + 63) / 64 * ((p.n + 63) / 64) < (int64_t(1) << 31) && (p.k < (int64_t(1) << 32) || p.batch == 1);
}

// Whole dwords everywhere and whole packets along K: the tile kernel without
// ODD.  (A split's slices but the last are whole K tiles.)
template <typename T>
bool whole_dwords(const void* x, int64_t ld, int64_t stride, bool kmajor, int64_t mn, int64_t k) {
    constexpr int64_t E = sizeof(typename Elem<T>::storage);
    if (kmajor && k % Mfma<T>::V != 0) return false;
    return E == 4 || (reinterpret_cast<uintptr_t>(x) % 4 == 0 && ld % 2 == 0 && stride % 2 == 0 && (kmajor || mn % 2 == 0));
}

template <typename T, int BM, int BN, int STAGES, int BLOCKS, bool F32OUT, Rows ROWS>
void launch_chunk(const GemmArgs& p, hipStream_t stream) {
    constexpr int THREADS = 4 * kWave;
    const int64_t tiles = ((p.m + BM - 1) / BM) * ((p.n + BN - 1) / BN);
    const dim3 grid(static_cast<unsigned>(tiles), 1u, static_cast<unsigned>(p.batch));
    const bool a_kmajor = !p.trans_a, b_kmajor = p.trans_b;
    if (a_kmajor && b_kmajor) {
        gemm_tile_kernel<T, true, true, BM, BN, STAGES, BLOCKS, F32OUT, ROWS><<<grid, THREADS, 0, stream>>>(p);
    } else if (a_kmajor) {
        gemm_tile_kernel<T, true, false, BM, BN, STAGES, BLOCKS, F32OUT, ROWS><<<grid, THREADS, 0, stream>>>(p);
    } else if (b_kmajor) {
        gemm_tile_kernel<T, false, true, BM, BN, STAGES, BLOCKS, F32OUT, ROWS><<<grid, THREADS, 0, stream>>>(p);
    } else {
        gemm_tile_kernel<T, false, false, BM, BN, STAGES, BLOCKS, F32OUT, ROWS><<<grid, THREADS, 0, stream>>>(p);
    }
    TP_AMD_HIP_CHECK(hipGetLastError());
}

template <typename T, int BM, int BN, int STAGES, int BLOCKS, bool F32OUT = false>
void launch_config(const GemmArgs& whole, hipStream_t stream) {
    constexpr int64_t kMaxZ = 65535;
    using S = typename Elem<T>::storage;
    for (int64_t b0 = 0; b0 < whole.batch; b0 += kMaxZ) {
        GemmArgs p = whole;
        p.batch = whole.batch - b0 < kMaxZ ? whole.batch - b0 : kMaxZ;
        p.a = static_cast<const S*>(whole.a) + b0 * whole.stride_a;
        p.b = static_cast<const S*>(whole.b) + b0 * whole.stride_b;
        p.c = F32OUT ? static_cast<void*>(static_cast<float*>(whole.c) + b0 * whole.stride_c)
                     : static_cast<void*>(static_cast<S*>(whole.c) + b0 * whole.stride_c);
        if (whole.cin != nullptr) p.cin = static_cast<const S*>(whole.cin) + b0 * whole.cin_stride_b;
        if (F32OUT) p.k_total = whole.k_total - b0 * whole.k;
        const int64_t k = F32OUT ? p.k_total : p.k;
        if (rows_far<T>(p)) {
            constexpr bool kSlices128 = F32OUT && BM == 128 && STAGES == 3;
            if constexpr ((BM == 64 && BN == 64) || kSlices128) launch_chunk<T, BM, BN, STAGES, BLOCKS, F32OUT, Rows::kFar>(p, stream);
            else TP_AMD_CHECK(false, "a tile that cannot take rows this far apart");
        } else if (whole_dwords<T>(p.a, p.lda, p.stride_a, !p.trans_a, p.m, k) &&
                   whole_dwords<T>(p.b, p.ldb, p.stride_b, p.trans_b, p.n, k)) {
            launch_chunk<T, BM, BN, STAGES, BLOCKS, F32OUT, Rows::kWhole>(p, stream);
        } else {
            launch_chunk<T, BM, BN, STAGES, BLOCKS, F32OUT, Rows::kOdd>(p, stream);
        }
    }
}
constexpr int kFinishBlock = 256;

// c = alpha * sum of the slices (+ beta Cin), the same expressions as the
// kernels' epilogue, rounded once to the output type.  A thread takes V
// consecutive columns of a row (V = 4 when the row length, ldc and C's
// address allow whole vectors, else 1) and adds slice 0 + slice 1 + ... in
// slice order, four slices' loads out at a time.  blockIdx.y walks the rows,
// so no index is divided.  Float32 partials just written: bound by the
// launch and one round trip (256 x 4096 in 4 slices 9.2 us with one element a
// thread and 64-bit divisions, 4.0 us so).
template <typename T, int V>
__global__ __launch_bounds__(kFinishBlock) void splitk_finish_kernel(
    const float* part, int slices, int64_t m, int64_t n, float alpha, float beta,
    const typename Elem<T>::storage* cin, int64_t cin_rs, int64_t cin_cs, typename Elem<T>::storage* c,
    int64_t ldc) {
    typedef float Vec __attribute__((ext_vector_type(V)));
    const int64_t col = (static_cast<int64_t>(blockIdx.x) * kFinishBlock + threadIdx.x) * V;
    if (col >= n) return;
    const int64_t mn = m * n;
    for (int64_t r = blockIdx.y; r < m; r += gridDim.y) {
        const float* at = part + r * n + col;
        auto slice = [&](int s) { return *reinterpret_cast<const Vec*>(at + s * mn); };
        Vec acc = slice(0);
        int s = 1;
        for (; s + 4 <= slices; s += 4) {
            const Vec v0 = slice(s), v1 = slice(s + 1), v2 = slice(s + 2), v3 = slice(s + 3);
            acc += v0;
            acc += v1;
            acc += v2;
            acc += v3;
        }
        for (; s < slices; ++s) acc += slice(s);
        typename Elem<T>::storage out[V];
#pragma unroll
        for (int j = 0; j < V; ++j) {
            float v;
            if (beta == 0.0f) {
                v = alpha * acc[j];
            } else if (cin_rs == 0) {
                v = fmaf(alpha, acc[j], beta * Elem<T>::load(cin[(col + j) * cin_cs]));
            } else {
                v = fmaf(beta, Elem<T>::load(cin[r * cin_rs + (col + j) * cin_cs]), alpha * acc[j]);
            }
            out[j] = Elem<T>::store(v);
        }
        if constexpr (V == 4 && sizeof(out) == 16) {
            *reinterpret_cast<uint4*>(c + r * ldc + col) = __builtin_bit_cast(uint4, out);
        } else if constexpr (V == 4) {
            *reinterpret_cast<uint2*>(c + r * ldc + col) = __builtin_bit_cast(uint2, out);
        } else {
            c[r * ldc + col] = out[0];
        }
    }
}

template <typename T>
void launch_finish(const float* part, int slices, const GemmArgs& p, hipStream_t stream) {
    using S = typename Elem<T>::storage;
    const bool vec = p.n % 4 == 0 && p.ldc % 4 == 0 &&
                     (reinterpret_cast<uintptr_t>(p.c) & (4 * sizeof(S) - 1)) == 0;
    const int64_t cols = vec ? p.n / 4 : p.n;
    const dim3 grid(static_cast<unsigned>((cols + kFinishBlock - 1) / kFinishBlock),
                    static_cast<unsigned>(std::min<int64_t>(p.m, 65535)));
    auto* kernel = vec ? splitk_finish_kernel<T, 4> : splitk_finish_kernel<T, 1>;
    kernel<<<grid, kFinishBlock, 0, stream>>>(part, slices, p.m, p.n, p.alpha, p.beta,
                                              static_cast<const S*>(p.cin), p.cin_rs, p.cin_cs,
                                              static_cast<S*>(p.c), p.ldc);
    TP_AMD_HIP_CHECK(hipGetLastError());
}

// Splits K: the slices, K tiles of ks = a multiple of BK (the last one
// shorter), ride on the tile kernel's batch index and write float32 partial
// products into `part`, [slices][M][N]; splitk_finish_kernel then adds
// them in slice order, so the result does not depend on timing.
template <typename T, int BM, int BN, int STAGES, int BLOCKS>
void launch_split(const GemmArgs& p, int64_t slices, int64_t ks, void* part, hipStream_t stream) {
    const int64_t mn = p.m * p.n;
    GemmArgs q = p;
    q.batch = slices;
    q.k = ks;
    q.k_total = p.k;
    q.stride_a = p.trans_a ? ks * p.lda : ks;  // slice s starts at k = s ks
    q.stride_b = p.trans_b ? ks : ks * p.ldb;
    q.alpha = 1.0f;
    q.beta = 0.0f;
    q.cin = nullptr;
    q.c = part;
    q.ldc = p.n;
    q.stride_c = mn;
    launch_config<T, BM, BN, STAGES, BLOCKS, true>(q, stream);
    launch_finish<T>(static_cast<const float*>(part), static_cast<int>(slices), p, stream);
}

// The tile kernel's shapes (LDS stages, blocks a CU) and what each is for.
enum class Tile {
    k128,      // 128 x 128, 2 stages, 2 blocks a CU: several rounds of tiles
    k128Deep,  // 128 x 128, 3 stages, 1 block a CU: one round (16-bit)
    k64x128,   // 64 x 128: 16-bit 3 stages, 2 blocks
    k64x128Many,  // 64 x 128: 16-bit 2 stages, 3 blocks
    k64,       // 64 x 64: 16-bit 3 stages, 3 blocks; float32 2 stages, 4 blocks
    k32x128,   // 32 x 128, 4 stages, 2 blocks (float32)
};

struct TilePlan {
    Tile tile;
    int64_t slices = 1, ks = 0;
};

int64_t tiles_of(const GemmArgs& p, int64_t bm, int64_t bn) {
    return (p.m + bm - 1) / bm * ((p.n + bn - 1) / bn) * p.batch;
}

// At most `most` slices of at least min_k.
TilePlan split_k(Tile tile, const GemmArgs& p, int64_t most, int64_t min_k, int64_t bk) {
    TilePlan plan{tile};
    const int64_t s = std::min(most, p.k / min_k);
    if (p.batch != 1 || s < 2) return plan;
    plan.ks = ((p.k + s - 1) / s + bk - 1) / bk * bk;
    plan.slices = (p.k + plan.ks - 1) / plan.ks;
    return plan;
}

// A product of few rows or columns (a small batch through a Linear) is bound
// by reading the other operand: enough blocks with enough loads in flight,
// whatever their tiles waste on padding rows.
//   * 16-bit, up to 64: 64 x 64 tiles, split into slices of at least 1024
//     for up to three blocks a CU and up to eight slices, or one a CU.
//     Measured with W rotated past the Infinity Cache (bf16, x W^T, us, the
//     thin kernel in brackets): 8 x 11008 x 4096 19.3 (23.9), 8 x 4096 x
//     11008 20.5 (21.6), 48 x 11008 x 4096 23.0 (40.7), 48 x 2048 x 5504
//     15.1 (22.1); x W 8 x 11008 x 4096 19.6 (26.3).  Unsplit with two
//     rounds of tiles (a vocabulary) 64 x 128 tiles halve the blocks.
//   * float32, 17 to 32 rows: 32 x 128 tiles (a taller tile's padding rows
//     cost MFMA time there), one block a CU in slices of at least 512, or 128
//     for the first 16 (the finish adds each in turn): 20 x 11008 x 4096 47.0
//     (54.6), 20 x 4096 x 11008 45.3 (56.7), 24 x 4096 x
//     1024 11.5 (13.9).  As many columns take plan_tiles' slices of 64 x 64
//     tiles up to 48 MiB of the wide operand (1024 x 24 x 4736 14.8, thin 20
//     to 27; 4096 x 24 x 4096 27.5, thin 26 to 31; 14848 x 24 x 15040 264, thin
//     191 to 252).
//   * float32, 33 to 64: 64 x 64 tiles, up to three blocks a CU: 48 x 4096 x
//     11008 58.5 (102), 48 x 4096 x 4096 27.3 (40.2); a K too short for
//     that, by plan_tiles' model: 48 x 4096 x 1024 13.0 (21.0), 33 x 12352 x
//     512 13.1 (29.1).
template <typename T>
TilePlan plan_small_batch(const GemmArgs& p, int64_t cus) {
    constexpr int64_t BK = Mfma<T>::BK;
    const int64_t t64 = tiles_of(p, 64, 64);
    if constexpr (std::is_same<T, float>::value) {
        if (p.m <= 32 && p.n > 64) {
            const int64_t most = std::max(p.k / 512, p.k < 512 ? 0 : std::min<int64_t>(16, p.k / 128));
            return split_k(Tile::k32x128, p, std::min(cus / tiles_of(p, 32, 128), most), 128, BK);
        }
        return split_k(Tile::k64, p, 3 * cus / t64, 1024, BK);
    } else {
        if (t64 >= 2 * cus && p.m <= 64) return TilePlan{Tile::k64x128};
        return split_k(Tile::k64, p, std::min(3 * cus / t64, std::max<int64_t>(8, cus / t64)), 1024, BK);
    }
}

template <typename T>
TilePlan plan_tiles(const GemmArgs& p, int64_t cus) {
    constexpr int64_t BK = Mfma<T>::BK;
    const int64_t thin = std::min(p.m, p.n);
    const int64_t t128 = tiles_of(p, 128, 128), t64 = tiles_of(p, 64, 64);
    // Rows this far apart have the 64 x 64 tiles, and 16-bit slices the 128 x
    // 128 ones (launch_config).
    if (rows_far<T>(p)) {
        if (sizeof(typename Elem<T>::storage) == 2 && thin > 64 && t128 <= cus / 4) {
            const TilePlan plan = split_k(Tile::k128Deep, p, cus / t128, 1024, BK);
            if (plan.slices > 1) return plan;
        }
        return split_k(Tile::k64, p, 3 * cus / t64, 1024, BK);
    }
    if constexpr (std::is_same<T, float>::value) {
        if (p.batch == 1 && thin > 16 && thin <= 64) {
            const TilePlan plan = plan_small_batch<T>(p, cus);
            if (plan.slices > 1 && (plan.tile == Tile::k32x128 || (thin > 32 && 2 * t64 * plan.slices >= cus))) return plan;
        }
        // MFMAs of 64 cycles leave LDS and L2 idle, so a CU is busy as long
        // as it has a tile, one of 64 x 64 at 93 % of the larger ones' rate
        // (8192 x 4096 x 4096 2010 against 1886 us), and the time is the
        // rounds of tiles times their K: kTileUs a k of a 64 x 64 tile, by
        // the instruction's rate.  Slices of K even out the last round for
        // the price of the finish: 2.2 us, a launch that a program bound by
        // its host calls pays too, and a pass over the partials.
        // 2048 x 3000 x 1000 125 us on 128 x 128 tiles, 102 on 64 x 64; 256 x
        // 4096 x 1024 66 and 22; 700 x 900 x 5000 89 whole, 63 in three
        // slices; 1500 x 1500 x 4000 184 and 157; 256 x 1024 x 4096 70, 26 in
        // four; 33 x 192 x 512 11.5, 7.8 in eight; 256^3 7.5, 8.7 in two.
        constexpr double kTileUs = 0.0137, kFinishUs = 4.0, kPartialsPerUs = 1.25e6;
        const double rounds128 = double((t128 + cus - 1) / cus);
        TilePlan best{Tile::k128};
        double least = rounds128 * double(p.k) * kTileUs * 4 * 0.93;
        // Few tiles and a long K take more slices, up to two blocks a CU; each
        // past 16 adds its loads to the finish's chain.  From K = 16384 on the
        // operands stream from memory, and one block a CU waits for its loads
        // (a k takes twice as long): 128 x 128 x 65536 57 us in 16 slices,
        // 36 in 128; x 2^20 2047 and 418; 256 x 256 x 65536 114 in 16, 78 in 32;
        // 512 x 512 x 16384 110 in 4, 80 in 8.
        constexpr double kSliceUs = 0.08;
        const int64_t min_slice = p.k >= 512 ? 64 : 192;
        const double wait = p.k >= 16384 ? 1.9 : 1.0;
        // 1 to 16, then 24, 32, 48, 64, ...
        auto next = [](int64_t s) { return s + (s < 16 ? 1 : (s & (s - 1)) == 0 ? s / 2 : s / 3); };
        for (int64_t slices = 1; slices <= 16 || t64 * slices <= 2 * cus; slices = next(slices)) {
            if (slices > 1 && (p.batch != 1 || p.k < slices * min_slice)) break;
            const TilePlan plan = split_k(Tile::k64, p, slices, min_slice, BK);
            const int64_t blocks = t64 * plan.slices;
            double us = double((blocks + cus - 1) / cus) * double(plan.slices == 1 ? p.k : plan.ks) * kTileUs;
            if (blocks <= cus) us *= wait;
            if (plan.slices > 16) us += kSliceUs * double(plan.slices - 16);
            if (plan.slices > 1) us += kFinishUs + double(p.m) * double(p.n) * double(2 * plan.slices + 1) / kPartialsPerUs;
            if (us < least) {
                least = us;
                best = plan;
            }
        }
        return best;
    } else {
        if (thin <= 64) return plan_small_batch<T>(p, cus);
        // A very long K on few tiles is read from memory: 128 x 128 tiles read
        // each operand half as often as 64 x 64 ones, one block a CU.  bf16 512
        // x 1024 x 15000 35.6 us against 46.0, 256 x 256 x 65536 34 against 37,
        // x 2^20 447 against 628; 128 x 128 x 2^20 158 against 208; 512 x 512 x
        // 16384 26 against 28; below, 64 x 64 tiles are level or faster (512 x
        // 1024 x 12288 28.9 against 30.2, 256 x 256 x 16384 15 against 19).
        // With so many 64 x 64 tiles that their slices are two, leaving some
        // CUs two blocks and others one, from K = 4096 on: 200 x 3000 x 3000
        // 17.8 against 18.2, x 4104 19.3 against 22.5, x 11000 33.4 against
        // 51.9; 1124 x 624 x 8192 28.4 against 31.3; 1500 x 400 (168 tiles) x
        // 8192 28.5 against 25.4, x 9000 34.1 against 35.7.  Not where 128 x
        // 128 tiles are mostly padding (129 x 144 x 84864 32.4 against 29.1).
        if (t128 <= cus / 4) {
            if (p.k > 12288 && p.k / (cus / t128) >= 1024 && 2 * t64 >= 5 * t128) {
                return split_k(Tile::k128Deep, p, cus / t128, 1024, BK);
            }
            if (t64 > cus * 5 / 8 && p.k >= (t64 > cus * 11 / 16 ? 4096 : 9000)) {
                return split_k(Tile::k128Deep, p, cus / t128, 768, BK);
            }
        }
        // One round of 128 x 128 tiles by splitting K: when K is long, or when
        // one row of tiles reads a wide operand once.  1500 x 700 x 5000
        // 30.8 us in three slices, 40.6 on 64 x 128 tiles whole; 1024 x 1536
        // x 8192 41.8 against 44.5; 128 x 11008 x 4096 33.6 against 37.3 on
        // 64 x 64 tiles; 1280 x 1280 x 3000 28.0 in two, 26.5 whole.  Where
        // whole slices leave a fifth of the CUs idle and K is long, two blocks a
        // CU come closer: 1200 x 1100 x 11000 (90 tiles) 69.6 and 63.0, 1536 x
        // 1024 x 15000 (96) 88 and 82; x 6000 40.6 and 42.
        if (t128 >= cus / 4 && t128 <= cus / 2 && (p.k > 4096 || (thin <= 128 && t64 > cus && p.k >= 2048))) {
            const bool idle = 5 * t128 * (cus / t128) < 4 * cus && p.k > 8192;
            const TilePlan plan = idle ? split_k(Tile::k128, p, 2 * cus / t128, 1024, BK)
                                       : split_k(Tile::k128Deep, p, cus / t128, 1024, BK);
            if (plan.slices > 1) return plan;
        }
        // Rounds of 128 x 128 tiles, two a CU.  A short K with at most half
        // of the last round used takes twice the tiles, three a CU (3001 x
        // 3072 x 768: 576 tiles 28.1 us, 1152 half tiles 25.5).
        if (t128 > cus) {
            const int64_t last = t128 % (2 * cus);
            if (p.k <= 1024 && t128 > 2 * cus && last != 0 && last <= cus) return TilePlan{Tile::k64x128Many};
            return TilePlan{Tile::k128};
        }
        // At most one round: one block a CU with a third stage (2048^3 22.7
        // against 26.1 us on two, 3001 x 768 x 3072 28.1 against 39.6), the
        // tile as large as still gives half the CUs one: 1777 x 1008 x 3336
        // 26.0 us on 64 x 128 against 35.1 on 128 x 128, 1024 x 1024 x 4096
        // 22.7 us on 64 x 64 against 25.5 on 64 x 128.
        if (t128 > cus / 2) {
            // A long K fills the CUs better in slices, two blocks a CU: 777 x
            // 3000 x 11000 79.6 us in three against 96.8 whole, 2000 x 1280
            // x 6000 48.3 against 53.3; with K = 3000 they are level.
            if (p.batch == 1 && p.k >= 4096 && t128 <= cus * 4 / 5) return split_k(Tile::k128, p, 2 * cus / t128, 1024, BK);
            return TilePlan{Tile::k128Deep};
        }
        if (tiles_of(p, 64, 128) > cus / 2) return TilePlan{Tile::k64x128};
        if (t64 >= cus || p.k <= 2048) return TilePlan{Tile::k64};
        return split_k(Tile::k64, p, 2 * cus / t64, 1024, BK);
    }
}

template <typename T>
void launch_mfma(const GemmArgs& p, hipStream_t stream) {
    int device = 0;
    TP_AMD_HIP_CHECK(hipGetDevice(&device));
    const int64_t cus = cu_count(device);
    constexpr bool k16 = sizeof(typename Elem<T>::storage) == 2;
    if constexpr (k16) {
        if (smallk::eligible<T>(p, cu_count(device))) {
            smallk::launch<T>(p, stream);
            return;
        }
        if (big::eligible<T>(p, cu_count(device))) {
            big::launch<T>(p, stream);
            return;
        }
    }
    TilePlan plan = plan_tiles<T>(p, cus);
    Workspace part;
    if (plan.slices > 1) {
        part = Workspace::if_room(static_cast<size_t>(plan.slices * p.m * p.n) * sizeof(float), device);
        if (part.get() == nullptr) {  // whole K needs no memory
            if (p.k >> 32) return launch_gemm_general<T>(p, stream);  // past a panel's 32-bit K
            plan = TilePlan{Tile::k64};
        }
    }
    if (plan.slices > 1) {
        if constexpr (k16) {
            if (plan.tile == Tile::k128) launch_split<T, 128, 128, 2, 2>(p, plan.slices, plan.ks, part.get(), stream);
            else if (plan.tile == Tile::k128Deep) launch_split<T, 128, 128, 3, 1>(p, plan.slices, plan.ks, part.get(), stream);
            else launch_split<T, 64, 64, 3, 3>(p, plan.slices, plan.ks, part.get(), stream);
        } else {
            if (plan.tile == Tile::k32x128) launch_split<T, 32, 128, 4, 2>(p, plan.slices, plan.ks, part.get(), stream);
            else launch_split<T, 64, 64, 2, 4>(p, plan.slices, plan.ks, part.get(), stream);
        }
        return;
    }
    if constexpr (k16) {
        switch (plan.tile) {
            case Tile::k128Deep: launch_config<T, 128, 128, 3, 1>(p, stream); return;
            case Tile::k64x128: launch_config<T, 64, 128, 3, 2>(p, stream); return;
            case Tile::k64x128Many: launch_config<T, 64, 128, 2, 3>(p, stream); return;
            case Tile::k64: launch_config<T, 64, 64, 3, 3>(p, stream); return;
            default: launch_config<T, 128, 128, 2, 2>(p, stream);
        }
    } else {
        if (plan.tile == Tile::k64) launch_config<T, 64, 64, 2, 4>(p, stream);
        else launch_config<T, 128, 128, 2, 2>(p, stream);
    }
}

template <typename T>
struct DtypeOf;
template <>
struct DtypeOf<float> { static constexpr int value = TP_AMD_FLOAT32; };
template <>
struct DtypeOf<bf16_t> { static constexpr int value = TP_AMD_BFLOAT16; };
template <>
struct DtypeOf<f16_t> { static constexpr int value = TP_AMD_FLOAT16; };

// dst [batch][rows_out][per_row packets] = src's rows x cols of each batch
// entry (rows ld apart, entries `stride`), zeros around them.  Bound by
// memory: a thread has four 16-byte packets in flight, read at any element.
constexpr int kRepackBlock = 256, kRepackUnroll = 4;

template <typename S>
__global__ __launch_bounds__(kRepackBlock) void repack_kernel(S* __restrict__ dst, const S* __restrict__ src,
                                                              int64_t total, int64_t rows_out, int64_t per_row,
                                                              FastDiv by_rows, FastDiv by_packets, int64_t rows,
                                                              int64_t cols, int64_t ld, int64_t stride) {
    constexpr int N = 16 / sizeof(S);
    const bool small = total < (int64_t{1} << 31);
    const int64_t first = static_cast<int64_t>(blockIdx.x) * (kRepackBlock * kRepackUnroll) + threadIdx.x;
    uint4 v[kRepackUnroll];
#pragma unroll
    for (int u = 0; u < kRepackUnroll; ++u) {
        const int64_t i = first + u * kRepackBlock;
        if (i >= total) break;
        const int64_t row = small ? fastdiv(static_cast<uint32_t>(i), by_packets) : i / per_row;
        const int64_t b = small ? fastdiv(static_cast<uint32_t>(row), by_rows) : row / rows_out;
        const int64_t r = row - b * rows_out, c = (i - row * per_row) * N;
        const S* from = src + b * stride + r * ld + c;
        if (r < rows && c + N <= cols) {
            v[u] = load_raw_any(from);
        } else {
            S t[N];
#pragma unroll
            for (int e = 0; e < N; ++e) t[e] = r < rows && c + e < cols ? from[e] : S{};
            __builtin_memcpy(&v[u], t, 16);
        }
    }
#pragma unroll
    for (int u = 0; u < kRepackUnroll; ++u) {
        const int64_t i = first + u * kRepackBlock;
        if (i < total) reinterpret_cast<uint4*>(dst)[i] = v[u];
    }
}

// An operand's copy: its layout kept, rows whole 128-byte lines, and K (the
// columns when K-major, the rows otherwise) zero-padded to kp.
template <typename T>
struct Repack {
    static constexpr int64_t E = sizeof(typename Elem<T>::storage), kLine = 128 / E;
    int64_t rows, cols, ld, stride, rows_out, ld_out, batch;

    Repack(int64_t ld_, int64_t stride_, bool kmajor, int64_t batch_, int64_t mn, int64_t k, int64_t kp)
        : rows(kmajor ? mn : k), cols(kmajor ? k : mn), ld(ld_), stride(stride_), rows_out(kmajor ? mn : kp),
          ld_out(((kmajor ? kp : mn) + kLine - 1) / kLine * kLine), batch(stride_ == 0 ? 1 : batch_) {}
    int64_t elems() const { return batch * rows_out * ld_out; }
    int64_t out_stride() const { return stride == 0 ? 0 : rows_out * ld_out; }  // a broadcast operand is copied once
    void launch(const void* src, void* dst, hipStream_t stream) const {
        using S = typename Elem<T>::storage;
        const int64_t per_row = ld_out * E / 16, total = batch * rows_out * per_row;
        const bool small = total < (int64_t{1} << 31);
        const FastDiv by_rows = make_fastdiv(small ? static_cast<uint32_t>(rows_out) : 1);
        const FastDiv by_packets = make_fastdiv(small ? static_cast<uint32_t>(per_row) : 1);
        constexpr int64_t kBlock = kRepackBlock * kRepackUnroll;
        repack_kernel<S><<<static_cast<unsigned>((total + kBlock - 1) / kBlock), kRepackBlock, 0, stream>>>(
            static_cast<S*>(dst), static_cast<const S*>(src), total, rows_out, per_row, by_rows, by_packets, rows, cols,
            ld, stride);
        TP_AMD_HIP_CHECK(hipGetLastError());
    }
};

template <typename T>
bool packets_aligned(const void* x, int64_t ld, int64_t stride) {
    constexpr int V = Mfma<T>::V;
    return aligned16(x) && ld % V == 0 && stride % V == 0;
}

// A product on copies of its operands that are not aligned packets: which
// ones, where in the workspace, and the product on them.  A K that is no whole
// number of packets is padded in both copies.
template <typename T>
struct Repacked {
    int64_t kp;
    bool fix_a, fix_b;
    Repack<T> a, b;
    size_t off_b, bytes;

    explicit Repacked(const GemmArgs& p)
        : kp(p.k % Mfma<T>::V != 0 ? (p.k + Mfma<T>::BK - 1) / Mfma<T>::BK * Mfma<T>::BK : p.k),
          fix_a(kp != p.k || !packets_aligned<T>(p.a, p.lda, p.stride_a)),
          fix_b(kp != p.k || !packets_aligned<T>(p.b, p.ldb, p.stride_b)),
          a(p.lda, p.stride_a, !p.trans_a, p.batch, p.m, p.k, kp),
          b(p.ldb, p.stride_b, p.trans_b, p.batch, p.n, p.k, kp),
          off_b(fix_a ? (a.elems() * a.E + 255) / 256 * 256 : 0),
          bytes(off_b + (fix_b ? b.elems() * b.E : 0)) {}

    GemmArgs product(const GemmArgs& p, void* ws) const {
        GemmArgs q = p;
        q.k = kp;
        if (fix_a) {
            q.a = ws;
            q.lda = a.ld_out;
            q.stride_a = a.out_stride();
        }
        if (fix_b) {
            q.b = static_cast<char*>(ws) + off_b;
            q.ldb = b.ld_out;
            q.stride_b = b.out_stride();
        }
        return q;
    }
};

// Whether a product gains by copies of its operands that are not whole
// aligned packets.
//   * 16-bit: read in place, such an operand costs a product that fills the
//     chip time per multiply-add (each load touches twice the cache lines):
//     about 0.70e-15 s for a K-major and 0.40e-15 s for an M/N-major one (bf16
//     8191 x 11007 x 4095 in place 1172 us NT, 1081 NN, 1006 TN, on copies
//     760, 794 and 815).  The copies cost one pass at about 5 TB/s and a launch
//     each: 2047^3 takes 32 us in place and would take 40.
//   * float32 is bound by its MFMAs and loses nothing in place, but a batch is
//     not split over K: a thin product of a long K walks it on few CUs, 18.5
//     ns a k, where the thin kernel reads its copies faster.  32 x (8 x 15 x
//     2121) 39.1 us in place, 22.0 on copies; 2 x (256 x 4 x 4001) 70.8 and
//     25.7; 32 x (256 x 4 x 2121) 43.0 and 46.4; 128 x (8 x 15 x 1023) 20.7
//     and 21.0.
template <typename T>
bool repack_pays(const GemmArgs& p) {
    constexpr int64_t E = sizeof(typename Elem<T>::storage);
    if constexpr (E == 4) {
        if (p.batch == 1 || std::min(p.m, p.n) > 64) return false;
        const Repacked<T> copies(p);
        if (copies.bytes == 0) return false;
        int device = 0;
        TP_AMD_HIP_CHECK(hipGetDevice(&device));
        const int64_t cus = cu_count(device);
        const double read = 4.0 * static_cast<double>((p.stride_a == 0 ? 1 : p.batch) * p.m + (p.stride_b == 0 ? 1 : p.batch) * p.n) *
                            static_cast<double>(p.k);
        const double in_place = static_cast<double>((tiles_of(p, 64, 64) + cus - 1) / cus) * static_cast<double>(p.k) * 18.5e-9;
        // two copies, the thin kernel's launch, the bytes at 5 and 4 TB/s
        if (in_place <= 20e-6 + 2.0 * read / 5e12 + read / 4e12) return false;
        void* any_aligned = reinterpret_cast<void*>(uintptr_t{256});
        return launch_gemm_thin(DtypeOf<T>::value, copies.product(p, any_aligned), nullptr, true);
    } else {
        const bool pad = p.k % Mfma<T>::V != 0;
        double in_place = 0.0, copies = 0.0;
        auto add = [&](const void* x, int64_t ld, int64_t stride, bool kmajor, int64_t mn) {
            const bool odd = !packets_aligned<T>(x, ld, stride);
            if (odd) in_place += kmajor ? 0.70e-15 : 0.40e-15;
            if (odd || pad) {
                copies += 5e-6 + 2.0 * E * static_cast<double>(stride == 0 ? 1 : p.batch) * static_cast<double>(mn) *
                                     static_cast<double>(p.k) / 5e12;
            }
        };
        add(p.a, p.lda, p.stride_a, !p.trans_a, p.m);
        add(p.b, p.ldb, p.stride_b, p.trans_b, p.n);
        return in_place * static_cast<double>(p.batch) * static_cast<double>(p.m) * static_cast<double>(p.n) *
                   static_cast<double>(p.k) > copies;
    }
}

// A product on copies of its operands, where that pays.
template <typename T>
void launch_repacked(const GemmArgs& p, hipStream_t stream) {
    int device = 0;
    TP_AMD_HIP_CHECK(hipGetDevice(&device));
    const Repacked<T> copies(p);
    const Workspace ws = Workspace::if_room(copies.bytes, device);
    if (ws.get() == nullptr) {
        launch_mfma<T>(p, stream);  // in place
        return;
    }
    const GemmArgs q = copies.product(p, ws.get());
    if (copies.fix_a) copies.a.launch(p.a, const_cast<void*>(q.a), stream);
    if (copies.fix_b) copies.b.launch(p.b, const_cast<void*>(q.b), stream);
    // A thin product reads its copies through the thin kernel.
    if (!launch_gemm_thin(DtypeOf<T>::value, q, stream)) launch_mfma<T>(q, stream);
}

template <typename T>
void launch_typed(const GemmArgs& p, hipStream_t stream) {
    if (p.k <= 0 || !tiles_fit(p)) launch_gemm_general<T>(p, stream);
    else if (repack_pays<T>(p)) launch_repacked<T>(p, stream);
    else launch_mfma<T>(p, stream);
}

}  // namespace

bool tiles_take_thin(int dtype, const GemmArgs& p, int device) {
    const int64_t cus = cu_count(device), thin = std::min(p.m, p.n);
    const int64_t t64 = tiles_of(p, 64, 64);
    if (p.batch > 1) return thin > 32 && t64 >= cus;
    if (dtype == TP_AMD_FLOAT32) {
        if (thin > 32) return true;
        if (thin <= 16) return false;
        if (p.m <= 32 && p.n > 64) return plan_small_batch<float>(p, cus).slices > 1;
        return std::max(p.m, p.n) * p.k * 4 < (int64_t{48} << 20);
    }
    const TilePlan plan = plan_small_batch<bf16_t>(p, cus);
    const int64_t blocks = (plan.tile == Tile::k64 ? t64 : tiles_of(p, 64, 128)) * plan.slices;
    if (thin > 32) return blocks >= cus / 4;
    if (thin > 16) return blocks >= cus / 2;
    // As few columns write C column by column: 18368 x 8 x 2176 bf16 24.7 us
    // on tiles, 21.4 on the thin kernel; 4416 x 16 x 7296 17.5 and 20.4.
    return plan.slices > 1 && 2 * blocks >= 3 * cus && (p.m <= 64 || t64 < cus / 2);
}

void launch_gemm(int dtype, const GemmArgs& p, hipStream_t stream) {
    if (launch_gemm_thin(dtype, p, stream)) return;
    switch (dtype) {
        case TP_AMD_FLOAT32: launch_typed<float>(p, stream); break;
        case TP_AMD_BFLOAT16: launch_typed<bf16_t>(p, stream); break;
        case TP_AMD_FLOAT16: launch_typed<f16_t>(p, stream); break;
        default:
            TP_AMD_CHECK(false, "GEMM takes float32, float16 or bfloat16, got ", dtype_name(dtype));
    }
}

}  // namespace tp_amd
