// CSR x dense kernels for gfx950 (wave64, 256 CUs in 8 XCDs).
//
//   csr_rows_in_order  role of spmm_baseline and spmm_memopt/_v2
//                      (spmm_baseline.cu:11-25, spmm_memopt.cu:11-38)
//   csr_rowblock       role of spmm_tiled* (spmm_tiled_v3.cu:21-104), the engine
//   csr_rowblock_wide  the engine on wide B and balanced partitions
//   csr_row_groups     the engine's role on narrow B and short rows
//
// All accumulate in fp32 with fused multiply-adds.  C is fully written
// (rows without nonzeros get zeros), so callers never clear it.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "engine.h"
#include "spmm/utils.h"

typedef float spmm_f32x2 __attribute__((ext_vector_type(2)));
typedef float spmm_f32x4 __attribute__((ext_vector_type(4)));

// Structured buffer loads (LLVM's AMDGPU intrinsics; index = record, offset =
// byte offset inside the record).  The intrinsic names are fixed by LLVM.
__device__ spmm_f32x4 sbuf_load_x4(__amdgpu_buffer_rsrc_t rsrc, int index, int offset,
                                   int soffset, int aux)
    __asm("llvm.amdgcn.struct.ptr.buffer.load.v4f32");
__device__ spmm_f32x2 sbuf_load_x2(__amdgpu_buffer_rsrc_t rsrc, int index, int offset,
                                   int soffset, int aux)
    __asm("llvm.amdgcn.struct.ptr.buffer.load.v2f32");
__device__ float sbuf_load_x1(__amdgpu_buffer_rsrc_t rsrc, int index, int offset, int soffset,
                              int aux) __asm("llvm.amdgcn.struct.ptr.buffer.load.f32");

namespace spmm {
namespace engine {

namespace {

constexpr int kWave = 64;

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// T: VEC floats in registers.  Mem: the same at any float address; rows of an N
// that is no multiple of VEC start there, and a 16-byte access needs no more.
template <int VEC> struct Vec;
template <> struct Vec<1> { using T = float; using Mem = float; };
template <> struct Vec<2> {
    using T = f32x2;
    typedef f32x2 Mem __attribute__((aligned(4)));
};
template <> struct Vec<4> {
    using T = f32x4;
    typedef f32x4 Mem __attribute__((aligned(4)));
};

template <int VEC>
__device__ __forceinline__ typename Vec<VEC>::T vzero() {
    return typename Vec<VEC>::T(0.0f);
}

// ---------------------------------------------------------------------------
// The engine (role: spmm_tiled / _v2 / _v3 / _v4).
//
// Partition.  Workgroup g owns rows [r_begin, r_end): either g*R .. g*R+R
// (implicit, R chosen from the average row length) or bounds[g] .. bounds[g+1]
// (an explicit nnz-balanced partition).  Merge-path mode (split_rows) cuts at
// the workgroup level too: workgroup g takes nonzeros [nnz*g/P, nnz*(g+1)/P)
// whatever rows they belong to; a row that began in an earlier workgroup is
// summed into carry[g] instead of C, and csr_split_fixup adds the carries to C
// in part order afterwards.
//
// Lane groups.  A wave is split into G groups of L lanes, any L that covers the
// columns of a pass with VEC-float (up to 16-byte) loads: 20 lanes and three
// groups for N = 77, eight lanes and eight groups for a slice of 32 columns.
// The nonzeros of the workgroup are cut into equal contiguous ranges, one per
// group, so a long row is shared by several groups and a group may take many
// short rows.  One load instruction fetches G different B row segments, and no
// group waits for another's row end: at one of its own a group stores (or puts
// aside) its sum under its lanes' mask and goes on.
//
// Per wave.  The wave copies (col, value) pairs of its groups' ranges into its
// LDS window (kWCap entries, one run per group, all loads issued at once);
// every lane then reads the entry of its group with a broadcast ds_read_b64 and
// gathers its B segment with a bounds-checked buffer load (one record per B
// row, so the row index is the load's index operand and needs no address
// arithmetic).  Each register of the U rows in flight is refilled as soon as it
// is used, and the entries are read from LDS one step ahead.  Every fourth entry
// of a range goes to the same of four partial sums (kChains), added at a row's
// end: the rounding error grows with the longest chain, and one chain per range
// is up to twice as far from 64 bits as the interleaved groups of
// csr_rowblock_wide (merge-path parts of 30000^2, 120 per row, N = 32: 1.8e-7 of the
// norm, with four 1.0e-7; 65536^2, 32 per row, N = 256 8.2e-8 and 6.5e-8).  They cost
// a row end 24 instructions (16384^2, 8 per row, N = 128 9.4 -> 10.4 us; 65536^2, 32
// per row, N = 256 210 -> 208).  At a row's end:
//   - a row that lies wholly inside the group's range is stored to C;
//   - the first row of a range that started in an earlier group goes to an LDS
//     slot of the group;
//   - the last row of a range that continues in a later group stays in the
//     registers of its owner, which after a barrier adds the LDS slots of the
//     following groups in order and stores it.
// The sum order is fixed by the partition and the launch shape, so results
// are deterministic run to run.
//
// What bounds it: the lines a CU has in flight towards L2 (20 TB/s of gathered
// rows at best where B fits the L2s), and past the L2s their misses (8 - 10
// TB/s).  Measured on MI355X against the form before it, in which the groups of
// a wave took alternate entries of one range, in whole steps of U * G entries,
// and reduced at every row end (csr_rowblock_wide is that form): 20011 x 17001,
// 40 per row, N = 77 30.8 -> 22.6 us; 65536^2, 32 per row, N = 256 243 -> 209 us
// with eight slices (298 in the old form, whose steps of 32 entries each held a
// row end); power-law 65536^2, N = 32 over B-row halves 67 -> 35 us; 8192^2
// power-law, 74 per row, N = 256 63 -> 40 us.
//
// Rows of the workgroup without nonzeros are zero-filled up front.  Row
// pointers are staged in LDS in windows of kRpCap rows.
// ---------------------------------------------------------------------------
// One sparse matrix, its B, its C and (merge-path) its partition.
struct RowblockPart {
    const int*   row_ptr;
    const int*   col_idx;
    const float* vals;
    const float* B;
    float*       C;
    // Merge-path partition (nullable split_rows): part g = nonzeros
    // [nnz*g/nblocks, nnz*(g+1)/nblocks); split_rows[g] is the row holding the
    // first of them (split_rows[0] = 0, split_rows[nblocks] = M); carry is a
    // nblocks x N workspace for the partial of a part's first row when that
    // row began in an earlier part.
    const int*   split_rows = nullptr;
    float*       carry = nullptr;
    long long    nnz = 0;
    int          K = 0;        // rows of B (records of the B buffer)
    int          nblocks = 0;  // row blocks (workgroups of one column slice)
};

struct RowblockArgs {
    RowblockPart part;
    const int*   bounds = nullptr;    // nullable: rows of each row block
    int          M = 0;
    int          N = 0;
    int          rows_per_block = 0;
    int          slices = 1;          // column slices: 1, 2, 4 or 8
    int          slice_cols = 0;      // columns per slice (a multiple of VEC)
    int          group_lanes = 64;    // lanes per group
    int          groups = 1;          // groups per wave: at most 64 / group_lanes
    int          window_log = 0;      // log2 of the entries a group stages at a time
    int          lanes_inv = 0;       // lane / group_lanes == lane * lanes_inv >> 16
    unsigned     groups_inv = 0;      // 2^32 / groups, rounded up
    // B-row halves only (merge-path only): workgroups on XCDs 4-7 take this
    // part -- the entries of A whose columns lie in B's upper rows, with
    // rebased columns, those B rows, their own output and merge-path table --
    // and XCDs 0-3 the first, so each XCD's L2 holds half of B at full width.
    // Last, so that the other launches read two cache lines less.
    RowblockPart upper{};
};

// Has every argument loaded before the first branch on one of them.  Left to
// itself the compiler loads each group of arguments where it is first needed,
// and every group costs a launch one more wait on the scalar cache (MI355X,
// over 60 launches of 4 to 100 us 0.1 - 0.4 us; 2048^2, 40 per row, N = 256: 6.84
// against 6.63 us).  The eight scalar registers that this spills cost less.
__device__ __forceinline__ void load_args(const RowblockArgs& a, const RowblockPart& m) {
    asm volatile("" ::"s"(m.row_ptr), "s"(m.col_idx), "s"(m.vals), "s"(m.B), "s"(m.C),
                 "s"(m.split_rows), "s"(m.carry), "s"(m.nnz), "s"(m.K), "s"(m.nblocks),
                 "s"(a.bounds), "s"(a.M), "s"(a.N), "s"(a.rows_per_block), "s"(a.slices),
                 "s"(a.slice_cols), "s"(a.group_lanes), "s"(a.groups), "s"(a.window_log),
                 "s"(a.lanes_inv), "s"(a.groups_inv));
}

constexpr int kRpCap = 1024;  // row pointers staged per window
constexpr int kWCap  = 256;   // (col, value) entries a wave stages at a time
constexpr int kMinWindow = 16;  // entries of a group's window: two steps
constexpr int kMaxGroups = kWCap / kMinWindow;  // lane groups of a wave
constexpr int kChains = 4;  // interleaved sums of a row in csr_rowblock

// Third dword of a gfx9 buffer resource: 32-bit data format, no swizzle.
constexpr int kBufWord3 = 0x00020000;

// VEC floats of B row k at byte offset colb: a structured-buffer load (record
// k of N*4 bytes; rows outside [0, K) read as zeros), or a plain 64-bit
// address when B is too large for the buffer form.
template <int VEC, bool SBUF>
__device__ __forceinline__ typename Vec<VEC>::T load_b(__amdgpu_buffer_rsrc_t rsrc,
                                                       const float* bcol, int k, int colb,
                                                       int N) {
    if constexpr (SBUF) {
        if constexpr (VEC == 4) return sbuf_load_x4(rsrc, k, colb, 0, 0);
        else if constexpr (VEC == 2) return sbuf_load_x2(rsrc, k, colb, 0, 0);
        else return sbuf_load_x1(rsrc, k, colb, 0, 0);
    } else {
        return *reinterpret_cast<const typename Vec<VEC>::Mem*>(bcol + static_cast<size_t>(k) * N);
    }
}

template <int VEC>
__device__ __forceinline__ void store_vec(float* p, typename Vec<VEC>::T v) {
    __builtin_nontemporal_store(v, reinterpret_cast<typename Vec<VEC>::Mem*>(p));
}

// First column of the VEC a lane owns: col, or the row's (slice's) last VEC
// columns when fewer than VEC are left from col on.  Those overlap the lane
// before, which sums the same entries in the same order, so both store the same
// bits.  Lanes past the end get that chunk too and store nothing.
template <int VEC>
__device__ __forceinline__ int lane_col(int col, int cend) {
    return VEC == 1 ? min(col, cend - 1) : min(col, max(cend - VEC, 0));
}

__device__ __forceinline__ float shfl_xor_f(float v, int m) { return __shfl_xor(v, m); }

template <int VEC>
__device__ __forceinline__ typename Vec<VEC>::T fma_vec(float v, typename Vec<VEC>::T b,
                                                        typename Vec<VEC>::T acc) {
    if constexpr (VEC == 1) {
        return __builtin_fmaf(v, b, acc);
    } else {
#pragma unroll
        for (int i = 0; i < VEC; ++i) acc[i] = __builtin_fmaf(v, b[i], acc[i]);
        return acc;
    }
}

// ---------------------------------------------------------------------------
// Role: spmm_baseline, spmm_memopt, spmm_memopt_v2: every output is one chain of
// fused multiply-adds in the row's order, the reference kernels' bits.
//
// The chain leaves the columns and the rows to run in parallel and, inside a
// row, the loads: L column lanes of VEC floats own a row (64 / L rows per wave),
// U entries' B segments are in flight while the chain takes them in order.  The
// group loads L column indices and values at a time, one each per lane, and
// hands them out by readlane (L = 64: one row per wave, so the B row's address
// is scalar) or shuffle; groups of under eight lanes load them directly.
// Latency bounds it: U x resident waves loads in flight.  Measured on MI355X
// (launches back to back; one call from Python 69 -> 11.7) against one wave per row
// with 4-byte lanes and one entry at a time: 4096^2, 41 per row, N = 256 64.1 -> 10.4
// us (2.7 -> 16.4 TB/s of gathered rows), N = 128 20.8 -> 6.7 us; 65536^2, 16 per row,
// N = 1 45.0 -> 8.2 us; and against one lane per output (spmm_baseline before) 25.8 ->
// 10.4, 13.9 -> 6.7 and 38.9 -> 8.2 us.
// ---------------------------------------------------------------------------
enum class Hand { Direct, Shuffle, Readlane };

template <int VEC, Hand HAND>
__global__ __launch_bounds__(256) void csr_rows_in_order(
    int M, int N, int lc_log, const int* __restrict__ row_ptr, const int* __restrict__ col_idx,
    const float* __restrict__ vals, const float* __restrict__ B, float* __restrict__ C) {
    using VT = typename Vec<VEC>::T;
    using MT = typename Vec<VEC>::Mem;
    constexpr int U = HAND == Hand::Readlane ? 16 : 8;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int L    = HAND == Hand::Readlane ? kWave : 1 << lc_log;
    const int gl   = lane & (L - 1);
    const int row  = (blockIdx.x * 4 + wave) * (kWave / L) +
                    (HAND == Hand::Readlane ? 0 : lane >> lc_log);
    if (row >= M) return;  // whole groups, and no barrier follows
    const int p0 = row_ptr[row];
    const int p1 = row_ptr[row + 1];
    float* crow = C + static_cast<size_t>(row) * N;
    for (int n0 = blockIdx.y * (L * VEC); n0 < N; n0 += gridDim.y * (L * VEC)) {
        const int    col  = lane_col<VEC>(n0 + gl * VEC, N);
        const float* bcol = B + col;
        VT acc = vzero<VEC>();
        // Entries [p, p + cnt) of the chain, cnt <= L, U at a time; entry j is
        // handed out by take(j).
        auto step = [&](int j0, int cnt, auto take, auto width) {
            constexpr int W = decltype(width)::value;
            VT    b[W];
            float v[W];
#pragma unroll
            for (int u = 0; u < W; ++u) {
                int k;
                take(min(j0 + u, cnt - 1), k, v[u]);
                b[u] = *reinterpret_cast<const MT*>(bcol + static_cast<size_t>(k) * N);
            }
            if (j0 + W <= cnt) {
#pragma unroll
                for (int u = 0; u < W; ++u) acc = fma_vec<VEC>(v[u], b[u], acc);
            } else {
#pragma unroll
                for (int u = 0; u < W; ++u) {
                    if (j0 + u < cnt) acc = fma_vec<VEC>(v[u], b[u], acc);
                }
            }
        };
        // Up to four entries left: four loads instead of U (3034 rows of 2.4, N = 320
        // 6.0 -> 4.8 us).
        auto chain = [&](int cnt, auto take) {
            for (int j0 = 0; j0 < cnt; j0 += U) {
                if (HAND == Hand::Readlane && cnt - j0 <= 4) {  // the wave's one row: uniform
                    step(j0, cnt, take, std::integral_constant<int, 4>());
                } else {
                    step(j0, cnt, take, std::integral_constant<int, U>());
                }
            }
        };
        if constexpr (HAND == Hand::Direct) {
            chain(p1 - p0, [&](int j, int& k, float& v) {
                k = col_idx[p0 + j];
                v = vals[p0 + j];
            });
        } else {
            for (int p = p0; p < p1; p += L) {
                const int   q  = min(p + gl, p1 - 1);
                const int   kc = col_idx[q];
                const float vc = vals[q];
                chain(min(L, p1 - p), [&](int j, int& k, float& v) {
                    if constexpr (HAND == Hand::Readlane) {
                        k = __builtin_amdgcn_readlane(kc, j);
                        v = __builtin_bit_cast(
                            float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, vc), j));
                    } else {
                        k = __shfl(kc, (lane & ~(L - 1)) + j);
                        v = __shfl(vc, (lane & ~(L - 1)) + j);
                    }
                });
            }
        }
        if (n0 + gl * VEC < N) store_vec<VEC>(crow + col, acc);
    }
}

// Orders a wave's LDS writes before its own lanes' reads of them.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One staged entry of A: the B row in the low half, the value in the high one
// (a single 8-byte LDS read; as two fields the compiler reads them apart).
typedef uint64_t Entry;
__device__ __forceinline__ Entry entry(int k, float v) {
    return static_cast<uint32_t>(k) | (static_cast<Entry>(__builtin_bit_cast(uint32_t, v)) << 32);
}
__device__ __forceinline__ int entry_row(Entry e) { return static_cast<int>(e); }
__device__ __forceinline__ float entry_value(Entry e) {
    return __builtin_bit_cast(float, static_cast<uint32_t>(e >> 32));
}

template <int VEC, int WAVES, int U, bool SBUF, bool HALVES, bool FOLD>
__global__ __launch_bounds__(WAVES * 64, U == 8 ? 4 : 5) void csr_rowblock(RowblockArgs a) {
    using VT = typename Vec<VEC>::T;
    static_assert(kWCap % kWave == 0 && kMinWindow % U == 0, "whole steps per window");
    static_assert(U % kChains == 0, "an entry's chain is fixed by its place in the step");

    __shared__ int  s_rp[kRpCap + 2];
    __shared__ VT   s_part[WAVES * kWave];   // by group and lane: the group's head piece
    __shared__ int  s_first[WAVES * kWave];  // by group: see below
    __shared__ Entry s_kv[WAVES][kWCap + kMaxGroups * (2 * U + 1)];

    load_args(a, a.part);
    const int lane  = threadIdx.x & (kWave - 1);
    const int wave  = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lpg   = a.group_lanes;
    const int G     = a.groups;
    const int NG    = WAVES * G;
    // A lane's place.  Lanes past the last group shadow its last lane and never
    // store.  Worked out anew where it is needed: held over the entry loop it
    // would take registers from the rows in flight.
    struct Place {
        int  grp, glane;
        int  gi;  // group of the workgroup
        bool live;
    };
    auto place = [&] {
        int l = lane;
        asm volatile("" : "+v"(l));
        const int g  = min(l * a.lanes_inv >> 16, G - 1);
        const int gl = min(l - g * lpg, lpg - 1);
        return Place{g, gl, wave * G + g, l < G * lpg};
    };
    const int N     = a.N;
    const int cap   = 1 << a.window_log;  // entries a group stages at a time
    const int cols  = lpg * VEC;          // columns per pass

    // Column slices are tied to XCDs: workgroups are dispatched round-robin
    // over the 8 XCDs, so workgroup g runs on XCD g % 8.  With S slices, XCDs
    // s*8/S .. (s+1)*8/S - 1 compute columns [s*SC, (s+1)*SC) of every row
    // block, so each XCD's L2 holds only 1/S of B.  With B-row halves, XCDs
    // 0-3 work through the parts of the first descriptor and XCDs 4-7 through
    // those of the second (all columns each).
    int rb = blockIdx.x, slice = 0, half = 0;
    if constexpr (HALVES) {
        const int x = blockIdx.x & 7;
        rb   = (blockIdx.x >> 3) * 4 + (x & 3);
        half = x >> 2;
    } else if (a.slices > 1) {
        const int per = 8 / a.slices;  // XCDs per slice
        const int x   = blockIdx.x & 7;
        rb    = (blockIdx.x >> 3) * per + x % per;
        slice = x / per;
    }
    const RowblockPart m = HALVES && half ? a.upper : a.part;
    if (rb >= m.nblocks) return;  // whole workgroup, before any barrier
    const int cbeg = slice * a.slice_cols;
    const int cend = min(N, cbeg + a.slice_cols);

    int r_begin, r_end, zero_end;
    const bool split = m.split_rows != nullptr;
    long long nz_lo = 0, nz_hi = 0;
    int wg_head = -1;  // first row, when it began in an earlier part (merge-path only)
    if (split) {
        nz_lo    = m.nnz * rb / m.nblocks;
        nz_hi    = m.nnz * (rb + 1) / m.nblocks;
        r_begin  = m.split_rows[rb];
        zero_end = m.split_rows[rb + 1];          // empty rows [r_begin, zero_end) are ours
        r_end    = min(a.M, zero_end + 1);         // + the row our last nonzeros start
        if (nz_lo < nz_hi && r_begin < a.M && m.row_ptr[r_begin] < nz_lo) wg_head = r_begin;
    } else if (a.bounds != nullptr) {
        r_begin  = a.bounds[rb];
        r_end    = a.bounds[rb + 1];
        zero_end = r_end;
    } else {
        r_begin  = rb * a.rows_per_block;
        r_end    = min(a.M, r_begin + a.rows_per_block);
        zero_end = r_end;
    }

    __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(m.B), static_cast<short>(SBUF ? N * 4 : 0), SBUF ? m.K : 0, kBufWord3);
    Entry* const kv = s_kv[wave];
    // A group's window and the 2U empty entries that the last steps' loads may
    // read; an odd stride puts the groups' windows on different banks.
    const int kv_len  = cap + 2 * U + 1;
    {
        const Place me = place();
        for (int i = me.glane; i <= 2 * U; i += lpg) {
            kv[me.grp * kv_len + cap + i] = entry(SBUF ? -1 : 0, 0.0f);
        }
    }

    for (int w0 = r_begin; w0 < r_end; w0 += kRpCap) {
        const int nr = min(r_end - w0, kRpCap);
        __syncthreads();  // the previous window is no longer read
        for (int i = threadIdx.x; i <= nr; i += WAVES * kWave) s_rp[i] = m.row_ptr[w0 + i];
        __syncthreads();

        // Zero-fill the rows of this window that hold no nonzeros.
        for (int base = wave * kWave; base < nr; base += WAVES * kWave) {
            const int i = base + lane;
            uint64_t empty = __ballot(i < nr && w0 + i < zero_end && s_rp[i] == s_rp[i + 1]);
            while (empty) {
                const int b = __builtin_ctzll(empty);
                empty &= empty - 1;
                float* crow = m.C + static_cast<size_t>(w0 + base + b) * N;
                for (int c = cbeg + lane * VEC; c < cend; c += kWave * VEC) {
                    store_vec<VEC>(crow + lane_col<VEC>(c, cend), vzero<VEC>());
                }
            }
        }

        int nz0 = s_rp[0];
        int nz_end = s_rp[nr];
        if (split) {
            nz0    = static_cast<int>(max(static_cast<long long>(nz0), nz_lo));
            nz_end = static_cast<int>(min(static_cast<long long>(nz_end), nz_hi));
        }
        const int total = nz_end - nz0;
        if (total <= 0) continue;  // uniform across the workgroup
        // Entries per group: an equal share, in whole steps (total / NG or
        // just over, by the reciprocal).
        const int share =
            (static_cast<int>(__umulhi(total, a.groups_inv)) / WAVES + U) / U * U;
        const unsigned rest = total;
        const unsigned from = min(rest, static_cast<unsigned>(wave * G) * share);  // the wave's first
        const int gi   = place().gi;
        const int pa   = nz0 + static_cast<int>(min(rest, static_cast<unsigned>(gi) * share));
        const int pb   = nz0 + static_cast<int>(min(rest, static_cast<unsigned>(gi + 1) * share));
        const int wlen = static_cast<int>(min<unsigned>(share, rest - from));  // its longest range

        // First local row: the last i in [0, nr) with s_rp[i] <= pa.
        int first = 0;
        {
            int lo = 0, hi = nr - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (s_rp[mid] <= pa) lo = mid; else hi = mid - 1;
            }
            first = lo;
        }

        // Copies entries win .. win + cap - 1 of each group's range into the
        // groups' LDS windows, one coalesced run per group, all loads issued
        // before the first LDS write.  Slots past a group's range hold record
        // -1 (reads zeros) and value 0.
        const char* cols_at = reinterpret_cast<const char*>(m.col_idx + nz0 + from);
        const char* vals_at = reinterpret_cast<const char*>(m.vals + nz0 + from);
        auto stage = [&](int win) {
            constexpr int NL = kWCap / kWave;
            int   kk[NL];
            float vx[NL];
            int   l = lane;
            asm volatile("" : "+v"(l));  // keeps the slot arithmetic out of the entry loop's registers
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const int idx = i * kWave + l;
                const int off = win + (idx & (cap - 1));
                const unsigned e  = static_cast<unsigned>(idx >> a.window_log) * share + off;
                const bool     in = off < share && e < rest - from;
                const unsigned at = (in ? e : 0u) * 4u;
                kk[i] = *reinterpret_cast<const int*>(cols_at + at);
                vx[i] = *reinterpret_cast<const float*>(vals_at + at);
                if (!in) {
                    kk[i] = SBUF ? -1 : 0;
                    vx[i] = 0.0f;
                }
            }
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const int idx = i * kWave + l;
                const int h   = idx >> a.window_log;
                if (h < G) {
                    kv[h * kv_len + (idx & (cap - 1))] =
                        entry(kk[i], vx[i]);
                }
            }
            wave_lds_sync();
        };

        // A range that fits one window is staged once for all column passes.
        const bool one_window = wlen <= cap;
        if (wlen > 0 && one_window) stage(0);

        for (int c0 = cbeg; c0 < cend; c0 += cols) {
            int  colb;    // byte offset of the lane's columns
            bool writer;  // whether the lane stores them
            {
                const Place me = place();
                colb   = lane_col<VEC>(c0 + me.glane * VEC, cend) * 4;
                writer = me.live && c0 + me.glane * VEC < cend;
                if (me.live && me.glane == 0) s_first[me.gi] = -1;
            }
            const float* bcol = reinterpret_cast<const float*>(reinterpret_cast<const char*>(m.B) + colb);
            // Puts v aside as the group's piece of local row r.
            auto put_piece = [&](int r, VT v) {
                const Place me = place();
                if (me.live) s_part[me.gi * lpg + me.glane] = v;
                if (me.live && me.glane == 0) s_first[me.gi] = r;
            };
            auto store_row = [&](float* base, unsigned r, VT v) {
                unsigned cb = colb;
                asm volatile("" : "+v"(cb));  // keeps base + cb out of the entry loop's registers
                if (writer) {
                    store_vec<VEC>(reinterpret_cast<float*>(
                        reinterpret_cast<char*>(base) + (static_cast<size_t>(r) * (4u * N) + cb)), v);
                }
            };

            int owner_row = -1;  // local row this group finishes after the barrier
            VT acc[kChains];
            const auto clear = [&] {
#pragma unroll
                for (int i = 0; i < kChains; ++i) acc[i] = vzero<VEC>();
            };
            const auto sum = [&] { return (acc[0] + acc[1]) + (acc[2] + acc[3]); };
            // v plus the pieces of local row r that groups from w on put aside, in two chains.
            auto add_pieces = [&](VT v, int w, int r) {
                const int at = place().glane;
                VT odd = vzero<VEC>();
                for (; w < NG && s_first[w] == r; w += 2) {
                    v += s_part[w * lpg + at];
                    if (w + 1 == NG || s_first[w + 1] != r) break;
                    odd += s_part[(w + 1) * lpg + at];
                }
                return v + odd;
            };
            clear();
            VT folded = vzero<VEC>();  // FOLD: the row's sum over earlier windows
            if (wlen > 0) {
                int  row  = first;
                bool head = s_rp[row] < pa;  // row began in an earlier group
                // Where the row ends inside the range (counted from its
                // start), or never.
                int row_len;
                {
                    const int e = s_rp[row + 1];
                    row_len = e < pb ? e - pa : 0x7fffffff;
                }

                int next_end = s_rp[row + 2 <= nr ? row + 2 : nr];

                auto flush = [&](int at) {
                    VT done = sum();
                    if constexpr (FOLD) {
                        done += folded;
                        folded = vzero<VEC>();
                    }
                    if (head) {
                        put_piece(row, done);
                        head = false;
                    } else {
                        store_row(m.C, w0 + row, done);
                    }
                    clear();
                    ++row;
                    int e = next_end;
                    while (e <= at + pa && row < nr - 1) {  // empty rows
                        ++row;
                        e = s_rp[row + 1];
                    }
                    next_end = s_rp[min(row + 2, nr)];
                    row_len = e < pb ? e - pa : 0x7fffffff;
                };

                for (int win = 0; win < wlen; win += cap) {
                    if (!one_window) stage(win);
                    const int n = min(cap, wlen - win);

                    // U rows in flight per group, each register refilled as
                    // soon as it is used; the entries of the next step are
                    // read from LDS one step ahead.
                    VT    bv[U];
                    float vv[U];
                    Entry next[U];
                    int at_kv = place().grp * kv_len;
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        vv[u] = entry_value(kv[at_kv + u]);
                        bv[u] = load_b<VEC, SBUF>(rsrc, bcol, entry_row(kv[at_kv + u]), colb, N);
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) next[u] = kv[at_kv + U + u];
                    // Only the row end branches, never the loads: values loaded
                    // on two paths would have to arrive before the paths join.
                    auto step = [&](int at0, auto refill) {
                        const bool ends = __ballot(row_len < at0 + U) != 0;
                        // Pointer loads cannot read zeros for entries past a range.
                        const bool past = !SBUF && __ballot(at0 + U > pb - pa) != 0;
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            if (__builtin_expect(ends, 0)) {
                                if (at0 + u == row_len) flush(at0 + u);
                            }
                            VT& a_u = acc[u % kChains];
                            if (!past || at0 + u < pb - pa) a_u = vv[u] * bv[u] + a_u;
                            if constexpr (decltype(refill)::value) {
                                __builtin_amdgcn_sched_barrier(0);  // into the registers just used
                                vv[u] = entry_value(next[u]);
                                bv[u] = load_b<VEC, SBUF>(rsrc, bcol, entry_row(next[u]), colb, N);
                                next[u] = kv[at_kv + 2 * U + u];
                                __builtin_amdgcn_sched_barrier(0);  // a step ahead of its use
                            }
                        }
                    };
                    int q = 0;
                    for (; q + U < n; q += U) {
                        step(win + q, std::true_type());
                        at_kv += U;
                        asm volatile("" : "+v"(at_kv));  // one address, the reads at constant offsets
                    }
                    step(win + q, std::false_type());
                    if constexpr (FOLD) {  // chains no longer than a window's
                        if (win + cap < wlen) {
                            folded += sum();
                            clear();
                        }
                    }
                }
                // The row being accumulated when the range ends.
                acc[0] = sum();
                if constexpr (FOLD) acc[0] += folded;
                if (pa < pb) {
                    if (head) {
                        put_piece(row, acc[0]);
                    } else if (s_rp[row + 1] <= pb) {
                        store_row(m.C, w0 + row, acc[0]);
                    } else {
                        owner_row = row;
                    }
                }
            }
            __syncthreads();
            const int gi_now = place().gi;
            if (owner_row >= 0) {
                store_row(m.C, w0 + owner_row, add_pieces(acc[0], gi_now + 1, owner_row));
            }
            if (wg_head >= 0 && w0 == r_begin && gi_now == 0) {
                // The part's first row began in an earlier part: the groups that
                // hold pieces of it (local row 0, leading groups) go to the carry.
                store_row(m.carry, rb, add_pieces(vzero<VEC>(), 0, 0));
            }
            __syncthreads();  // s_part / s_first are rewritten by the next column pass
        }
    }
}

// ---------------------------------------------------------------------------
// The engine on wide B (one or two lane groups per wave) where the partition
// is balanced beforehand: merge-path parts, and rows that the caller's longest
// row shows to be even.  As csr_rowblock, except that the groups of a wave take
// alternate entries of one range instead of a range each, in steps of U * G
// entries with the next step's loads issued before the current one is used, and
// sum their tiles with xor shuffles at a row end.  A scalar test per step sends
// only the steps that hold a row end to the slow path, so this form spends less
// per entry and starts half as many row pieces; csr_rowblock's groups wait for
// nobody and win from three groups on and on uneven rows.  MI355X, this form
// against csr_rowblock: 16384^2 power-law over B-row halves, N = 128 61.3 against
// 62.7 us; 8192^2, 100 per row, N = 256 36.2 against 36.3, N = 128 19.6 against 20.3;
// 2048^2, 235 per row, N = 256 19.1 against 19.9; merge-path 8192^2 power-law, N = 32
// (eight groups) 19.0 against 14.2.
// ---------------------------------------------------------------------------
// Sum of the G groups' tiles, returned to every lane.
template <int G>
__device__ __forceinline__ f32x4 reduce_groups(f32x4 v) {
#pragma unroll
    for (int m = kWave / G; m < kWave; m <<= 1) {
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = shfl_xor_f(v[e], m);
        v += o;
    }
    return v;
}

template <int G, int WAVES, bool HALVES>
__global__ __launch_bounds__(WAVES * 64) void csr_rowblock_wide(RowblockArgs a) {
    constexpr int VEC = 4, U = 4;
    using VT = f32x4;
    constexpr int LPG  = kWave / G;   // lanes per group
    constexpr int COLS = LPG * VEC;   // columns per pass
    constexpr int STEP = U * G;       // entries per step
    static_assert(kWave % STEP == 0 && kWCap % kWave == 0, "U * G must divide the wave size");

    __shared__ int  s_rp[kRpCap + 1];
    __shared__ VT   s_part[WAVES][LPG];
    __shared__ int  s_first[WAVES];
    __shared__ int2 s_kv[WAVES][kWCap + STEP];

    load_args(a, a.part);
    const int lane  = threadIdx.x & (kWave - 1);
    const int wave  = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp   = lane / LPG;
    const int glane = lane % LPG;
    const int N     = a.N;

    // Column slices and B-row halves as in csr_rowblock.
    int rb = blockIdx.x, slice = 0, half = 0;
    if constexpr (HALVES) {
        const int x = blockIdx.x & 7;
        rb   = (blockIdx.x >> 3) * 4 + (x & 3);
        half = x >> 2;
    } else if (a.slices > 1) {
        const int per = 8 / a.slices;
        const int x   = blockIdx.x & 7;
        rb    = (blockIdx.x >> 3) * per + x % per;
        slice = x / per;
    }
    const RowblockPart m = HALVES && half ? a.upper : a.part;
    if (rb >= m.nblocks) return;  // whole workgroup, before any barrier
    const int cbeg = slice * a.slice_cols;
    const int cend = min(N, cbeg + a.slice_cols);

    int r_begin, r_end, zero_end;
    const bool split = m.split_rows != nullptr;
    long long nz_lo = 0, nz_hi = 0;
    int wg_head = -1;  // first row, when it began in an earlier part (merge-path only)
    if (split) {
        nz_lo    = m.nnz * rb / m.nblocks;
        nz_hi    = m.nnz * (rb + 1) / m.nblocks;
        r_begin  = m.split_rows[rb];
        zero_end = m.split_rows[rb + 1];          // empty rows [r_begin, zero_end) are ours
        r_end    = min(a.M, zero_end + 1);         // + the row our last nonzeros start
        if (nz_lo < nz_hi && r_begin < a.M && m.row_ptr[r_begin] < nz_lo) wg_head = r_begin;
    } else {
        r_begin  = rb * a.rows_per_block;
        r_end    = min(a.M, r_begin + a.rows_per_block);
        zero_end = r_end;
    }

    __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(m.B), static_cast<short>(N * 4), m.K, kBufWord3);
    // Entries past a window's end read by the masked lanes of its last step.
    for (int i = lane; i < STEP; i += kWave) s_kv[wave][kWCap + i] = make_int2(0, 0);

    // Copies entries [lo, hi) (hi - lo <= kWCap) into the wave's LDS window;
    // the rest of the window holds (0, 0).  All loads are issued before the
    // first LDS write.
    auto stage = [&](int lo, int hi) {
        constexpr int NL = kWCap / kWave;
        int   kk[NL];
        float vx[NL];
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int e = min(lo + i * kWave + lane, hi - 1);
            kk[i] = m.col_idx[e];
            vx[i] = m.vals[e];
        }
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const bool in = lo + i * kWave + lane < hi;
            s_kv[wave][i * kWave + lane] =
                make_int2(in ? kk[i] : 0, in ? __builtin_bit_cast(int, vx[i]) : 0);
        }
        wave_lds_sync();
    };

    for (int w0 = r_begin; w0 < r_end; w0 += kRpCap) {
        const int nr = min(r_end - w0, kRpCap);
        __syncthreads();  // the previous window is no longer read
        for (int i = threadIdx.x; i <= nr; i += WAVES * kWave) s_rp[i] = m.row_ptr[w0 + i];
        __syncthreads();

        // Zero-fill the rows of this window that hold no nonzeros.
        for (int base = wave * kWave; base < nr; base += WAVES * kWave) {
            const int i = base + lane;
            uint64_t empty = __ballot(i < nr && w0 + i < zero_end && s_rp[i] == s_rp[i + 1]);
            while (empty) {
                const int b = __builtin_ctzll(empty);
                empty &= empty - 1;
                float* crow = m.C + static_cast<size_t>(w0 + base + b) * N;
                for (int c = cbeg + lane * VEC; c < cend; c += kWave * VEC) {
                    store_vec<VEC>(crow + lane_col<VEC>(c, cend), vzero<VEC>());
                }
            }
        }

        int nz0 = s_rp[0];
        int nz_end = s_rp[nr];
        if (split) {
            nz0    = static_cast<int>(max(static_cast<long long>(nz0), nz_lo));
            nz_end = static_cast<int>(min(static_cast<long long>(nz_end), nz_hi));
        }
        const int total = nz_end - nz0;
        if (total <= 0) continue;  // uniform across the workgroup
        const int pa = nz0 + static_cast<int>((static_cast<long long>(total) * wave) / WAVES);
        const int pb = nz0 + static_cast<int>((static_cast<long long>(total) * (wave + 1)) / WAVES);

        // First local row: the last i in [0, nr) with s_rp[i] <= pa.
        int first = 0;
        {
            int lo = 0, hi = nr - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (s_rp[mid] <= pa) lo = mid; else hi = mid - 1;
            }
            first = lo;
        }

        // A range that fits one window is staged once for all column passes.
        const bool one_window = pb - pa <= kWCap;
        if (one_window && pa < pb) stage(pa, pb);

        for (int c0 = cbeg; c0 < cend; c0 += COLS) {
            const int  col    = lane_col<VEC>(c0 + glane * VEC, cend);
            const bool writer = grp == 0 && c0 + glane * VEC < cend;
            if (lane == 0) s_first[wave] = (pa < pb) ? -1 : -2;

            int owner_row = -1;  // local row this wave finishes after the barrier
            VT acc = vzero<VEC>();
            if (pa < pb) {
                int  row     = first;
                int  row_end = s_rp[row + 1];
                bool head    = s_rp[row] < pa;  // row began in an earlier wave

                auto flush = [&]() {
                    const VT t = reduce_groups<G>(acc);
                    if (head) {
                        if (grp == 0) s_part[wave][glane] = t;
                        if (lane == 0) s_first[wave] = row;
                        head = false;
                    } else if (writer) {
                        store_vec<VEC>(m.C + static_cast<size_t>(w0 + row) * N + col, t);
                    }
                    acc = vzero<VEC>();
                };

                for (int win = pa; win < pb; win += kWCap) {
                    const int win_end = min(pb, win + kWCap);
                    if (!one_window) stage(win, win_end);

                    VT    bA[U], bB[U];
                    float vA[U], vB[U];
                    // Loads of the step starting at entry q.
                    auto issue = [&](VT (&bv)[U], float (&vv)[U], int q) {
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            const int2 kv = s_kv[wave][q - win + u * G + grp];
                            vv[u] = __builtin_bit_cast(float, kv.y);
                            bv[u] = load_b<VEC, true>(rsrc, nullptr, kv.x, col * 4, N);
                        }
                    };
                    // Accumulates the step starting at entry q.
                    auto consume = [&](VT (&bv)[U], float (&vv)[U], int q) {
                        if (q + STEP <= row_end && q + STEP <= win_end) {
#pragma unroll
                            for (int u = 0; u < U; ++u) acc = vv[u] * bv[u] + acc;
                        } else {
#pragma unroll
                            for (int u = 0; u < U; ++u) {
#pragma unroll
                                for (int h = 0; h < G; ++h) {
                                    const int P = q + u * G + h;
                                    if (P < win_end) {
                                        if (P >= row_end) {
                                            flush();
                                            // bounded by the window even for a malformed row_ptr
                                            do {
                                                ++row;
                                                row_end = s_rp[row + 1];
                                            } while (row_end <= P && row < nr - 1);
                                        }
                                        if (grp == h) acc = vv[u] * bv[u] + acc;
                                    }
                                }
                            }
                        }
                    };
                    issue(bA, vA, win);
                    for (int q = win; q < win_end; q += 2 * STEP) {
                        if (q + STEP < win_end) issue(bB, vB, q + STEP);
                        consume(bA, vA, q);
                        if (q + STEP >= win_end) break;
                        if (q + 2 * STEP < win_end) issue(bA, vA, q + 2 * STEP);
                        consume(bB, vB, q + STEP);
                    }
                }
                // The row being accumulated when the range ends.
                acc = reduce_groups<G>(acc);
                if (row_end == pb && !head) {
                    if (writer) store_vec<VEC>(m.C + static_cast<size_t>(w0 + row) * N + col, acc);
                } else if (head) {
                    if (grp == 0) s_part[wave][glane] = acc;
                    if (lane == 0) s_first[wave] = row;
                } else {
                    owner_row = row;
                }
            }
            __syncthreads();
            if (owner_row >= 0) {
                for (int w = wave + 1; w < WAVES; ++w) {
                    const int f = s_first[w];
                    if (f == -2) continue;
                    if (f != owner_row) break;
                    acc += s_part[w][glane];
                }
                if (writer) store_vec<VEC>(m.C + static_cast<size_t>(w0 + owner_row) * N + col, acc);
            }
            if (wg_head >= 0 && w0 == r_begin && wave == 0) {
                // The part's first row began in an earlier part: the waves that
                // hold pieces of it (local row 0, leading waves) go to the carry.
                VT sum = vzero<VEC>();
                for (int w = 0; w < WAVES; ++w) {
                    const int f = s_first[w];
                    if (f == -2) continue;
                    if (f != 0) break;
                    sum += s_part[w][glane];
                }
                if (writer) store_vec<VEC>(m.carry + static_cast<size_t>(rb) * N + col, sum);
            }
            __syncthreads();  // s_part / s_first are rewritten by the next column pass
        }
    }
}

// Merge-path fix-up: row r that continues into parts g0+1 .. g1 was stored by
// the part where it starts; the first continuation part adds the carries of
// parts g0+1 .. g1 in part order (deterministic) to C[r].  Every part holds at
// least one nonzero (the launcher requires parts <= nnz), so part q > g
// continues row r exactly when split_rows[q] == r.  One wave per part, and
// the loads are arranged in three dependent rounds: the part's row; that
// row's first nonzero together with the rows of the next 64 parts (a ballot
// finds where the run ends); the carries together with C.
constexpr int kFixupCols = 4;  // columns per lane in flight

__global__ __launch_bounds__(64) void csr_split_fixup(const int* __restrict__ row_ptr,
                                                      const int* __restrict__ split_rows,
                                                      const float* __restrict__ carry,
                                                      float* __restrict__ C, int M, int N,
                                                      long long nnz, int parts) {
    const int g    = blockIdx.x;
    const int lane = threadIdx.x;
    const long long lo = nnz * g / parts;
    const long long hi = nnz * (g + 1) / parts;
    const int r  = split_rows[g];
    const int rp = g > 0 ? split_rows[g - 1] : -1;
    if (!(lo < hi && r >= 0 && r < M)) return;
    int base = g + 1;
    int q    = base + lane;
    int w    = q < parts ? split_rows[q] : -1;  // issued before row_ptr[r] returns
    const int rs = row_ptr[r];
    if (rs >= lo) return;  // part g starts row r and stored it
    // part g continues row r; the previous part also continues it when it
    // holds row r and r began before that part's first nonzero
    if (g > 0 && rp == r && rs < nnz * (g - 1) / parts) return;
    int last;
    for (;;) {
        const unsigned long long stop = __ballot(!(q < parts && w == r));
        if (stop != 0ull) {
            last = base + __ffsll(static_cast<long long>(stop)) - 2;
            break;
        }
        base += 64;
        q = base + lane;
        w = q < parts ? split_rows[q] : -1;
    }
    float* crow = C + static_cast<size_t>(r) * N;
    for (int c0 = 0; c0 < N; c0 += 64 * kFixupCols) {
        float cv[kFixupCols], s[kFixupCols];
#pragma unroll
        for (int j = 0; j < kFixupCols; ++j) {
            const int c = c0 + lane + 64 * j;
            cv[j] = c < N ? crow[c] : 0.f;
            s[j]  = 0.f;
        }
        for (int p = g; p <= last; ++p) {
            const float* cr = carry + static_cast<size_t>(p) * N;
#pragma unroll
            for (int j = 0; j < kFixupCols; ++j) {
                const int c = c0 + lane + 64 * j;
                if (c < N) s[j] += cr[c];
            }
        }
#pragma unroll
        for (int j = 0; j < kFixupCols; ++j) {
            const int c = c0 + lane + 64 * j;
            if (c < N) crow[c] = cv[j] + s[j];
        }
    }
}

// Fix-up of the B-row halves: C = (C + carries of half 0) + (partial +
// carries of half 1), row by row, each sum of carries in part order --
// the same order on every launch.  runs[r] = (first, last) continuation part
// of row r in half 0, then in half 1, -1 for none.  One 16-byte chunk of C and
// of the partial per thread (N % 4 == 0); both are read once, so the loads
// stream (measured on c5: 61.4 -> 60.2 us per launch against cached loads
// two chunks per thread).
__global__ __launch_bounds__(256) void csr_khalf_fixup(float* __restrict__ C,
                                                       const float* __restrict__ partial,
                                                       const float* __restrict__ carry0,
                                                       const float* __restrict__ carry1,
                                                       const int4* __restrict__ runs, int N,
                                                       long long chunks) {
    const long long t = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
    if (t >= chunks) return;
    const int4 ru = runs[t * 4 / N];
    f32x4 cv = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(C) + t);
    f32x4 pv = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(partial) + t);
    const int c = static_cast<int>(t * 4 % N);
    if (ru.x >= 0) {
        f32x4 s = f32x4(0.f);
        for (int p = ru.x; p <= ru.y; ++p) {
            s += *reinterpret_cast<const f32x4*>(carry0 + static_cast<size_t>(p) * N + c);
        }
        cv += s;
    }
    if (ru.z >= 0) {
        f32x4 s = f32x4(0.f);
        for (int p = ru.z; p <= ru.w; ++p) {
            s += *reinterpret_cast<const f32x4*>(carry1 + static_cast<size_t>(p) * N + c);
        }
        pv += s;
    }
    __builtin_nontemporal_store(cv + pv, reinterpret_cast<f32x4*>(C) + t);
}

// ---------------------------------------------------------------------------
// Sub-wave row groups (the short-row / narrow-N form of spmm_tiled_v3).
//
// A group of L = LC * LE lanes owns one row: LC column lanes cover LC * VEC
// contiguous columns (one pass; more passes when N is wider) and LE entry
// lanes take the row's entries e, e + LE, e + 2*LE, ... so each lane gathers
// whole VEC-float segments of B rows for its own entries.  A wave holds
// 64 / L rows, a 256-thread workgroup four waves; rows never cross groups, so
// there is no row bookkeeping in the loop, and the group phase needs no LDS
// and no barrier.  At the end of a row the entry lanes' partials are summed
// with xor shuffles (fixed order) and entry lane 0 stores the row.
//
// For N of a few columns the row-block engine leaves most lanes idle (its
// groups cover columns, at most 16 per wave) and pays its per-step row tests on
// every entry; here a wave gathers 64 / LC entries per load instruction.
// Measured on MI355X: 1.5 - 4x faster than the engine for N <= 32 on uniform
// rows of 1 .. 300 entries, up to 2x at N = 64, and for N = 128 / 256 on rows
// of a few entries.
//
// A row longer than 8 iterations of its group (8 * LE * U entries) and than
// 4x the average row is not taken by the group but by the whole workgroup
// afterwards (4 * 64 / LC entry lanes, partials added through LDS), so it is
// taken by 256 / L times the lanes.  (Rows of about average length stay in
// their groups: moving them would only serialise the workgroup's rows.)  Rows far longer than that belong
// to the engine or the merge-path partition, which share a row between waves
// and workgroups; the dispatch rule below keeps them there.
// ---------------------------------------------------------------------------
struct RowGroupArgs {
    const int*   row_ptr;
    const int*   col_idx;
    const float* vals;
    const float* B;
    float*       C;
    int          M;
    int          N;
    int          K;
    int          lc_log;    // column lanes per row: 1 << lc_log
    int          le_log;    // entry lanes per row: 1 << le_log
    int          long_len;  // rows with more entries go to the workgroup-wide pass
    int          slices;    // XCD-tied column slices: 1, 2, 4 or 8
    int          slice_cols;
    int          nblocks;   // row blocks (workgroups of one column slice)
    // Rows of up to few_len entries take 1 << few_log entry lanes of the 1 << le_log.
    int          few_log = 0;
    int          few_len = 0;
};

template <int VEC>
__device__ __forceinline__ typename Vec<VEC>::T xor_add(typename Vec<VEC>::T v, int m) {
    if constexpr (VEC == 1) {
        return v + shfl_xor_f(v, m);
    } else {
        typename Vec<VEC>::T o;
#pragma unroll
        for (int i = 0; i < VEC; ++i) o[i] = shfl_xor_f(v[i], m);
        return v + o;
    }
}

// Sum over the entries p0, p0 + stride, ... (< p1) of the row: U entries per
// iteration, their column indices and values loaded before their B segments.
template <int VEC, int U>
__device__ __forceinline__ typename Vec<VEC>::T row_segment_sum(
    const RowGroupArgs& a, __amdgpu_buffer_rsrc_t rb, int p0, int p1, int stride, int colb) {
    using VT = typename Vec<VEC>::T;
    VT acc = vzero<VEC>();
    for (int p = p0; p < p1; p += stride * U) {
        int   ks[U];
        float vs[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int q = p + u * stride;
            const bool in = q < p1;
            ks[u] = in ? a.col_idx[q] : -1;  // -1: outside the buffer, reads zeros
            vs[u] = in ? a.vals[q] : 0.0f;
        }
        VT bs[U];
#pragma unroll
        for (int u = 0; u < U; ++u) bs[u] = load_b<VEC, true>(rb, nullptr, ks[u], colb, a.N);
#pragma unroll
        for (int u = 0; u < U; ++u) acc += vs[u] * bs[u];
    }
    return acc;
}

// Cooperative form of a group's pass over entries [p0, p1): the L lanes of
// the group (lanes g0 .. g0+L-1, this lane gl) load L consecutive entries with
// one coalesced load for the columns and one for the values, and sub-step j
// hands entry j*LE + e to lane (e, c) with a shuffle -- one load per L entries
// instead of one per entry lane and entry.
template <int VEC, int U>
__device__ __forceinline__ typename Vec<VEC>::T row_chunks_sum(
    const RowGroupArgs& a, __amdgpu_buffer_rsrc_t rb, int p0, int p1, int g0, int gl, int e,
    int L, int LE, int colb, int chunk_stride) {
    using VT = typename Vec<VEC>::T;
    VT acc = vzero<VEC>();
    const int sub = L / LE;  // sub-steps per chunk (= column lanes)
    for (int base = p0; base < p1; base += chunk_stride) {
        const int   q   = base + gl;
        const int   kc  = q < p1 ? a.col_idx[q] : -1;
        const float vc  = q < p1 ? a.vals[q] : 0.0f;
        const int   cnt = min(L, p1 - base);
        for (int j0 = 0; j0 < sub && j0 * LE < cnt; j0 += U) {
            int   ks[U];
            float vs[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int src = g0 + (((j0 + u) * LE + e) & (L - 1));
                ks[u] = __shfl(kc, src);
                vs[u] = __shfl(vc, src);
                if (j0 + u >= sub) {
                    ks[u] = -1;
                    vs[u] = 0.0f;
                }
            }
            VT bs[U];
#pragma unroll
            for (int u = 0; u < U; ++u) bs[u] = load_b<VEC, true>(rb, nullptr, ks[u], colb, a.N);
#pragma unroll
            for (int u = 0; u < U; ++u) acc += vs[u] * bs[u];
        }
    }
    return acc;
}

template <int VEC, int U, bool COOP, bool LONG_ROWS, bool FEW = false>
__global__ __launch_bounds__(256) void csr_row_groups(RowGroupArgs a) {
    using VT = typename Vec<VEC>::T;
    const int LC   = 1 << a.lc_log;
    const int LE   = 1 << a.le_log;
    const int L    = LC * LE;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x >> 6;
    const int gl   = lane & (L - 1);
    const int c    = gl & (LC - 1);
    const int e    = gl >> a.lc_log;
    // Column slices tied to XCDs as in the engine: workgroup g runs on XCD
    // g % 8, and with S slices XCDs s*8/S .. (s+1)*8/S - 1 compute columns
    // [s*SC, (s+1)*SC) of every row block, so each XCD's L2 holds 1/S of B.
    int rblk = blockIdx.x, slice = 0;
    if (a.slices > 1) {
        const int per = 8 / a.slices;
        const int x   = blockIdx.x & 7;
        rblk  = (blockIdx.x >> 3) * per + x % per;
        slice = x / per;
    }
    if (rblk >= a.nblocks) return;  // whole workgroup, before any barrier
    const int cbeg = slice * a.slice_cols;
    const int cend = min(a.N, cbeg + a.slice_cols);
    const int row  = (rblk * 4 + wave) * (kWave / L) + (lane >> (a.lc_log + a.le_log));
    const bool live = row < a.M;
    int start = 0, end = 0;
    if (live) {
        start = a.row_ptr[row];
        end   = a.row_ptr[row + 1];
    }
    // LONG_ROWS = false: the caller knows no row exceeds long_len.
    const bool is_long = LONG_ROWS && end - start > a.long_len;
    const int  g_end   = is_long ? start : end;
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.B), static_cast<short>(a.N * 4), a.K, kBufWord3);

    for (int n0 = cbeg; n0 < cend; n0 += LC * VEC) {
        const int  n    = lane_col<VEC>(n0 + c * VEC, cend);
        const bool col  = n0 + c * VEC < cend;
        VT acc;
        if constexpr (COOP) {
            acc = row_chunks_sum<VEC, U>(a, rb, start, g_end, lane & ~(L - 1), gl, e, L, LE, n * 4,
                                         L);
        } else {
            // FEW: lanes by the row; otherwise the stride is the wave's (500000 rows of 20
            // 1 - 5% less time).
            const int lanes = !FEW || g_end - start > a.few_len ? LE : 1 << a.few_log;
            acc = row_segment_sum<VEC, U>(a, rb, !FEW || e < lanes ? start + e : g_end, g_end, lanes,
                                          n * 4);
        }
        for (int m = LC; m < L; m <<= 1) acc = xor_add<VEC>(acc, m);
        if (live && !is_long && e == 0 && col) {
            store_vec<VEC>(a.C + static_cast<size_t>(row) * a.N + n, acc);
        }
    }

    if constexpr (!LONG_ROWS) return;
    // Long rows of this workgroup, one at a time with all four waves: wave w
    // takes the entries of lanes w*WE .. w*WE+WE-1 of every 4*WE (per-lane
    // loads) or every fourth 64-entry chunk (cooperative loads), and wave 0
    // adds the four waves' partials in wave order (deterministic).
    __shared__ int s_long_rows[4][kWave];
    __shared__ int s_long_cnt[4];
    __shared__ VT  s_part[4][kWave];
    const unsigned long long longs = __ballot(live && is_long && gl == 0);
    if (lane == 0) s_long_cnt[wave] = __popcll(longs);
    if (live && is_long && gl == 0) {
        s_long_rows[wave][__popcll(longs & ((1ull << lane) - 1))] = row;
    }
    __syncthreads();
    const int WE = kWave / LC;  // entry lanes per wave
    const int we = lane >> a.lc_log;
    for (int w2 = 0; w2 < 4; ++w2) {
        const int cnt = s_long_cnt[w2];
        for (int i = 0; i < cnt; ++i) {
            const int r  = s_long_rows[w2][i];
            const int rs = a.row_ptr[r];
            const int re = a.row_ptr[r + 1];
            for (int n0 = cbeg; n0 < cend; n0 += LC * VEC) {
                const int  n   = lane_col<VEC>(n0 + c * VEC, cend);
                const bool col = n0 + c * VEC < cend;
                VT acc;
                // One row at a time: four entries per lane in flight.
                if constexpr (COOP) {
                    acc = row_chunks_sum<VEC, 4>(a, rb, rs + wave * kWave, re, 0, lane, we, kWave,
                                                 WE, n * 4, 4 * kWave);
                } else {
                    acc = row_segment_sum<VEC, 4>(a, rb, rs + wave * WE + we, re, 4 * WE, n * 4);
                }
                for (int m = LC; m < kWave; m <<= 1) acc = xor_add<VEC>(acc, m);
                if (we == 0) s_part[wave][c] = acc;
                __syncthreads();
                if (wave == 0 && we == 0 && col) {
                    const VT sum = ((s_part[0][c] + s_part[1][c]) + s_part[2][c]) + s_part[3][c];
                    store_vec<VEC>(a.C + static_cast<size_t>(r) * a.N + n, sum);
                }
                __syncthreads();
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Launch helpers
// ---------------------------------------------------------------------------

Error ok() { return Error{}; }

Error fail(int status, std::string msg) { return Error{status, std::move(msg)}; }

Error from_hip(hipError_t e, const char* what) {
    if (e == hipSuccess) return ok();
    return fail(kHipError, std::string(what) + ": " + hipGetErrorString(e));
}

bool aligned(const void* p, size_t bytes) {
    return (reinterpret_cast<uintptr_t>(p) % bytes) == 0;
}

// Widest VEC (<= want, 4 when want == 0) that a row holds once.  Rows need no
// alignment beyond their floats (see Vec) and N need not be a multiple of VEC
// (see lane_col): one float per lane, which other widths took before, is bound
// by the 4x as many load instructions and lanes (MI355X, 20011 x 17001, 40 per
// row, N = 77: 119.2 -> 32.4 us, 0.25 TB/s -> 7.6 TB/s of gathered rows).
int pick_vec(int N, int want) {
    if (want == 0) want = 4;
    while (want > 1 && N < want) want >>= 1;
    return want;
}

// Threads of a launch.  HIP 7.0 takes a launch of 2^32 and more without an error
// and runs none or a part of it.
constexpr long kMaxThreads = 0xffffffffL;

Error check_threads(long grid, int threads) {
    if (grid * threads <= kMaxThreads) return ok();
    return fail(kUnsupported, "the launch would need 2^32 threads or more");
}

// Workgroups of nblocks row blocks in column slices (see the kernels).
long sliced_grid(long nblocks, int slices) {
    const int per = 8 / slices;
    return slices == 1 ? nblocks : (nblocks + per - 1) / per * 8;
}

// Most lane groups of a wave, whose ranges cut the rows into pieces that the owner of a
// row adds one by one.  On explicit partitions and merge-path parts a range has 8
// entries, or a row where rows are shorter (power-law 2048^2, N = 16 11.1 us with eight
// waves' reductions, 14.2 with 64 groups of 4 entries; parts of 2.5 per row, N = 272 18.7 us
// with groups of one row, 29.8 with one group).  Even rows of a few in a workgroup
// besides take no more than eight pieces a row: 823 rows of 147, N = 48 13.6 -> 6.3 us,
// 955 of 43, N = 64 8.3 -> 5.2.  Uneven rows of an implicit partition take what fits: there
// the groups share the long ones (over 700 power-law inputs 4% less time than with ranges
// of 8 entries).  Two are always taken: csr_rowblock_wide cuts nothing between them.
int most_groups(int M, double avg, long per_wave, int slices, bool even, bool partition) {
    if (!even && !partition) return kMaxGroups;
    long most = per_wave / std::clamp(std::lround(avg), 1L, 8L);
    if (even) most = std::min<long>(most, M / (slices == 1 ? 512 : 128));
    return static_cast<int>(std::clamp<long>(most, 2, kMaxGroups));
}

// Lane groups of a wave: with L = lanes of one row (slice) and p column passes
// a group takes ceil(L / p) lanes; the pass count with the fewest passes per
// entry slot (p / groups) wins, fewer passes first.  want: groups asked for.
// per_wave: entries of a wave.  More passes need 18 entries a group (1050 rows of 200,
// N = 160 15.2 us in two passes of 51 entries, 12.2 in one; 2100 of 100, N = 320 25.2
// and 23.4; 4096 of 60, 60 entries, 11.0 and 11.7), 40 on merge-path
// parts (power-law 2048^2, mean 64, N = 260 24.6 us in two passes, 29.1 in four; 8192^2,
// mean 40 50 against 36).  most: see most_groups.
void set_groups(RowblockArgs& a, int cols, int vec, int want, long per_wave, int most) {
    const int lanes = ceil_div(cols, vec);
    if (want == 1 || want == 2 || want == 4 || (want == 8 && vec == 4)) {
        a.groups      = want;
        a.group_lanes = kWave / want;
    } else {
        const bool split = a.part.split_rows != nullptr;
        int passes = ceil_div(lanes, kWave), best = passes;
        const auto groups_of = [&](int p) { return std::min(most, kWave / ceil_div(lanes, p)); };
        for (int p = passes + 1; p <= 2 * passes; ++p) {
            if (4 * p * groups_of(best) < 3 * best * groups_of(p) && per_wave >= (split ? 40 : 18) * groups_of(p)) {
                best = p;
            }
        }
        a.group_lanes = ceil_div(lanes, best);
        a.groups      = groups_of(best);
    }
    a.lanes_inv  = ceil_div(1 << 16, a.group_lanes);
    a.groups_inv = static_cast<unsigned>(
        std::min<unsigned long long>(0xffffffffull, ((1ull << 32) + a.groups - 1) / a.groups));
    a.window_log = 0;
    while ((2 << a.window_log) * a.groups <= kWCap) ++a.window_log;
}

template <int VEC, int WAVES, int U, bool SBUF, bool HALVES = false, bool FOLD = false>
hipError_t run_rowblock(const RowblockArgs& args, int grid, hipStream_t stream) {
    hipLaunchKernelGGL((csr_rowblock<VEC, WAVES, U, SBUF, HALVES, FOLD>), dim3(grid),
                       dim3(WAVES * kWave), 0, stream, args);
    return hipGetLastError();
}

// Merge-path ranges of eight groups and more fold their chains at every window's
// end: csr_rowblock_wide's form had as many interleaved chains there, and four
// over a whole range are up to 18% further from 64 bits (30000^2, 120 per row, N = 32
// 0.86e-7 of the norm, 1.01e-7 and, folded, 0.78e-7; 34.5 -> 35 us).  Fewer groups and
// shorter ranges need none.
bool fold_windows(const RowblockArgs& a) {
    return a.part.split_rows != nullptr && a.groups >= 8;
}

// Launch shapes: waves per workgroup (2, 4, 8) x entries in flight per group
// per step (4, 8).  B loads through a structured buffer unless B is too large
// for one (then only 8 waves x 4 is built).
template <int VEC>
hipError_t dispatch_shape(int waves, int unroll, bool sbuf, const RowblockArgs& args, int grid,
                          hipStream_t stream) {
    if (!sbuf) return run_rowblock<VEC, 8, 4, false>(args, grid, stream);
    if (waves == 4 && unroll == 4 && fold_windows(args)) {
        return run_rowblock<VEC, 4, 4, true, false, true>(args, grid, stream);
    }
    if (waves == 8) {
        return unroll == 8 ? run_rowblock<VEC, 8, 8, true>(args, grid, stream)
                           : run_rowblock<VEC, 8, 4, true>(args, grid, stream);
    }
    if (waves == 2) {
        return unroll == 8 ? run_rowblock<VEC, 2, 8, true>(args, grid, stream)
                           : run_rowblock<VEC, 2, 4, true>(args, grid, stream);
    }
    return unroll == 8 ? run_rowblock<VEC, 4, 8, true>(args, grid, stream)
                       : run_rowblock<VEC, 4, 4, true>(args, grid, stream);
}

template <bool HALVES>
hipError_t dispatch_wide(int waves, const RowblockArgs& args, int grid, hipStream_t stream) {
    const auto run = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(waves * kWave), 0, stream, args);
        return hipGetLastError();
    };
    if constexpr (!HALVES) {
        if (waves == 8) {
            return args.groups == 1 ? run(csr_rowblock_wide<1, 8, false>)
                                    : run(csr_rowblock_wide<2, 8, false>);
        }
    }
    return args.groups == 1 ? run(csr_rowblock_wide<1, 4, HALVES>)
                            : run(csr_rowblock_wide<2, 4, HALVES>);
}

// Rows whose lengths stay within twice the average (plus a constant for
// short rows): uniform random rows qualify, power-law rows do not.
bool rows_even(int M, long long nnz, int max_row) {
    return max_row > 0 && M > 0 &&
           max_row <= 2.0 * static_cast<double>(nnz) / M + 32.0;
}

// Column slices for a K x N fp32 B: the fewest (a power of two, at most 8) that
// bring one XCD's share of B down to its 4 MiB L2, each at least 32 columns
// wide (one 128-byte line of a B row); on rows of 16 entries and more, while
// slices stay 64 columns wide, down to half of the L2, which A and C pass
// through too.  Measured on MI355X over 70 uniform and power-law inputs with B
// of 8 .. 256 MiB, against slices of at least 64 columns: 65536^2, 32 per row,
// N = 256 252 -> 212 us; 32768^2, 32 per row, N = 128 46.7 -> 38.9 us; 8192^2, 100
// per row, N = 512 70 -> 64 us.  B of 4 MiB or less is fastest unsliced.  Slices
// that are no whole number of lines keep 64 columns: every one touches a line
// more (131072^2, 8 per row, N = 500: 414 us with 4 slices, 447 with 8; 65536^2, 32
// per row, N = 96 99 us whole, 131 with 2; N = 192 226 with 2, 263 with 4).
// wide: slices of at least 64 columns and none for the half of an L2.  For groups of
// a number asked for, whose lanes narrower slices would leave idle (8192^2, 82 per
// row, N = 256, one group: 50 us with two slices, 80 with four), and B past the
// buffer's 2 GiB, which no slice brings near an L2 (65536 x 2.2 M, 24 per row, N = 256
// 327 us with four, 361 with eight).
// On even rows and merge-path parts, whose one or two groups csr_rowblock_wide takes,
// slices whose columns fill those groups' lanes (128 and more) stay until a share is
// 3.75 MiB, others until 2.25 (merge-path parts of 192 columns 3.25): 5000^2, 300 per
// row, N = 256 58 us with four slices, 54 with two; 6000^2, 20 per row, N = 512 15.4 with
// eight, 13.9 with four; parts of 4200^2, 41 per row, N = 256 17.4 and 15.1; at 4 MiB
// four win (8192^2, 82 per row 31.7 with two, 30.4).  Uneven rows gain more by the finer
// ones (power-law 5000^2, N = 256 37.7 with two, 30.3).
// Slices of 32 columns and more that are no whole lines pay where they bring a share of
// 4.75 MiB and more to 5 (20000^2, 60 per row, N = 160 68.5 us with two, 61.4 with four;
// 14000^2, 4.3 MiB, 53.7 and 58.8), but not against whole rows (N = 96 of 24576^2 75 and 80).
int auto_slices(int K, int N, double avg_row, bool even, bool split, bool wide) {
    const long long b_bytes = static_cast<long long>(K) * N * 4;
    if (b_bytes <= (4LL << 20)) return 1;
    const auto narrowest = [&](int slices) { return !wide && N % (32 * slices) == 0 ? 32 : 64; };
    const auto over = [&](int slices, int quarter_mib) {  // an XCD's share of B
        return b_bytes > (static_cast<long long>(quarter_mib) << 18) * slices;
    };
    const auto half = [&](int slices) {
        if (!even && !split) return 8;
        if (N % (128 * slices) == 0) return 15;
        return split && N % (64 * slices) == 0 ? 13 : 9;
    };
    int s = 1;
    while (s < 8 && ((over(s, 16) && N / (2 * s) >= narrowest(2 * s)) ||
                     (!wide && over(s, half(s)) && N / (2 * s) >= 64 && avg_row >= 16.0))) {
        s *= 2;
    }
    if (!wide && s > 1 && s < 8 && N / (2 * s) >= 32 && over(s, 19) && !over(2 * s, 20)) s *= 2;
    return s;
}

// Waves of the engine resident at once on the chip: 16 per CU (four 4-wave
// workgroups) on 256 CUs.
constexpr long kRoundWaves = 4096;

// Rows per workgroup of the 4-wave row-block launch for even rows: the grid
// is a whole number of rounds of kRoundWaves waves, one round per ~2 M entry
// visits (nnz x slices, ~512 entries per wave).  A partial last round leaves
// CUs idle while it runs.  Measured on MI355X over uniform rows (M 2048 ..
// 32768, 8 .. 164 entries per row, N 64 .. 256), whole rounds gain up to
// 1.35x over ~160 entries per wave (1.2 - 1.6 rounds at M = 12288 .. 16384).
// Skewed rows need the many small workgroups of the default instead: a
// static one-round partition loses up to 1.5x on power-law rows.
int round_rows_per_block(int M, long long nnz, int slices, int waves) {
    const double visits = static_cast<double>(nnz) * slices;
    const long rounds = std::max(1L, std::lround(visits / (kRoundWaves * 512.0)));
    const long blocks = std::max(1L, rounds * kRoundWaves / (static_cast<long>(waves) * slices));
    return static_cast<int>(std::min<long>(kRpCap, std::max(1L, (M + blocks - 1) / blocks)));
}

// Rows per workgroup of csr_rowblock on even rows, near rpb: the grid is a whole
// number of rounds where it would be four or fewer.  512 workgroups of 8 waves fill the
// chip, and M / 512 rows, rounded down, make a few more of them: 4200 rows of 41, N =
// 160 12.9 -> 10.0 us, 5000 of 100 21.3 -> 16.8, 3000 of 200, N = 320 44.4 -> 34.9.  Rows that may
// be uneven only leave a second round that is not full, and only where a wave has
// under 32 entries (1000 uniform inputs of 64 K entries and fewer 0.86 -> 0.73 of the time
// of one group without it, as many power-law ones 0.72 -> 0.70); with more, the finer cut
// spreads the long rows (power-law 3100 of 100 16.0 us, 20.7 without).
int near_round_rows(int M, int rpb, int slices, int waves, bool even) {
    const double round = static_cast<double>(kRoundWaves) / waves / slices;  // row blocks
    const double rounds = ceil_div(M, rpb) / round;
    if (!even) return rounds > 1.0 && rounds < 2.0 ? static_cast<int>(std::ceil(M / round)) : rpb;
    if (rounds > 4.0) return rpb;
    return static_cast<int>(std::ceil(M / (std::max(1.0, std::round(rounds)) * round)));
}

// B rows as buffer records: the record stride field holds at most 16383
// bytes and the buffer's byte range must fit a signed 32-bit offset.
bool b_fits_buffer(int K, int N) {
    return static_cast<long long>(N) * 4 <= 16383 &&
           static_cast<long long>(K) * N * 4 <= 0x7fffffffLL;
}
}  // namespace

int default_partition_parts(int num_rows, int nnz) {
    // About 1280 nonzeros per workgroup (160 per wave of the default 8-wave
    // shape), at least two workgroups per CU and at most one per row.
    long parts = (static_cast<long>(nnz) + 1279) / 1280;
    parts = std::max<long>(parts, 512);
    parts = std::min<long>(parts, std::max(num_rows, 1));
    return static_cast<int>(std::max<long>(parts, 1));
}

namespace {

int pow2_log_at_least(int x) {
    int l = 0;
    while ((1 << l) < x && l < 6) ++l;
    return l;
}

// Column lanes (log2) of a row group: enough to cover N in one pass, at most
// 64; 32 or 64 drop to 16 (two or four column passes) while the matrix would
// still give >= 16384 waves.
constexpr long kRowGroupTargetWaves = 8192;
int row_group_lc_log(int M, int N, int vec) {
    int lc_log = pow2_log_at_least(ceil_div(N, vec));
    while (lc_log > 4 && N % 32 == 0 && (static_cast<long>(M) << lc_log) / kWave >= 2 * kRowGroupTargetWaves) {
        --lc_log;
    }
    return lc_log;
}

// XCD-tied column slices of the row groups: on rows of up to 24 entries with
// a B larger than one XCD's 4 MiB L2, the fewest slices (a power of two, at
// most 8, each at least 32 columns wide) that bring an XCD's share of B under
// 4 MiB (measured on MI355X: M = 16384, N = 256, 16 per row 28.4 -> 20.2 us
// with 4 slices; M = 32768, N = 128: 28.5 -> 25.0 us).  Longer rows keep one
// slice: every slice re-reads the rows' column indices, which then costs more
// than the L2 misses it saves.  Widths that are no whole lines take slices only
// where wide ones (64 columns, 48 from four slices on) do bring the share down,
// to 6 MiB: every slice touches a line more (M = 16384, 16 per row, N = 500 64 us
// with four slices, 54 with eight; N = 250 33 with two, 29 with four; M = 65536, N =
// 250 168 whole, 211 with two; N = 100 66 whole, 83 with two).
int row_group_slices(int K, int N, double avg_row) {
    if (avg_row > 24.0) return 1;
    const long long b_bytes = static_cast<long long>(K) * N * 4;
    int s = 1;
    if (N % 32 != 0) {
        while (s < 8 && b_bytes > (6LL << 20) * s) s *= 2;
        return b_bytes <= (6LL << 20) * s && N / s >= (s == 2 ? 64 : 48) ? s : 1;
    }
    while (s < 8 && b_bytes > (4LL << 20) * s && N / (2 * s) >= 32) s *= 2;
    return s;
}

template <int VEC, bool COOP, bool LONG_ROWS>
hipError_t run_row_groups(const RowGroupArgs& args, int unroll, int grid, hipStream_t stream) {
    if constexpr (!COOP) {
        if (args.few_len > 0) {
            hipLaunchKernelGGL((csr_row_groups<VEC, 2, false, LONG_ROWS, true>), dim3(grid),
                               dim3(256), 0, stream, args);
            return hipGetLastError();
        }
    }
    if (unroll == 4) {
        hipLaunchKernelGGL((csr_row_groups<VEC, 4, COOP, LONG_ROWS>), dim3(grid), dim3(256), 0,
                           stream, args);
    } else {
        hipLaunchKernelGGL((csr_row_groups<VEC, 2, COOP, LONG_ROWS>), dim3(grid), dim3(256), 0,
                           stream, args);
    }
    return hipGetLastError();
}

template <int VEC>
hipError_t run_row_groups(const RowGroupArgs& args, bool coop, bool long_rows, int unroll,
                          int grid, hipStream_t stream) {
    if (long_rows) {
        return coop ? run_row_groups<VEC, true, true>(args, unroll, grid, stream)
                    : run_row_groups<VEC, false, true>(args, unroll, grid, stream);
    }
    return coop ? run_row_groups<VEC, true, false>(args, unroll, grid, stream)
                : run_row_groups<VEC, false, false>(args, unroll, grid, stream);
}

// Whether rows take their entry lanes past the cap that keeps the grid near 8192
// waves.  Long rows of narrow B are bound by one 128-byte line per entry into the
// L1s (262144 rows of 24, N = 1: 6.3 M lines in 31 us, 26 TB/s, where gathers
// saturate), and a lane that walks much of a row alone also takes a line of
// col_idx and of values per step.  le_log: the capped lanes.  MI355X, capped
// against uncapped (M = K, uniform rows unless said):
//  - up to 2 column lanes from 10 entries per lane on (49152 rows of 80, N = 8 26.3
//    -> 21.8 us; 20000 of 60 at 7.5 per lane 13.3 -> 14.0), from 49152 rows on from 5
//    (98304 rows of 24, N = 1 13.3 -> 12.5; 262144 45.3 -> 30.6);
//  - at 4 from 11 (24576 rows of 80, N = 16 12.9 -> 12.3; of 40, 10 per lane, 7.6 -> 7.8);
//  - at 8 where B is past the L2s (65536 rows of 40, N = 32 37.0 -> 33.5; 49152 rows, a
//    B of 6 MiB, 21.1 -> 23.5), on rows of 128 and more (32768 of 160 39.1 -> 37.2),
//    and on uneven rows (power-law 32768 of 76 58 -> 39); without a longest-row
//    hint, which would tell, on rows of 64 and more of a B in an L2 (24576 of 80
//    16.0 -> 16.4);
//  - not from 16 column lanes on, nor on rows of under 20.
bool more_entry_lanes(int M, int K, int N, long long nnz, int max_row, int lc_log, int le_log) {
    const double avg = static_cast<double>(nnz) / M;
    const double per_lane = avg / (1 << le_log);
    if (avg < 20.0 || lc_log > 3) return false;
    if (lc_log <= 1) return per_lane >= (M >= 49152 ? 5.0 : 10.0);
    if (lc_log == 2) return per_lane >= 11.0;
    const long long b_bytes = static_cast<long long>(K) * N * 4;
    if (avg >= 128.0 || b_bytes >= (8LL << 20)) return true;
    return max_row > 0 ? !rows_even(M, nnz, max_row) : avg >= 64.0 && b_bytes <= (4LL << 20);
}

// Shape of the sub-wave row groups, measured on MI355X over uniform rows of
// 1 .. 300 entries, M = 2048 .. 65536 and N = 1 .. 256:
//  - column lanes cover N in one pass (up to 64 lanes), except that 32 or 64
//    column lanes drop to 16 (two or four passes) where N is whole 128-byte
//    lines and the matrix still gives >= 16384 waves (M = 32768, N = 128: 96 -> 89
//    us; at other widths every pass would touch a line more);
//  - entry lanes ~1.5 * sqrt(average row) as a power of two, but no more than
//    keep the grid near 8192 waves (32 per CU): beyond that, more rows per wave
//    beat more lanes per row -- except on the rows of more_entry_lanes;
//  - 4 entries per entry lane per iteration on those, and from 32 entries per
//    row on while B is at most 2 MiB (latency-bound: few, long rows), else 2 -- with B
//    beyond one XCD's L2, fewer gathers in flight keep more of it cached
//    (M = 32768, N = 128, 82 entries per row: 123 -> 88 us);
//  - the cooperative loads (one column/value load per L entries, handed out
//    by shuffles) from 4 column lanes on when rows average >= 32 entries or
//    column lanes x rows >= 2^18: redundant per-lane index loads then cost
//    more than the shuffles (M = 8192, N = 64, 82 per row: 11.4 -> 9.1 us;
//    M = 32768, N = 128: 119 -> 87 us); on short rows of a smaller matrix the
//    per-lane loads are 5-15% ahead.
// row_groups: 1 picks the load form by that rule, 2 forces per-lane loads,
// 3 forces the cooperative loads.
Error launch_row_groups(const CSR& A, const float* B, float* C, int N, hipStream_t stream,
                        int vec, const EngineOpts& o) {
    constexpr long kTargetWaves = kRowGroupTargetWaves;
    const int M = A.num_rows;
    const double avg = A.nnz > 0 ? static_cast<double>(A.nnz) / M : 0.0;
    int slices = o.slices;
    if (slices == 0) slices = row_group_slices(A.num_cols, N, avg);
    if (slices != 1 && slices != 2 && slices != 4 && slices != 8) slices = 1;
    const int slice_cols = ceil_div(ceil_div(N, slices), vec) * vec;
    const int lc_log = row_group_lc_log(M, slice_cols, vec);
    int le_log, few_log = 0, few_len = 0;
    bool more = false;
    if (o.entry_lanes != 0) {
        if (o.entry_lanes < 0 || o.entry_lanes > 64 || (o.entry_lanes & (o.entry_lanes - 1)) != 0) {
            return fail(kInvalid, "entry_lanes must be a power of two up to 64");
        }
        le_log = pow2_log_at_least(o.entry_lanes);
    } else {
        // Lanes by row length; fewer suffice at 4 column lanes and more.
        const auto lanes_for = [&](double factor) {
            return static_cast<int>(std::lround(std::log2(factor * std::sqrt(std::max(avg, 1.0)))));
        };
        const long cap =
            kTargetWaves * kWave / std::max(1L, (static_cast<long>(M) << lc_log) * slices);
        int cap_log = 0;
        while ((2L << cap_log) <= cap) ++cap_log;
        le_log = std::max(0, std::min(lanes_for(1.5), cap_log));
        const int long_log = std::min(lanes_for(lc_log >= 2 ? 1.0 : 1.5), 6 - lc_log);
        more = long_log > le_log &&
               more_entry_lanes(M, A.num_cols, N, A.nnz, o.max_row_hint, lc_log, le_log);
        if (more) le_log = long_log;
        // Rows that may be uneven, up to 16 columns: eight lanes while that is under 2048
        // waves, for the long rows of a nearly empty chip (power-law 2544 of 2.7, N = 6
        // 5.5 -> 3.3 us; over 1234 power-law inputs 0.84 -> 0.76 of one float a lane, uniform
        // ones 0.81 -> 0.80; rows known to be even 1.00).  Rows of two entries a lane and
        // fewer keep the lanes they had: each lane rounds its first product, so with
        // eight a row of 3 to 10 would be 4 - 10% further from 64 bits.
        int spare = 3;
        while (spare > 0 && (static_cast<long>(M) << (lc_log + spare)) * slices > kWave * 2048L) --spare;
        if (lc_log <= 2 && avg < 32.0 && o.unroll == 0 && o.row_groups != 3 && spare > le_log && !rows_even(M, A.nnz, o.max_row_hint)) {
            few_log = le_log;
            few_len = 2 << spare;
            le_log  = spare;
        }
    }
    le_log = std::max(0, std::min(le_log, 6 - lc_log));
    const bool b_small = static_cast<long long>(A.num_cols) * N * 4 <= (2LL << 20);
    const int unroll = (o.unroll == 2 || o.unroll == 4) ? o.unroll
                                                        : (more || (avg >= 32.0 && b_small) ? 4 : 2);
    bool coop;
    if (o.row_groups == 2) coop = false;
    else if (o.row_groups == 3) coop = true;
    else coop = lc_log >= 2 && (avg >= 32.0 || (static_cast<long>(M) << lc_log) >= (1L << 18));
    // Entry lanes that no cap holds down may be more than a launch has threads
    // for (17 M rows of 20, N = 132 in eight slices of five column lanes).
    const auto blocks_of = [&](int le) { return ceil_div(M, 4 * (kWave >> (lc_log + le))); };
    while (o.entry_lanes == 0 && le_log > 0 &&
           sliced_grid(blocks_of(le_log), slices) * 256 > kMaxThreads) {
        --le_log;
    }
    const int nblocks = blocks_of(le_log);
    if (Error e = check_threads(sliced_grid(nblocks, slices), 256); e.status != kOk) return e;
    const int grid = static_cast<int>(sliced_grid(nblocks, slices));
    const int long_len = std::max(8 << le_log << (unroll == 4 ? 2 : 1),
                                  static_cast<int>(std::ceil(std::min(4.0 * avg, 1.0e9))));
    RowGroupArgs args{A.row_ptr, A.col_idx,  A.values,   B,          C,
                      M,         N,          A.num_cols, lc_log,     le_log,
                      long_len,  slices,     slice_cols, nblocks,    few_log,
                      few_len};
    // Without a longest-row hint any row may be long: the workgroup-wide pass
    // (one barrier even when no row needs it) is compiled in.
    const bool long_rows = o.max_row_hint <= 0 || o.max_row_hint > long_len;
    hipError_t e;
    if (vec == 4) e = run_row_groups<4>(args, coop, long_rows, unroll, grid, stream);
    else if (vec == 2) e = run_row_groups<2>(args, coop, long_rows, unroll, grid, stream);
    else e = run_row_groups<1>(args, coop, long_rows, unroll, grid, stream);
    return from_hip(e, "csr row groups launch");
}

// Column lanes: the fewest (a power of two, at most 64) that cover N; wider N in
// column tiles of 256, a workgroup each.  Rows past a launch's threads (67 M at 64
// lanes) go into further launches.
// A whole wave takes each row at up to 8 columns where the rows are few and hold
// 16 entries and more: the chip is nearly empty then, one row's chain is the whole
// time, and the wave has its entries and 16 B rows in flight where a lane or two
// waits for 8 entries and then for their B rows.  1000 rows of 451, N = 1 90 -> 20
// us, N = 8 88 -> 24; 2048 rows of 63 14.6 -> 6.1 and 13.8 -> 8.1; 4096 rows of 157
// 35.2 -> 13.9 and 30.8 -> 24.6.  Past that many rows the waves are what is waited
// for: 8192 rows of 82, N = 3 17.2 -> 24.2, but N = 1 19.2 -> 13.4 still.  4096 rows
// of 2, N = 8 3.0 -> 4.6.
bool wave_a_row(int M, int nnz, int N) {
    const double avg = static_cast<double>(nnz) / M;
    return N <= 8 && avg >= 16.0 && M <= (N == 1 ? 8192 : avg >= 128.0 ? 5120 : 4096);
}

Error launch_in_order(const CSR& A, const float* B, float* C, int N, hipStream_t stream) {
    const int  vec    = pick_vec(N, 0);
    const bool wave   = wave_a_row(A.num_rows, A.nnz, N);
    const int  lc_log = wave ? 6 : pow2_log_at_least(ceil_div(N, vec));
    const int  per_wg = 4 * (kWave >> lc_log);
    const long most   = kMaxThreads / 256 * per_wg;
    for (long first = 0; first < A.num_rows; first += most) {
        const int  rows = static_cast<int>(std::min(most, A.num_rows - first));
        const dim3 grid(ceil_div(rows, per_wg), std::min(ceil_div(N, vec << lc_log), 65535));
        const auto run = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, rows, N, lc_log,
                               A.row_ptr + first, A.col_idx, A.values, B,
                               C + static_cast<size_t>(first) * N);
            return from_hip(hipGetLastError(), "csr in-order launch");
        };
        const Error e = vec == 1      ? run(wave ? csr_rows_in_order<1, Hand::Readlane>
                                                 : csr_rows_in_order<1, Hand::Direct>)
                        : vec == 2    ? run(wave ? csr_rows_in_order<2, Hand::Readlane>
                                                 : csr_rows_in_order<2, Hand::Direct>)
                        : lc_log == 6 ? run(csr_rows_in_order<4, Hand::Readlane>)
                        : lc_log >= 3 ? run(csr_rows_in_order<4, Hand::Shuffle>)
                                      : run(csr_rows_in_order<4, Hand::Direct>);
        if (e.status != kOk) return e;
    }
    return ok();
}

Error launch_csr_impl(CsrRole role, const CSR& A, const float* B, float* C, int N,
                      hipStream_t stream, const int* bounds, int parts, const EngineOpts* opts,
                      const SplitPlan* split) {
    if (A.num_rows < 0 || A.num_cols < 0 || A.nnz < 0 || N < 0) {
        return fail(kInvalid, "negative matrix dimension");
    }
    if (A.num_rows == 0 || N == 0) return ok();
    if (A.row_ptr == nullptr || B == nullptr || C == nullptr) {
        return fail(kInvalid, "null device pointer");
    }
    if (A.nnz > 0 && (A.col_idx == nullptr || A.values == nullptr)) {
        return fail(kInvalid, "null device pointer");
    }
    if (bounds != nullptr && parts < 1) return fail(kInvalid, "partition needs parts >= 1");

    const int M = A.num_rows;
    if (role == CsrRole::Baseline || role == CsrRole::Memopt || role == CsrRole::MemoptV2) {
        return launch_in_order(A, B, C, N, stream);
    }

    EngineOpts o = opts ? *opts : EngineOpts{};
    int want_vec = o.vec;
    int want_groups = o.groups;
    if (role == CsrRole::Tiled && want_vec == 0) {
        want_vec = 1;  // one lane per column, 64 columns per pass
        if (want_groups == 0) want_groups = 1;
    }
    if ((role == CsrRole::TiledV2 || role == CsrRole::TiledV4) && want_vec == 0) want_vec = 4;
    if (role == CsrRole::TiledV2) {
        if (N % 128 != 0) {
            return fail(kUnsupported, "spmm_tiled_v2 requires N % 128 == 0 (got N=" +
                                          std::to_string(N) + ")");
        }
        if (!aligned(B, 16) || !aligned(C, 16)) {
            return fail(kUnsupported, "spmm_tiled_v2 requires 16-byte aligned B and C");
        }
    }
    if (want_vec != 0 && want_vec != 1 && want_vec != 2 && want_vec != 4) {
        return fail(kInvalid, "engine vec must be 1, 2 or 4");
    }
    const int vec = pick_vec(N, want_vec);
    // Default launches of the production roles at N of a few columns (at most
    // four column lanes of VEC floats, e.g. N <= 16 with 16-byte lanes) take
    // the sub-wave row groups: the engine keeps half or more of its lanes idle
    // there, and with 64 .. 256 entry lanes the row groups' workgroup-wide
    // pass shares a long row among many lanes.  Measured on MI355X without
    // row-length knowledge: 1.6 - 3.4x faster on uniform rows at N <= 8 and
    // 2.5 - 3.6x on power-law rows of up to 4096 entries; at N = 12 - 16 over
    // 32 uniform and power-law inputs (M 2048 .. 65536) 2.0x on average, never
    // slower (1.18x at worst).  At five to eight lanes (N <= 32) they win 1.07 -
    // 1.75x on the inputs of up to 2.5 M nonzeros.  Past 4 M the engine stays: of
    // larger inputs the row groups take some in less (20000 rows of 298, N = 32 36
    // against 60 us; power-law 30000 of 147 51 against 64), others in more (65536 of
    // 80, N = 20 62 against 60; 300000 of 16 97 against 95; power-law 131072 of 39
    // 96 against 92), and no rule on sizes parts them yet.  Any explicit engine option keeps the
    // engine, and so does a longest-row hint: a caller that knows its rows
    // (spmm_hybrid_run) chooses the form itself.
    const bool engine_defaults = o.vec == 0 && o.waves == 0 && o.unroll == 0 &&
                                 o.rows_per_block == 0 && o.groups == 0 && o.slices == 0 &&
                                 o.global_loads == 0 && o.entry_lanes == 0 &&
                                 o.max_row_hint == 0;
    if (o.row_groups == 0 && engine_defaults && bounds == nullptr && split == nullptr &&
        (role == CsrRole::TiledV3 || role == CsrRole::TiledV4) &&
        b_fits_buffer(A.num_cols, N) &&
        (pow2_log_at_least(ceil_div(N, vec)) <= 2 ||
         (pow2_log_at_least(ceil_div(N, vec)) <= 3 && A.nnz <= (1 << 22)))) {
        EngineOpts rg = o;
        rg.row_groups = 1;
        return launch_row_groups(A, B, C, N, stream, vec, rg);
    }
    if (o.row_groups != 0) {
        if (o.row_groups < 0 || o.row_groups > 3) {
            return fail(kInvalid, "row_groups must be 0 (engine), 1 (auto), 2 or 3");
        }
        if (bounds != nullptr || split != nullptr) {
            return fail(kInvalid, "row groups take no explicit partition");
        }
        if (!b_fits_buffer(A.num_cols, N)) {
            return fail(kUnsupported, "row groups need N <= 4095 and B within 2 GiB");
        }
        return launch_row_groups(A, B, C, N, stream, vec, o);
    }
    const double avg = A.nnz > 0 ? static_cast<double>(A.nnz) / M : 1.0;
    // Column slices (XCD-aware, see the kernel): 1, 2, 4 or 8.
    int slices = o.slices;
    const bool sbuf = o.global_loads == 0 && b_fits_buffer(A.num_cols, N);
    if (slices == 0) {
        slices = role == CsrRole::Tiled
                     ? 1
                     : auto_slices(A.num_cols, N, avg, rows_even(M, A.nnz, o.max_row_hint),
                                   split != nullptr, want_groups != 0 || !sbuf);
    }
    if (slices != 1 && slices != 2 && slices != 4 && slices != 8) slices = 1;
    int slice_cols = ceil_div(N, slices);
    slice_cols = ceil_div(slice_cols, vec) * vec;
    // Defaults measured on MI355X (uniform and power-law sweeps): 8 waves per
    // workgroup without column slices (a workgroup's nonzeros are split over
    // its waves, so a long row is shared by eight: power-law 2048^2, N = 128 9.5
    // us with 8, 12.1 with 4), 4 with them (more workgroups per row block) and
    // on merge-path parts, except csr_rowblock_wide's without slices (8, see
    // wg_waves); 4 rows in flight per group; about 160 nonzeros per
    // wave and at least 512 row blocks (256 with slices) when the matrix allows
    // it: many small workgroups keep skewed rows balanced.  Rows known to be
    // even (max_row_hint): the whole-round grid of 4-wave workgroups.
    const int unroll = o.unroll == 8 ? 8 : 4;

    RowblockArgs args{};
    RowblockPart& part = args.part;
    part = RowblockPart{A.row_ptr, A.col_idx, A.values, B, C};
    part.K          = A.num_cols;
    args.M          = M;
    args.N          = N;
    args.slices     = slices;
    args.slice_cols = slice_cols;
    const long per_wave = split != nullptr    ? A.nnz / (4L * split->parts)
                          : bounds != nullptr ? A.nnz / (8L * parts)
                                              : std::min(160L, A.nnz / (slices == 1 ? 8L * 512 : 4L * 256));
    if (split != nullptr) {
        part.split_rows = split->rows;
        part.carry      = split->carry;
        part.nnz        = A.nnz;
        part.nblocks    = split->parts;
    }
    args.bounds = split == nullptr ? bounds : nullptr;
    const bool even_rows = split == nullptr && bounds == nullptr && o.rows_per_block <= 0 &&
                           rows_even(M, A.nnz, o.max_row_hint);
    set_groups(args, slice_cols, vec, want_groups, per_wave,
               most_groups(M, avg, per_wave, slices, even_rows, split != nullptr || bounds != nullptr));
    // The whole-round grid is for few groups: it leaves more of them too few
    // row pieces each (65536^2, 40 per row, N = 256, eight slices of four groups:
    // 305 us with it, 260 without).
    const bool even = even_rows && args.groups <= 2;
    const int waves = (o.waves == 2 || o.waves == 4 || o.waves == 8) ? o.waves
                      : even || slices > 1 || split != nullptr       ? 4
                                                                     : 8;
    if (args.bounds != nullptr) {
        part.nblocks = parts;
    } else if (split == nullptr) {
        int rpb = o.rows_per_block;
        if (rpb <= 0 && even) {
            rpb = round_rows_per_block(M, A.nnz, slices, waves);
        } else if (rpb <= 0) {
            rpb = static_cast<int>(160.0 * waves / std::max(avg, 1.0) + 0.5);
            rpb = std::min(rpb, M / (slices == 1 ? 512 : 256));
            if (rpb > 0 && (even_rows || (vec > 1 && per_wave < 32))) {
                rpb = near_round_rows(M, rpb, slices, waves, even_rows);
            }
        }
        rpb = std::max(1, std::min(rpb, kRpCap));
        // 160 entries per wave in eight slices are more threads than a launch
        // has from 1.3 G entries on.
        while (o.rows_per_block <= 0 && rpb < kRpCap &&
               sliced_grid(ceil_div(M, rpb), slices) * (waves * kWave) > kMaxThreads) {
            rpb = std::min(2 * rpb, kRpCap);
        }
        args.rows_per_block = rpb;
        part.nblocks = ceil_div(M, rpb);
    }
    const bool balanced = even || split != nullptr;
    const bool wide = balanced && sbuf && vec == 4 && args.groups <= 2 && o.groups == 0 &&
                      o.waves == 0 && o.unroll == 0;
    const int wg_waves = !sbuf ? 8 : wide ? (even || slices > 1 ? 4 : 8) : waves;
    if (Error t = check_threads(sliced_grid(part.nblocks, slices), wg_waves * kWave); t.status != kOk) {
        return t;
    }
    const int grid = static_cast<int>(sliced_grid(part.nblocks, slices));
    hipError_t e;
    if (wide) {
        e = dispatch_wide<false>(wg_waves, args, grid, stream);
    } else if (vec == 4) {
        e = dispatch_shape<4>(waves, unroll, sbuf, args, grid, stream);
    } else if (vec == 2) {
        e = dispatch_shape<2>(waves, unroll, sbuf, args, grid, stream);
    } else {
        e = dispatch_shape<1>(waves, unroll, sbuf, args, grid, stream);
    }
    if (e == hipSuccess && split != nullptr) {
        hipLaunchKernelGGL(csr_split_fixup, dim3(split->parts), dim3(64), 0, stream, A.row_ptr,
                           split->rows, split->carry, C, M, N, static_cast<long long>(A.nnz),
                           split->parts);
        e = hipGetLastError();
    }
    return from_hip(e, "csr engine launch");
}

}  // namespace

Error launch_csr(CsrRole role, const CSR& A, const float* B, float* C, int N,
                 hipStream_t stream, const int* bounds, int parts, const EngineOpts* opts) {
    return launch_csr_impl(role, A, B, C, N, stream, bounds, parts, opts, nullptr);
}

int split_partition_parts(int nnz) {
    // Two workgroups per CU: measured on MI355X over power-law inputs of 0.6 M
    // to 2.5 M nonzeros, 256 .. 1536 parts are within 10% of each other and
    // 4096 parts lose 15-40% to per-workgroup set-up and the fix-up; more
    // parts only for very large inputs (at most 64 K nonzeros per part).
    long parts = std::max<long>(512, (static_cast<long>(nnz) + 65535) / 65536);
    return static_cast<int>(std::min<long>(parts, std::max(nnz, 1)));
}

bool split_pays(int max_row_nnz) {
    // A row longer than four workgroups' share (4 x 640 nonzeros at 4 waves
    // of 160) keeps one row-partitioned workgroup busy long after the others:
    // then the merge-path partition wins (power-law 8192^2: 32 -> 23 us;
    // 16384^2 with two column slices: 88 -> 69 us); on rows of similar length
    // it costs its second launch (5-50%).
    return max_row_nnz > 4 * 640;
}

bool row_groups_pay(int M, int N, int K, double avg_row, int max_row) {
    // Measured on MI355X against the row-block engine as the hybrid runs it
    // (uniform rows of 8 .. 300 entries, M = 1024 .. 32768, N = 64 .. 256,
    // the engine with the longest row as its hint; power-law rows capped at
    // 512 / 4096).  Row groups win 1.5 - 4x for N <= 32 and 1.1 - 1.7x for
    // N = 64 (not on 1024 rows of > 100 entries, 0.75 - 0.9x).  Above
    // N = 64 they win on short rows (N x average <= 4096), on rows of up to 24
    // entries of a B past an L2, and at N = 128 on >= 4096 rows (1.03 - 1.6x) or >= 2048
    // rows of up to 10600 / N entries -- except at 4097 .. 8192 rows of
    // >= 64 entries, where the engine's whole-round grid holds 1 - 2 rows
    // per wave and matches or beats them (0.97 - 1.00x).  Those wins need
    // even rows: power-law rows of mean 164 capped at 512 run 0.6 - 0.7x.
    // With this rule the mean loss to the faster form over the sweep is
    // 0.14% (worst 5.6%).  A row longer than both 16384 / column-lanes
    // entries and 8x the average would keep one workgroup busy far longer
    // than the rest (more than ~16 iterations of its workgroup-wide pass):
    // then the engine, which shares long rows between eight waves with more
    // entries per step, is the safer choice.
    if (N <= 0 || M <= 0 || !b_fits_buffer(K, N)) return false;
    const int vec    = pick_vec(N, 0);
    const int slices = row_group_slices(K, N, avg_row);
    const int lc     = 1 << row_group_lc_log(M, ceil_div(ceil_div(N, slices), vec) * vec, vec);
    if (max_row > std::max(16384.0 / lc, 8.0 * avg_row)) return false;
    // A B past the L2s whose rows are whole lines: the engine's slices of 32
    // columns beat the row groups on longer rows (65536^2, 40 per row, N = 64 61
    // against 72 us, N = 128 120 against 155 us; 32768^2, 40 per row, N = 256 94
    // against 131 us) and from rows of 8 on once B is far larger (47000 x 110000, 2 per
    // row, N = 128 13 us in row groups, 14.7).  Other widths
    // cannot be cut that narrow, and there the row groups win on even rows
    // (24576^2, 100 per row, N = 100 65 against 99 us; over 90 inputs with N = 33
    // .. 250 they lose at most 3%, and at N = 250 on rows of 24 and fewer 15%), but
    // not on few (2320 x 6134, 101 per row, N = 180 22.3 us, 12.8 in the engine).
    const double b_mib = static_cast<double>(K) * N / (1 << 18);
    const bool lines = N % (N <= 128 ? 64 : 32) == 0;  // N = 96 has no halves of whole lines
    // Narrow B and rows just too short for more_entry_lanes, on many rows with a B
    // past the L2s (or so many that the lines of A alone bound a lane per row):
    // 262144 x 400000, 17 per row, N = 8 90 against 66 us, 500000 x 131072, N = 1 72
    // against 62; 131072 x 400000, N = 4 26.5 against 30.4, 262144 x 131072, N = 4 34
    // against 49, 20000 x 131072, N = 1 3.8 against 7.4 (over 180 shapes of 16 to 19 per
    // row; longer rows: 262144^2, 24 per row, N = 1 31 against 42, N = 16 97 against 95).
    if (N <= 32 && avg_row >= 16.0 && avg_row < 20.0 &&
        ((M >= 131072 && b_mib > 4.0 && b_mib * M >= 8.0 * 131072) || (M >= 400000 && K > 65536))) {
        return false;
    }
    if (lines && N > 32 && N <= 64 && b_mib >= 16.0 && avg_row >= 16.0) return false;
    if (lines && N > 64 && b_mib > 4.0 &&
        (avg_row >= (N > 128 ? 16.0 : 24.0) || (N <= 128 && b_mib >= 32.0 && avg_row >= 8.0))) {
        return false;
    }
    // Few long rows: at N <= 32 the row groups take 0.55 - 0.8 of the engine's time (1650
    // inputs of 60 .. 2100 rows of 60 .. 900), at 33 .. 64 0.9 - 1.2.
    if (N <= 64) return N <= 32 || M >= 2048 || avg_row <= 100.0;
    const bool b_large = avg_row <= 24.0 && b_mib > 4.0 && N >= (N % 32 == 0 ? 64 : 128);
    if (N * avg_row <= 2048.0 || (N <= 256 && b_large)) return true;
    if (max_row > 2.0 * avg_row + 32.0) return false;  // uneven rows
    if (!lines && N <= 256 && b_mib > 4.0 && M >= 4096) return true;
    if (N * avg_row <= 4096.0) return true;
    if (N > 128) return false;
    if (M > 4096 && M <= 8192 && avg_row >= 64.0) return false;
    return M >= 4096 || (M >= 2048 && N * avg_row <= 10600.0);
}

Error launch_csr_split(const CSR& A, const float* B, float* C, int N, hipStream_t stream,
                       const SplitPlan& plan, const EngineOpts* opts) {
    if (plan.parts < 1 || plan.rows == nullptr) {
        return fail(kInvalid, "split partition needs parts >= 1 and its row table");
    }
    if (plan.parts > std::max(A.nnz, 1)) {
        // an empty part would break the fix-up's runs of continuation parts
        return fail(kInvalid, "split partition needs parts <= max(nnz, 1) (got parts=" +
                                  std::to_string(plan.parts) + ", nnz=" +
                                  std::to_string(A.nnz) + ")");
    }
    if (plan.carry == nullptr && N > 0 && A.num_rows > 0) {
        return fail(kInvalid, "split partition needs a carry workspace of parts x N floats");
    }
    return launch_csr_impl(CsrRole::TiledV3, A, B, C, N, stream, nullptr, 0, opts, &plan);
}

bool khalf_pays(int K, int N) {
    // B over one XCD's 4 MiB L2 at full width, its half of the rows within it.
    // Measured on MI355X on c5 (16384^2 power-law, N = 128, B 8 MiB): the
    // merge-path engine 64.0 -> 53.9 us with each half's B rows resident in
    // its four XCDs' L2s, the fix-up 4.7 -> 6.5 us (it now also adds the
    // second half's partial C), 67.7 -> 60.1 us per launch.
    const long long row_bytes = static_cast<long long>(N) * 4;
    return N > 0 && N % 4 == 0 && K >= 2 && b_fits_buffer(K, N) &&
           static_cast<long long>(K) * row_bytes > (4LL << 20) &&
           static_cast<long long>((K + 1) / 2) * row_bytes <= (4LL << 20);
}

Error launch_csr_khalf(const KHalfPlan& p, const float* B, float* C, hipStream_t stream) {
    if (p.M < 0 || p.N < 0) return fail(kInvalid, "negative matrix dimension");
    if (p.M == 0 || p.N == 0) return ok();
    if (B == nullptr || C == nullptr || p.partial == nullptr || p.runs == nullptr) {
        return fail(kInvalid, "null device pointer");
    }
    if (p.N % 4 != 0 || !aligned(B, 16) || !aligned(C, 16)) {
        return fail(kUnsupported, "B-row halves need N % 4 == 0 and 16-byte aligned B and C");
    }
    for (int h = 0; h < 2; ++h) {
        if (p.parts[h] < 1 || p.parts[h] > std::max(p.half[h].nnz, 1) || p.rows[h] == nullptr ||
            p.carry[h] == nullptr) {
            return fail(kInvalid, "B-row halves: incomplete plan");
        }
    }
    const int N = p.N;
    RowblockArgs args{};
    for (int h = 0; h < 2; ++h) {
        RowblockPart& part = h == 0 ? args.part : args.upper;
        part = RowblockPart{p.half[h].row_ptr, p.half[h].col_idx, p.half[h].values,
                            h == 0 ? B : B + static_cast<size_t>(p.K0) * N,
                            h == 0 ? C : p.partial};
        part.split_rows = p.rows[h];
        part.carry      = p.carry[h];
        part.nnz        = p.half[h].nnz;
        part.K          = h == 0 ? p.K0 : p.K - p.K0;
        part.nblocks    = p.parts[h];
    }
    args.M          = p.M;
    args.N          = N;
    args.slice_cols = N;
    const long per_wave = std::min(args.part.nnz / p.parts[0], args.upper.nnz / p.parts[1]) / 4;
    set_groups(args, N, 4, 0, per_wave, static_cast<int>(std::clamp<long>(per_wave / 8, 1, kMaxGroups)));
    const int grid   = 8 * ceil_div(std::max(p.parts[0], p.parts[1]), 4);
    hipError_t e = args.groups <= 2 ? dispatch_wide<true>(4, args, grid, stream)
                   : fold_windows(args)
                       ? run_rowblock<4, 4, 4, true, true, true>(args, grid, stream)
                       : run_rowblock<4, 4, 4, true, true>(args, grid, stream);
    if (e == hipSuccess) {
        const long long chunks = static_cast<long long>(p.M) * N / 4;
        hipLaunchKernelGGL(csr_khalf_fixup, dim3(static_cast<unsigned>((chunks + 255) / 256)),
                           dim3(256), 0, stream, C, p.partial, p.carry[0], p.carry[1],
                           reinterpret_cast<const int4*>(p.runs), N, chunks);
        e = hipGetLastError();
    }
    return from_hip(e, "csr B-row halves launch");
}

}  // namespace engine
}  // namespace spmm
