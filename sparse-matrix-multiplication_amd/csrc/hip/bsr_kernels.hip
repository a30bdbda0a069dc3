// BSR (16x16 fp16 blocks) x dense fp16 B on gfx950 matrix cores, and the
// fp32 -> fp16 conversion (roles of spmm_wmma and float_to_half,
// spmm_wmma.cu:18-23 and :49-117).
//
// MFMA operand layout used (v_mfma_f32_16x16x32_f16, wave64, lane = 16*g + t):
//   A operand: lane holds A[t][kmap(g, 0..7)]       (8 fp16)
//   B operand: lane holds B[kmap(g, 0..7)][t]       (8 fp16)
//   D        : lane holds D[4*g + i][t], i = 0..3   (4 fp32)
// kmap(g, i) = 8*g + i.  The contraction only needs A and B to use the same
// kmap, so blocks pair up as: g = 0,1 -> block b (its columns 8*g .. 8*g+7),
// g = 2,3 -> block b+1.
//
// B is K-contiguous in the operand but N-contiguous in memory, so each wave
// stages the 32 B rows of a block pair (its 16*J columns) in LDS with plain
// 16-byte row loads and reads the operand back column-wise.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <initializer_list>
#include <type_traits>

#include "amdgcn.h"
#include "engine.h"
#include "spmm/utils.h"

namespace spmm {
namespace engine {

namespace {

using namespace dev;  // vector types, buffer loads, waits, barriers (amdgcn.h)

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// fp32 -> fp16 (round to nearest even), 8 elements per lane on the aligned body.
__global__ __launch_bounds__(256) void f32_to_f16_kernel(const float* __restrict__ src,
                                                         _Float16* __restrict__ dst, long n,
                                                         int vector_ok) {
    const long tid = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (vector_ok) {
        const long i = tid * 8;
        if (i + 8 <= n) {
            const f32x4 lo = *reinterpret_cast<const f32x4*>(src + i);
            const f32x4 hi = *reinterpret_cast<const f32x4*>(src + i + 4);
            f16x8 h;
            h[0] = static_cast<_Float16>(lo[0]);
            h[1] = static_cast<_Float16>(lo[1]);
            h[2] = static_cast<_Float16>(lo[2]);
            h[3] = static_cast<_Float16>(lo[3]);
            h[4] = static_cast<_Float16>(hi[0]);
            h[5] = static_cast<_Float16>(hi[1]);
            h[6] = static_cast<_Float16>(hi[2]);
            h[7] = static_cast<_Float16>(hi[3]);
            *reinterpret_cast<f16x8*>(dst + i) = h;
        } else {
            for (long e = i; e < n; ++e) dst[e] = static_cast<_Float16>(src[e]);
        }
    } else if (tid < n) {
        dst[tid] = static_cast<_Float16>(src[tid]);
    }
}

// C is written once and not read back by the kernel: streaming stores keep
// it from displacing A and B in L2 (measured on c4: 7.8 -> 7.5 us).
__device__ __forceinline__ void store_c(float* p, float v) { __builtin_nontemporal_store(v, p); }

// The record kernel stores its 16-byte C row chunks with device scope
// (kStoreDevice, the sc1 bit).  Measured on MI355X against streaming stores of
// the same chunks (A/B over three rounds, results bit-identical): c3 3.84 ->
// 3.65 us, c4 5.88 -> 5.79 us per launch.  The CSR kernels measured slower
// with it (c1 +7%, c2 +1.5%, c5 +2-3%) and keep streaming stores.

struct BsrArgs {
    const int*      row_ptr;
    const int*      col_idx;
    const _Float16* vals;
    const _Float16* B;
    float*          C;
    int             M;
    int             K;
    int             N;
    int             block_rows;
    int             b_vec_ok;  // N % 8 == 0 and B 16-byte aligned
    int             block_cols;
    int             tiles_n;    // wave kernel: column tiles (grid is 1-D)
    int             wg_total;   // wave kernel: tiles, one workgroup each
    int             xcd_order;  // wave kernel: 1 = XCD-grouped workgroup order
    int             sample_step;  // between the eight places of RunSample
    int             slices;     // record kernel: column slices where A's blocks lie in no runs
    int             num_blocks;
    int             c_vec_ok;   // C 16-byte aligned (with b_vec_ok: rows of 16-byte chunks)
};

__device__ __forceinline__ int div_up(int a, int b) { return (a + b - 1) / b; }

// Whether A's blocks lie in runs (banded, block-diagonal) rather than all over
// the block-rows: of eight entries in each of eight places of the list
// (num_blocks >= 8), most are followed by the next block-column.  Every wave of
// a launch reads the same entries and decides alike; the host cannot, A is on
// the device.  Only one load deep: the block-rows' ends through row_ptr cost 0.4
// - 0.9 us a launch, scalar loads 1.5 - 2.
struct RunSample {
    int here = 0;
    __device__ __forceinline__ void load(const BsrArgs& a) {
        const int lane = threadIdx.x & 63;
        here = a.col_idx[(lane >> 3) * a.sample_step + (lane & 7)];
    }
    __device__ __forceinline__ bool in_runs() const {
        const int next = __builtin_amdgcn_update_dpp(here, here, 0x101, 0xF, 0xF, false);  // row_shl:1
        return __popcll(__ballot(next - here == 1 && (threadIdx.x & 7) != 7)) > 28;  // of 56
    }
};

// Workgroup -> (block-row group, column tile) for the 1-D wave-kernel grid; bx
// = block_rows for a workgroup that has no tile.
// The hardware hands workgroup L to XCD L % 8.  With xcd_order, XCD x gets
// the contiguous logical range [x*T/8, (x+1)*T/8) (the first T % 8 XCDs one
// more), and logical ids run column tile fastest: each XCD works on its own
// band of block-rows with all their column tiles, so A blocks and the B rows
// that neighbouring block-rows share are fetched into one L2 only.
// With S > 1 slices, XCDs s*8/S .. (s+1)*8/S - 1 take the s-th part of the
// column tiles, each a band of the block-rows: its L2 holds 1/S of B.
// ONE: one slice and a grid of just the tiles.
template <bool ONE = false>
__device__ __forceinline__ void wave_tile_of(const BsrArgs& a, int slices, int& bx, int& by) {
    const int L = blockIdx.x;
    const int xcd = L & 7, idx = L >> 3;
    if (!ONE && slices > 1) {
        const int bands = 8 / slices;
        const int tiles = div_up(a.tiles_n, slices);
        const int rows  = div_up(div_up(a.block_rows, 4), bands);
        const int slice = xcd / bands;
        const int r     = idx / tiles;
        bx = (xcd - slice * bands) * rows + r;
        by = slice * tiles + idx - r * tiles;
        if (r >= rows || by >= a.tiles_n) bx = a.block_rows;
        return;
    }
    int l = L;
    bool live = L < a.wg_total;
    if (a.xcd_order) {
        const int per = a.wg_total >> 3, rem = a.wg_total & 7;
        live = idx < per + (xcd < rem ? 1 : 0);
        l = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
    }
    bx = l / a.tiles_n;
    by = l - bx * a.tiles_n;
    if (!ONE && !live) bx = a.block_rows;
}

// ---------------------------------------------------------------------------
// Wave kernel (pointer addressing: what the record kernel below does not take):
// one wave = one block-row x 16*J columns, four independent waves per
// workgroup, no workgroup barriers.  Maximum parallelism and a small LDS
// footprint (one 32 x (16J+16) fp16 tile per wave) keep many waves resident,
// which is what hides the latency of the short dependent chain row_ptr ->
// col_idx -> (A, B) -> MFMA.  Latency and the B re-reads of every block-row
// bound it.  Rows of B may start at any element: 16-byte chunks at any N and
// alignment (MI355X against one load per element, which bound those widths
// before: 5003 x 6997 blocks at 15%, N = 100 65.4 -> 15.6 us, one call from Python
// 66.8 -> 17.6; 8192^2 at 12.5%, N = 500 226 -> 48 us).
//   - The block-row's block-columns come in with one vector load (lane i
//     holds col_idx[first + i], 64 per chunk) and are broadcast with
//     v_readlane, so pairs need no further index loads.
//   - The A operands and B rows of the next D pairs are in flight while a
//     pair is multiplied (a ring of D register sets).
//   - B rows are written to the wave's LDS tile row-major (16-byte stores) and
//     read back as MFMA operands with ds_read_b64_tr_b16 (two per operand).
// LDS accesses of one wave execute in program order, so the single tile
// needs no barrier between a pair's reads and the next pair's writes.
// ---------------------------------------------------------------------------
// Eight fp16 at any element address (a 16-byte global load needs no alignment).
typedef f16x8 Mem __attribute__((aligned(2)));

// The 8 - n upper elements of v moved down, zeros above them.
__device__ __forceinline__ f16x8 drop_low(f16x8 v, int n) {
    unsigned __int128 x = __builtin_bit_cast(unsigned __int128, v);
    return __builtin_bit_cast(f16x8, n < 8 ? x >> (16 * n) : static_cast<unsigned __int128>(0));
}

// How a lane gets its eight elements of a B row: one at a time (B smaller than a
// chunk), 16 bytes at any element, or 16 bytes at a 16-byte address of rows
// that are whole chunks.  The last needs neither end of B nor shift: 3 - 30% less
// time than the any-element form there (32768^2 diagonal blocks of 256, N = 32 4.8
// against 6.8 us; 8192^2 blocks at 12.5%, N = 64 11.2 against 13.9).
enum class Chunks { Elements, Any, Aligned };

template <int J, int D, Chunks B_CHUNKS>
__global__ __launch_bounds__(256) void bsr_wave_kernel(BsrArgs a) {
    constexpr int NT  = 16 * J;          // columns per wave
    constexpr int S   = NT + 16;         // LDS row stride in fp16 (S/2 = 8 mod 32 banks)
    constexpr int CH  = NT / 8;          // 16-byte chunks per staged row
    constexpr int CPL = 32 * CH / 64;    // chunks per lane (J for the 32-row tile)
    __shared__ __attribute__((aligned(16))) _Float16 s_b[4][32 * S];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g    = lane >> 4;
    const int t    = lane & 15;
    int bx, by;
    wave_tile_of<true>(a, 1, bx, by);
    const int br   = bx * 4 + wave;
    const int n0   = by * NT;
    if (br >= a.block_rows) return;  // waves are independent: no barrier anywhere
    _Float16* tile = s_b[wave];

    const int bs = a.row_ptr[br];
    const int be = a.row_ptr[br + 1];

    f32x4 acc[J];
#pragma unroll
    for (int j = 0; j < J; ++j) acc[j] = f32x4(0.0f);

    // Registers of one pair: this lane's B chunks and A operand, and which of
    // them hold data.  Loads never branch: a lane whose row lies outside B
    // (past K, or the absent second block of an odd tail) reads a clamped,
    // valid address and its value is replaced by zero when it is used, so the
    // loads of all pairs in flight stay independent of each other.
    struct PairRegs {
        f16x8 b[CPL];
        f16x8 af;
        int   shift[CPL];  // elements the chunk was loaded before its own first
        bool  b_ok[CPL];
        bool  a_ok;
    };
    // Pair = blocks base+p and base+p+1 of the row (p and p+1 inside the
    // column-index chunk ci that starts at block base).
    auto load_pair = [&](int base, int p, int cnt, int ci, PairRegs& r) {
        const bool two = p + 1 < cnt;
        const int bc0 = __builtin_amdgcn_readlane(ci, p);
        const int bc1 = __builtin_amdgcn_readlane(ci, two ? p + 1 : p);
        const int blk = base + p;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            const int idx = lane + c * 64;
            const int s   = idx / CH;                 // staged row 0..31
            const int k   = (s < 16 ? bc0 : bc1) * 16 + (s & 15);
            const int n   = n0 + (idx % CH) * 8;
            const bool ok = (s < 16 || two) && k < a.K && n < a.N;
            r.b_ok[c] = ok;
            if constexpr (B_CHUNKS == Chunks::Aligned) {
                const size_t off = ok ? static_cast<size_t>(k) * a.N + n : 0;
                r.shift[c] = 0;
                r.b[c] = *reinterpret_cast<const f16x8*>(a.B + off);
            } else if constexpr (B_CHUNKS == Chunks::Any) {
                // A row may start at any element (Mem) and the last chunk of a
                // row may run into the next row: those products land in output
                // columns >= N, which are never stored.  Only past the end of
                // B is the chunk taken from B's last 8 elements instead and
                // shifted into place when it is used -- no branch here, so the
                // loads of all pairs in flight stay independent.
                const size_t off = ok ? static_cast<size_t>(k) * a.N + n : 0;
                const size_t at  = min(off, static_cast<size_t>(a.K) * a.N - 8);
                r.shift[c] = static_cast<int>(off - at);
                r.b[c] = *reinterpret_cast<const Mem*>(a.B + at);
            } else {
                const size_t row = ok ? static_cast<size_t>(k) * a.N : 0;
                r.shift[c] = 0;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const bool in = ok && n + e < a.N;
                    const _Float16 x = a.B[in ? row + n + e : 0];
                    r.b[c][e] = in ? x : static_cast<_Float16>(0.0f);
                }
            }
        }
        // A operand: row t of block blk (g < 2) or blk+1 (g >= 2), columns 8*(g&1) .. +7
        r.a_ok = g < 2 || two;
        r.af = *reinterpret_cast<const f16x8*>(
            a.vals + static_cast<size_t>(blk + (r.a_ok ? (g >> 1) : 0)) * 256 + t * 16 +
            8 * (g & 1));
    };
    auto multiply = [&](const PairRegs& r) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            const int idx = lane + c * 64;
            const f16x8 zero = f16x8(static_cast<_Float16>(0.0f));
            f16x8 b = r.b[c];
            if constexpr (B_CHUNKS == Chunks::Any) {
                if (__builtin_expect(__any(r.shift[c] != 0), 0)) b = drop_low(b, r.shift[c]);
            }
            *reinterpret_cast<f16x8*>(&tile[(idx / CH) * S + (idx % CH) * 8]) =
                r.b_ok[c] ? b : zero;
        }
        const f16x8 af = r.a_ok ? r.af : f16x8(static_cast<_Float16>(0.0f));
        const _Float16* rowp = &tile[(8 * g + (t >> 2)) * S + 4 * (t & 3)];
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const s16x4 lo = lds_read_tr16(rowp + 16 * j);
            const s16x4 hi = lds_read_tr16(rowp + 4 * S + 16 * j);
            const s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, __builtin_bit_cast(f16x8, both),
                                                             acc[j], 0, 0, 0);
        }
    };

    // D pairs in flight.  Pair i of a chunk lives in ring slot i % D.  The
    // steady-state loop refills every slot it empties, so each slot's loads
    // are issued unconditionally and the wait before a multiply covers only
    // that slot's loads; the drain finishes the last (fewer than 2D) pairs.
    for (int c0 = bs; c0 < be; c0 += 64) {  // 64 blocks per column-index chunk
        const int cnt = min(64, be - c0);
        const int np  = (cnt + 1) >> 1;     // pairs in this chunk
        const int ci  = lane < cnt ? a.col_idx[c0 + lane] : 0;
        PairRegs ring[D];
#pragma unroll
        for (int d = 0; d < D; ++d) load_pair(c0, 2 * min(d, np - 1), cnt, ci, ring[d]);
        int i0 = 0;
        for (; i0 + 2 * D <= np; i0 += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                multiply(ring[d]);
                load_pair(c0, 2 * (i0 + d + D), cnt, ci, ring[d]);
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (i0 + d < np) {
                multiply(ring[d]);
                if (i0 + d + D < np) load_pair(c0, 2 * (i0 + d + D), cnt, ci, ring[d]);
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (i0 + D + d < np) multiply(ring[d]);
        }
    }

    // D layout: lane holds rows 4*g + i, column t of each 16-column tile.
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int col = n0 + 16 * j + t;
        if (col >= a.N) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = br * 16 + 4 * g + i;
            if (row < a.M) store_c(a.C + static_cast<size_t>(row) * a.N + col, acc[j][i]);
        }
    }
}

// ---------------------------------------------------------------------------
// Record-addressed wave kernel (the default where it applies): the wave
// kernel's work split and ring, with B and the A blocks read as structured
// buffers -- one record per B row (N fp16) and one per 16x16 block.  The row
// or block number is the load's index operand, and the buffer range check
// returns zeros for an index past the end: rows >= K of a partial last
// block-column, and index -1 for the absent second block of an odd tail.  So
// a pair needs one index add per 16-byte chunk instead of 64-bit address
// arithmetic and per-lane zero selects (~30 -> ~6 vector instructions per
// pair).  The B rows of a pair go straight into the wave's LDS slot with
// buffer-to-LDS loads (no VGPR staging, no ds_write), one slot per pair in
// flight, each slot its own LDS object.  Measured on MI355X against the same
// kernel staging through VGPRs and ds_write (both at their default tiles):
// banded 8192^2 N=128 4.3 -> 4.1 us, block-diagonal 8192^2 N=256 6.4 -> 6.1
// us, identical results.  Needs N % 8 == 0 with 16-byte aligned B, N * 2 <= 16383 (record
// stride field), and B and A within 2 GiB each.
// ---------------------------------------------------------------------------
__device__ u32x4 sbuf_load_u32x4_dev(__amdgpu_buffer_rsrc_t rsrc, int index, int offset) {
    return sbuf_load_u32x4(rsrc, index, offset, 0, 0);
}

template <int J, int D, bool ONE = false>
__device__ __forceinline__ void bsr_record_body(const BsrArgs& a, int slices,
                                                _Float16* __restrict__ s0,
                                                _Float16* __restrict__ s1,
                                                _Float16* __restrict__ s2,
                                                _Float16* __restrict__ s3) {
    constexpr int NT   = 16 * J;       // columns per wave
    constexpr int CH   = NT / 8;       // 16-byte chunks per staged row
    constexpr int CPL  = 32 * CH / 64; // chunks per lane (one load instruction each)
    constexpr int TILE = 32 * NT;      // fp16 per slot: the pair's 32 B rows, row-major
    constexpr int PER  = CPL + 1;      // vector-memory instructions per pair

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g    = lane >> 4;
    const int t    = lane & 15;
    int bx, by;
    wave_tile_of<ONE>(a, slices, bx, by);
    const int br   = bx * 4 + wave;
    const int n0   = by * NT;
    if (br >= a.block_rows) return;  // waves are independent: no barrier anywhere
    auto slot = [&](int d) -> _Float16* {
        return (d == 0 ? s0 : d == 1 ? s1 : d == 2 ? s2 : s3) + wave * TILE;
    };

    const __amdgpu_buffer_rsrc_t rec_b = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16*>(a.B), static_cast<short>(a.N * 2), a.K, kBufWord3);
    const __amdgpu_buffer_rsrc_t rec_a = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16*>(a.vals), static_cast<short>(512), a.num_blocks, kBufWord3);

    // Lane constants: load instruction c fills 16-byte position idx = lane +
    // 64c of the slot, staged row srow (block srow >= 16 of the pair).  The
    // slot is row-major with its chunks XOR-swizzled per row (chunk k of row
    // r at position k ^ swz(r)), which spreads the rows one
    // ds_read_b64_tr_b16 touches over all LDS banks; so position idx holds
    // chunk (idx % CH) ^ swz(srow): columns n .. n+7, byte offset nbyte of
    // its B row.  Columns past N read a valid chunk of the row instead; their
    // products land in output columns >= N, which are never stored.
    auto swz = [](int r) { return (2 * ((r >> 1) ^ (r >> 3))) & (CH - 1); };
    int srow[CPL], nbyte[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
        const int idx = lane + c * 64;
        srow[c] = idx / CH;
        const int n = n0 + ((idx % CH) ^ swz(srow[c])) * 8;
        nbyte[c] = (n < a.N ? n : 0) * 2;
    }
    // B operand reads: rows 8g + t/4 (lo) and +4 (hi), chunk 2j + (t & 3) / 2
    // of the row, bytes 8 * (t & 1) of it; swz(r) is even, so the swizzle
    // XORs the tile index j with swz(r) / 2.
    const int h_lo  = swz(8 * g + (t >> 2)) >> 1;
    const int h_hi  = swz(8 * g + (t >> 2) + 4) >> 1;
    const int in_lo = (8 * g + (t >> 2)) * NT + ((t & 3) >> 1) * 8 + (t & 1) * 4;  // fp16 units
    const int in_hi = in_lo + 4 * NT;
    // A operand: row t of block (first, g < 2) or (second, g >= 2), columns 8*(g&1) .. +7
    const int a_off = t * 32 + 16 * (g & 1);
    const int a_hi  = g >> 1;

    const int bs = a.row_ptr[br];
    const int be = a.row_ptr[br + 1];

    f32x4 acc[J];
#pragma unroll
    for (int j = 0; j < J; ++j) acc[j] = f32x4(0.0f);

    u32x4 af[D];
    // Pair = blocks base+p and base+p+1 of the row (p and p+1 inside the
    // column-index chunk ci that starts at block base), into ring slot d.
    auto load_pair = [&](int d, int base, int p, int cnt, int ci) {
        const bool two = p + 1 < cnt;
        const int bc0 = __builtin_amdgcn_readlane(ci, p);
        const int bc1 = two ? __builtin_amdgcn_readlane(ci, p + 1) : -1;  // rows -16..-1: zeros
        _Float16* dst = slot(d);
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            const int sr = srow[c];
            sbuf_load_lds(rec_b, (spmm_lds_ptr)(dst + c * 512), 16,
                          (sr < 16 ? bc0 : bc1) * 16 + (sr & 15), nbyte[c], 0, 0, 0);
        }
        af[d] = sbuf_load_u32x4_dev(rec_a, (two || a_hi == 0) ? base + p + a_hi : -1, a_off);
    };
    auto multiply = [&](int d) {
        const f16x8 afv = __builtin_bit_cast(f16x8, af[d]);
        const _Float16* st = slot(d);
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const s16x4 lo = lds_read_tr16(st + in_lo + (j ^ h_lo) * 16);
            const s16x4 hi = lds_read_tr16(st + in_hi + (j ^ h_hi) * 16);
            const s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(afv, __builtin_bit_cast(f16x8, both),
                                                             acc[j], 0, 0, 0);
        }
    };

    // D pairs in flight.  Vector-memory instructions retire in issue order,
    // so before slot d is read, waiting until at most (D-1) pairs' loads are
    // outstanding guarantees slot d's are done.  A slot is refilled only after
    // the MFMAs that consumed its reads, so its reads are complete by then.
    // The drain (fewer loads after each slot) waits for everything.
    for (int c0 = bs; c0 < be; c0 += 64) {  // 64 blocks per column-index chunk
        const int cnt = min(64, be - c0);
        const int np  = (cnt + 1) >> 1;
        const int ci  = lane < cnt ? a.col_idx[c0 + lane] : 0;
#pragma unroll
        for (int d = 0; d < D; ++d) load_pair(d, c0, 2 * min(d, np - 1), cnt, ci);
        int i0 = 0;
        for (; i0 + 2 * D <= np; i0 += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                wait_vmcnt<(D - 1) * PER>();
                multiply(d);
                load_pair(d, c0, 2 * (i0 + d + D), cnt, ci);
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (i0 + d < np) {
                wait_vmcnt<0>();
                multiply(d);
                if (i0 + d + D < np) load_pair(d, c0, 2 * (i0 + d + D), cnt, ci);
            }
        }
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (i0 + D + d < np) {
                wait_vmcnt<0>();
                multiply(d);
            }
        }
    }

    // D layout: lane holds rows 4*g + i, column t of each 16-column tile.
    if (a.c_vec_ok) {
        // The tile goes through the wave's first ring slot (16 x NT fp32 is
        // exactly its size, and every load into it has landed) and leaves
        // row-major in 16-byte stores: each store instruction writes whole
        // NT-column row segments instead of 64-byte pieces of four rows.
        // Measured on MI355X: c3 3.87 -> 3.71 us, c4 5.83 -> 5.74 us per launch.
        wait_vmcnt<0>();
        float* ct = reinterpret_cast<float*>(slot(0));
#pragma unroll
        for (int j = 0; j < J; ++j) {
#pragma unroll
            for (int i = 0; i < 4; ++i) ct[(4 * g + i) * NT + 16 * j + t] = acc[j][i];
        }
        constexpr int LPR = NT / 4;    // lanes per row, 4 floats each
        constexpr int RPI = 64 / LPR;  // rows per store instruction
        const int lr = lane / LPR;
        const int lc = (lane % LPR) * 4;
        // The block-row's C rows as one raw buffer (at most 16 x 8191 floats,
        // so byte offsets fit 32 bits whatever the size of C).
        const int rows_here = min(16, a.M - br * 16);
        const __amdgpu_buffer_rsrc_t c_rows = __builtin_amdgcn_make_buffer_rsrc(
            a.C + static_cast<size_t>(br) * 16 * a.N, static_cast<short>(0),
            rows_here * a.N * 4, kBufWord3);
#pragma unroll
        for (int s = 0; s < 16 / RPI; ++s) {
            const int r   = s * RPI + lr;
            const f32x4 v = *reinterpret_cast<const f32x4*>(ct + r * NT + lc);
            const int col = n0 + lc;  // N % 8 == 0: a chunk is all in or all out
            if (r < rows_here && col < a.N) {
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), c_rows,
                                                       (r * a.N + col) * 4, 0, kStoreDevice);
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int col = n0 + 16 * j + t;
        if (col >= a.N) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = br * 16 + 4 * g + i;
            if (row < a.M) store_c(a.C + static_cast<size_t>(row) * a.N + col, acc[j][i]);
        }
    }
}

// The ring slots are separate LDS objects passed as restrict pointers: after
// inlining, every slot access carries its own alias scope, which lets the
// compiler's wait-count pass tell a read of slot d from the buffer-to-LDS
// writes still in flight into the other slots.
template <int J, int D, bool SLICES>
__global__ __launch_bounds__(256) void bsr_record_kernel(BsrArgs a) {
    constexpr int TILE = 32 * 16 * J;
    static_assert(D == 2 || D == 4, "ring depth 2 or 4");
    __shared__ __attribute__((aligned(16))) _Float16 s_b0[4 * TILE];
    __shared__ __attribute__((aligned(16))) _Float16 s_b1[4 * TILE];
    __shared__ __attribute__((aligned(16))) _Float16 s_b2[D == 4 ? 4 * TILE : 8];
    __shared__ __attribute__((aligned(16))) _Float16 s_b3[D == 4 ? 4 * TILE : 8];
    if constexpr (SLICES) {
        RunSample sample;
        sample.load(a);
        bsr_record_body<J, D>(a, sample.in_runs() ? 1 : a.slices, s_b0, s_b1, s_b2, s_b3);
    } else {
        bsr_record_body<J, D, true>(a, 1, s_b0, s_b1, s_b2, s_b3);
    }
}

// ---------------------------------------------------------------------------
// Shared-panel kernel: a workgroup owns R consecutive block-rows (16R rows of
// C) and NT = 16*J columns, and multiplies them by B one union block pair at
// a time.
//   1. Union of the R block-rows' block-column lists (contiguous in col_idx).
//      Fast path, when every block-column lies within 64 of the smallest and
//      there are at most 256 entries: each wave ORs a 64-bit mask per
//      block-row with DPP and one barrier combines the waves.  Otherwise an
//      LDS bitmap over all block-columns (up to kPanelMaxWords * 32) and an
//      exclusive prefix of its words' popcounts rank every block-column.
//   2. The union's slots go into lane-indexed registers (per slot: the
//      block-column, and this wave's blocks there or -1), which the pipeline
//      reads with v_readlane: a pair costs the scalar unit only its slot
//      numbers, and the pipeline reads no LDS but the B stages.
//   3. Slots are multiplied in pairs (two 16-deep blocks are one K = 32 step
//      of v_mfma_f32_16x16x32_f16).  A pair's 32 B rows x NT columns are
//      loaded once per workgroup straight into an LDS stage (buffer-to-LDS
//      loads, XOR-swizzled against bank conflicts) and read by every wave
//      with ds_read_b64_tr_b16; each wave loads the A operands of its own
//      block-rows (an absent block has index -1 and reads as zeros through
//      the buffer range check).  D stages in flight, one barrier per pair.
//   4. The four waves form a WR x (4/WR) grid over the tile: a wave multiplies
//      R/WR block-rows by J/(4/WR) 16-column tiles.
// Lists that are not strictly ascending or hold block-columns outside the
// matrix, and matrices wider than the bitmap, use the identity union (slot u =
// entry u of the concatenated lists): correct for any BSR, at up to R times
// the matrix-core work.
//
// What it buys, measured on MI355X (rocprofv3 counters, c4): the wave
// kernel's four waves of a workgroup already share their B tiles through the
// vector L1 -- both kernels make the same 263 K L2 read requests per launch
// -- so the panel saves L1 accesses (0.66 M vs 1.44 M of 64 bytes) but pays
// barriers, lockstep phases and LDS read bandwidth.  It is faster only on
// wide B with long block-rows (N >= 256 and 24 - 64 blocks per block-row:
// 1.03 - 1.31x, e.g. block-diagonal 512 at N = 512 12.6 -> 10.8 us), and
// the launcher picks it there for A in runs; c3 and c4 stay on the wave kernel.
// ---------------------------------------------------------------------------
constexpr int kPanelMaxWords = 256;  // union bitmap: up to 8192 block-columns (K <= 131072)
constexpr int kPanelSlots    = 126;  // union slots per pass (two registers per lane, lane 127 free)

__device__ __forceinline__ int wave_inclusive_scan(int v, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(v, d, 64);
        if (lane >= d) v += u;
    }
    return v;
}

// OR of a 64-bit value over the 64 lanes of a wave (all lanes active): DPP
// xor-1 and xor-2 inside quads, then half-row and row mirrors give every
// lane its row's OR, and the four rows are combined from lanes 0, 16, 32, 48.
__device__ __forceinline__ uint64_t wave_or64(uint64_t v) {
    unsigned lo = static_cast<unsigned>(v), hi = static_cast<unsigned>(v >> 32);
    lo |= __builtin_amdgcn_update_dpp(0u, lo, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
    hi |= __builtin_amdgcn_update_dpp(0u, hi, 0xB1, 0xF, 0xF, false);
    lo |= __builtin_amdgcn_update_dpp(0u, lo, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
    hi |= __builtin_amdgcn_update_dpp(0u, hi, 0x4E, 0xF, 0xF, false);
    lo |= __builtin_amdgcn_update_dpp(0u, lo, 0x141, 0xF, 0xF, false);  // row_half_mirror
    hi |= __builtin_amdgcn_update_dpp(0u, hi, 0x141, 0xF, 0xF, false);
    lo |= __builtin_amdgcn_update_dpp(0u, lo, 0x140, 0xF, 0xF, false);  // row_mirror
    hi |= __builtin_amdgcn_update_dpp(0u, hi, 0x140, 0xF, 0xF, false);
    const unsigned rlo = __builtin_amdgcn_readlane(lo, 0) | __builtin_amdgcn_readlane(lo, 16) |
                         __builtin_amdgcn_readlane(lo, 32) | __builtin_amdgcn_readlane(lo, 48);
    const unsigned rhi = __builtin_amdgcn_readlane(hi, 0) | __builtin_amdgcn_readlane(hi, 16) |
                         __builtin_amdgcn_readlane(hi, 32) | __builtin_amdgcn_readlane(hi, 48);
    return (static_cast<uint64_t>(rhi) << 32) | rlo;
}

__device__ __forceinline__ uint64_t below(int p) {  // bits 0 .. p-1, p in [0, 64)
    return (1ull << p) - 1ull;
}

// Block-rows br0 .. br0+rows-1 of `tiles` 16-column tiles from n0, by one wave and
// block by block straight from memory: what a panel's wave does with sums that are
// not finite.  The order of the sums is the panel's.
__device__ void bsr_tiles_apart(const BsrArgs& a, int br0, int rows, int n0, int tiles, int lane) {
    const int g = lane >> 4, t = lane & 15;
    for (int br = br0; br < min(br0 + rows, a.block_rows); ++br) {
        for (int j = 0; j < tiles; ++j) {
            const int col = n0 + 16 * j + t;
            f32x4 acc = f32x4(0.0f);
            for (int e = a.row_ptr[br]; e < a.row_ptr[br + 1]; ++e) {
                const int  bc = a.col_idx[e];
                const bool in = static_cast<unsigned>(bc) < static_cast<unsigned>(a.block_cols);
                f16x4 b;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int  k  = bc * 16 + 4 * g + i;
                    const bool ok = in && k < a.K && col < a.N;
                    b[i] = ok ? a.B[static_cast<size_t>(k) * a.N + col] : static_cast<_Float16>(0.0f);
                }
                const f16x4 av = *reinterpret_cast<const f16x4*>(
                    a.vals + static_cast<size_t>(e) * 256 + t * 16 + 4 * g);
                acc = __builtin_amdgcn_mfma_f32_16x16x16f16(av, b, acc, 0, 0, 0);
            }
            if (col >= a.N) continue;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int row = br * 16 + 4 * g + k;
                if (row < a.M) store_c(a.C + static_cast<size_t>(row) * a.N + col, acc[k]);
            }
        }
    }
}

// CHOOSE: returns false, with nothing done, where A's blocks lie in no runs.
// The sample's loads go out before the panel's own and wait with them.
template <int R, int J, int WR, int D, bool CHOOSE = false>
__device__ __forceinline__ bool bsr_panel_body(const BsrArgs& a, _Float16* __restrict__ s0,
                                               _Float16* __restrict__ s1,
                                               _Float16* __restrict__ s2,
                                               _Float16* __restrict__ s3,
                                               uint32_t* __restrict__ s_bits,
                                               int* __restrict__ s_pre, int* __restrict__ s_ucol,
                                               int* __restrict__ s_blk,
                                               uint64_t* __restrict__ s_mask,
                                               int* __restrict__ s_misc) {
    constexpr int WC  = 4 / WR;
    constexpr int TR  = R / WR;          // block-rows per wave
    constexpr int TC  = J / WC;          // 16-column tiles per wave
    constexpr int NT  = 16 * J;          // columns per workgroup
    constexpr int CH  = NT / 8;          // 16-byte chunks per staged B row
    constexpr int CPT = 32 * CH / 256;   // chunks per thread per pair
    constexpr int PER = CPT + TR;        // vector-memory instructions per thread per pair
    static_assert(WR * WC == 4 && TR * WR == R && TC * WC == J, "wave grid");
    static_assert(CPT >= 1 && CPT * 256 == 32 * CH, "whole chunks per thread");
    static_assert(64 / CH <= 16, "a wave's chunks of one load stay inside one block");
    static_assert(D == 2 || D == 4, "2 or 4 stages");

    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g    = lane >> 4;
    const int t    = lane & 15;
    const int wr   = wave / WC;
    const int wc   = wave % WC;
    int bx, by;
    wave_tile_of<!CHOOSE>(a, 1, bx, by);
    const int br0 = bx * R;  // to choose, a workgroup without a tile has empty block-rows
    const int n0  = by * NT;
    auto stage = [&](int d) -> _Float16* { return d == 0 ? s0 : d == 1 ? s1 : d == 2 ? s2 : s3; };

    const __amdgpu_buffer_rsrc_t rec_b = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16*>(a.B), static_cast<short>(a.N * 2), a.K, kBufWord3);
    const __amdgpu_buffer_rsrc_t rec_a = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16*>(a.vals), static_cast<short>(512), a.num_blocks, kBufWord3);

    RunSample sample;
    if constexpr (CHOOSE) sample.load(a);
    // Block-rows br0 .. br0+R-1 (those past the matrix are empty); their
    // lists are contiguous in col_idx from e0.
    int rp[R + 1];
#pragma unroll
    for (int r = 0; r <= R; ++r) rp[r] = a.row_ptr[min(br0 + r, a.block_rows)];
    const int e0 = rp[0];
    const int T  = rp[R] - e0;
    auto list_of = [&](int e) {  // block-row (0 .. R-1) of entry e0 + e
        int r = 0;
#pragma unroll
        for (int i = 1; i < R; ++i) r += (e0 + e >= rp[i]) ? 1 : 0;
        return r;
    };
    auto list_start = [&](int e) {  // first entry of e0 + e's block-row (selects, no indexing)
        int st = rp[0];
#pragma unroll
        for (int i = 1; i < R; ++i) st = (e0 + e >= rp[i]) ? rp[i] : st;
        return st;
    };
    // Span of the block-columns from the lists' first and last entries.
    int lo = 0x7fffffff, hi = -1;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (rp[r + 1] > rp[r]) {
            lo = min(lo, a.col_idx[rp[r]]);
            hi = max(hi, a.col_idx[rp[r + 1] - 1]);
        }
    }
    if constexpr (CHOOSE) {
        if (!sample.in_runs()) return false;
        if (br0 >= a.block_rows) return true;
    }
    // Stage layout: row-major 32 x NT fp16, its 16-byte chunks XOR-swizzled
    // per row (chunk c of row r sits at position c ^ swz(r)), which spreads
    // the sixteen rows one ds_read_b64_tr_b16 touches over all banks (4
    // conflict-free cycles instead of 16 with 32 banks).  A buffer-to-LDS load
    // puts lane i's 16 bytes at a fixed position, so the swizzle picks which
    // chunk each lane loads: load c of a pair fills position idx = 256c + tid,
    // i.e. staged row srow, with chunk (idx % CH) ^ swz(srow): columns n ..
    // n+7.  Rows 0-15 hold the pair's first block-column, 16-31 the second
    // (the same half for a whole wave's load).  Columns past N read a valid
    // chunk of the row instead; their products land in output columns >= N,
    // which are never stored.
    auto swz = [](int r) { return (2 * ((r >> 1) ^ (r >> 3))) & (CH - 1); };
    int srow[CPT], nbyte[CPT];
    bool second[CPT];
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
        const int idx = c * 256 + tid;
        srow[c]   = idx / CH;
        second[c] = __builtin_amdgcn_readfirstlane(srow[c] >> 4) != 0;
        const int n = n0 + ((idx % CH) ^ swz(srow[c])) * 8;
        nbyte[c] = (n < a.N ? n : 0) * 2;
    }

    // A operand: row t of the pair's block g >> 1, columns 8 * (g & 1) .. +7
    const int a_off = t * 32 + 16 * (g & 1);
    // B operand reads: lane (g, t) addresses rows 8g + t/4 (lo) and +4 (hi),
    // chunk 2 * tile + (t & 3) / 2 of the row, bytes 8 * (t & 1) of it; with
    // swz(r) even, the swizzle XORs the tile index with swz(r) / 2.
    const int row_lo = 8 * g + (t >> 2);
    const int h_lo   = swz(row_lo) >> 1;
    const int h_hi   = swz(row_lo + 4) >> 1;
    const int in_lo  = row_lo * NT + ((t & 3) >> 1) * 8 + (t & 1) * 4;  // fp16 units
    const int in_hi  = in_lo + 4 * NT;

    f32x4 acc[TR][TC];
#pragma unroll
    for (int i = 0; i < TR; ++i) {
#pragma unroll
        for (int j = 0; j < TC; ++j) acc[i][j] = f32x4(0.0f);
    }
    u32x4 af[D][TR];

    int off_lo[TC], off_hi[TC];  // per tile: this lane's B operand addresses in a stage
#pragma unroll
    for (int j = 0; j < TC; ++j) {
        off_lo[j] = in_lo + ((wc * TC + j) ^ h_lo) * 16;
        off_hi[j] = in_hi + ((wc * TC + j) ^ h_hi) * 16;
    }
    auto compute = [&](int d) {
        const _Float16* st = stage(d);
#pragma unroll
        for (int j = 0; j < TC; ++j) {
            const s16x4 lo4 = lds_read_tr16(st + off_lo[j]);
            const s16x4 hi4 = lds_read_tr16(st + off_hi[j]);
            const s16x8 both = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
            const f16x8 bop = __builtin_bit_cast(f16x8, both);
#pragma unroll
            for (int i = 0; i < TR; ++i) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                    __builtin_bit_cast(f16x8, af[d][i]), bop, acc[i][j], 0, 0, 0);
            }
        }
    };

    // This thread's entry (the fast path needs at most one per thread).
    const int  x    = tid < T ? a.col_idx[e0 + tid] : 0;
    const int  xp   = tid < T && tid > 0 ? a.col_idx[e0 + tid - 1] : -1;
    const int  my_r = list_of(tid);
    // ---- 1. union of the R lists (fast path: DPP masks and one barrier;
    // otherwise the LDS bitmap and its word prefix; identity union for lists
    // that fail the checks or matrices wider than the bitmap).
    const bool fast_shape = T > 0 && T <= 256 && lo >= 0 && hi - lo < 64;
    const int  nwords     = (a.block_cols + 31) >> 5;
    const bool fits       = nwords <= kPanelMaxWords;
    bool bad = false;
    if (fast_shape) {
        const bool ok = tid >= T || (static_cast<unsigned>(x) < static_cast<unsigned>(a.block_cols) &&
                                     x >= lo && x - lo < 64 &&
                                     (e0 + tid == list_start(tid) || xp < x));
        const uint64_t bit = (tid < T && ok) ? (1ull << (x - lo)) : 0ull;
        uint64_t wm[R];
#pragma unroll
        for (int r = 0; r < R; ++r) wm[r] = wave_or64(my_r == r ? bit : 0ull);
        const bool wbad = __ballot(!ok) != 0;
        if (lane == 0) {
#pragma unroll
            for (int r = 0; r < R; ++r) s_mask[wave * R + r] = wm[r];
            s_misc[4 + wave] = wbad ? 1 : 0;
        }
    } else {
        if (fits) {
            for (int w = tid; w < nwords; w += 256) s_bits[w] = 0u;
        }
        if (tid == 0) s_misc[0] = fits ? 0 : 1;  // 1: identity union
    }
    for (int i = tid; i < kPanelSlots * R; i += 256) s_blk[i] = -1;
    __syncthreads();
    uint64_t rmask[R];  // fast path: block-row r's block-columns, bit = column - lo
    if (fast_shape) {
        bad = (s_misc[4] | s_misc[5] | s_misc[6] | s_misc[7]) != 0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            rmask[r] = s_mask[r] | s_mask[R + r] | s_mask[2 * R + r] | s_mask[3 * R + r];
        }
    }
    const bool use_fast = fast_shape && !bad;
    bool identity = fast_shape ? bad : false;
    if (!fast_shape) {
        for (int e = tid; e < T; e += 256) {
            const int xe = e < 256 ? x : a.col_idx[e0 + e];
            const bool wrong = static_cast<unsigned>(xe) >= static_cast<unsigned>(a.block_cols) ||
                               (e0 + e != list_start(e) && a.col_idx[e0 + e - 1] >= xe);
            if (wrong) {
                s_misc[0] = 1;  // every writer stores 1
            } else if (fits) {
                atomicOr(&s_bits[xe >> 5], 1u << (xe & 31));
            }
        }
        __syncthreads();
        identity = s_misc[0] != 0;
        if (!identity) {
            if (wave == 0) {  // lane l: words 4l .. 4l+3 (nwords <= 256)
                int pc[4], sum = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int w = 4 * lane + k;
                    pc[k] = w < nwords ? __builtin_popcount(s_bits[w]) : 0;
                    sum += pc[k];
                }
                const int incl = wave_inclusive_scan(sum, lane);
                int run = incl - sum;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if (4 * lane + k < nwords) s_pre[4 * lane + k] = run;
                    run += pc[k];
                }
                if (lane == 63) s_misc[1] = incl;
            }
            __syncthreads();
        }
    }
    uint64_t umask = 0ull;
    if (use_fast) {
#pragma unroll
        for (int r = 0; r < R; ++r) umask |= rmask[r];
    }
    const int U = use_fast ? __builtin_popcountll(umask) : (identity ? T : s_misc[1]);
    // This wave's block-rows wr*TR .. wr*TR+TR-1: first entries and masks,
    // picked with selects (a runtime index into rp / rmask would put the
    // arrays in scratch memory).
    int      my_rp[TR];
    uint64_t my_mask[TR];
#pragma unroll
    for (int i = 0; i < TR; ++i) {
        my_rp[i]   = 0;
        my_mask[i] = 0ull;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r == wr * TR + i) {
                my_rp[i] = rp[r];
                if (use_fast) my_mask[i] = rmask[r];
            }
        }
    }

    // ---- 2. the pass's slot tables in registers: lane l of tcol[k] holds the
    // block-column of union slot 64k + l (-1 past the pass's end), lane l of
    // tblk[i][k] the block of this wave's block-row i at that slot (-1 where
    // it has none).  The pipeline reads them with v_readlane (a vector
    // instruction), so a pair costs the scalar unit only its slot numbers and
    // reads no LDS but the B stages.  Lane 63 of the last table always holds
    // -1 (a pass has at most kPanelSlots <= 126 slots): slot numbers are
    // clamped to it, so the zero pairs past the end need no test.
    int tcol[2], tblk[TR][2];
    // Pipeline over a pass of uc slots: pair q (slots 2q, 2q+1) lives in
    // stage q % D.  Before pair q is read, each thread waits until its own
    // loads of pair q have landed (loads retire in issue order, so the D - 2
    // later pairs' loads may stay outstanding) and the barrier makes every
    // thread's share visible.  The barrier is a bare s_barrier:
    // __syncthreads' release fence would also wait for the later pairs'
    // buffer-to-LDS writes, draining the ring at every pair.  A wave reaches
    // it with its LDS reads of pair q - 1 complete (the matrix-core
    // instructions consumed them), and the stage refilled right after it held
    // pair q - 1.  Every issue is unconditional: pairs past the last one read
    // -1 and load zeros (out of range, no memory traffic), so the loads in
    // flight are the same on every path and the compiler's own wait counts
    // stay exact.
    auto pipeline = [&](int uc, auto two_tables) {
        constexpr bool TWO = decltype(two_tables)::value;
        auto pick = [&](const int (&v)[2], int u) -> int {
            if constexpr (TWO) {
                const int uu = min(u, 127);
                return uu < 64 ? __builtin_amdgcn_readlane(v[0], uu)
                               : __builtin_amdgcn_readlane(v[1], uu - 64);
            } else {
                return __builtin_amdgcn_readlane(v[0], min(u, 63));
            }
        };
        auto issue = [&](int d, int q) {
            _Float16* dst = stage(d);
#pragma unroll
            for (int c = 0; c < CPT; ++c) {
                const int bc = pick(tcol, 2 * q + (second[c] ? 1 : 0));  // -1: rows -16..-1, zeros
                sbuf_load_lds(rec_b, (spmm_lds_ptr)(dst + (c * 256 + wave * 64) * 8), 16,
                              bc * 16 + (srow[c] & 15), nbyte[c], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < TR; ++i) {
                const int b0 = pick(tblk[i], 2 * q);
                const int b1 = pick(tblk[i], 2 * q + 1);
                af[d][i] = sbuf_load_u32x4_dev(rec_a, (g >> 1) ? b1 : b0, a_off);
            }
        };
        const int npairs = (uc + 1) >> 1;
#pragma unroll
        for (int d = 0; d < D - 1; ++d) issue(d, d);
        const int rounds = (npairs + D - 1) / D * D;
        for (int q0 = 0; q0 < rounds; q0 += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                wait_vmcnt<(D - 2) * PER>();
                lds_barrier();
                issue((d + D - 1) % D, q0 + d + D - 1);
                if (q0 + d < npairs) compute(d);
            }
        }
        wait_vmcnt<0>();  // the zero loads of the pairs past the end
    };

    if (use_fast) {
        // Lane p stands for block-column lo + p: if it is in the union, its
        // slot is the number of union columns below it, and ds_permute pushes
        // its table entries to that lane (lanes outside the union push to lane
        // 63, which is at or past U and is reset to -1).
        const bool in_u = ((umask >> lane) & 1ull) != 0;
        const int  addr = (in_u ? __builtin_popcountll(umask & below(lane)) : 63) * 4;
        const int  col  = __builtin_amdgcn_ds_permute(addr, lo + lane);
        tcol[0] = lane < U ? col : -1;
        tcol[1] = -1;
#pragma unroll
        for (int i = 0; i < TR; ++i) {
            const bool has = ((my_mask[i] >> lane) & 1ull) != 0;
            const int blk = has ? my_rp[i] + __builtin_popcountll(my_mask[i] & below(lane)) : -1;
            const int got = __builtin_amdgcn_ds_permute(addr, blk);
            tblk[i][0] = lane < U ? got : -1;
            tblk[i][1] = -1;
        }
        if (U <= 63) {
            pipeline(U, std::integral_constant<bool, false>());
        } else {
            pipeline(U, std::integral_constant<bool, true>());
        }
    } else {
        for (int u0 = 0; u0 < U; u0 += kPanelSlots) {
            const int uc = min(kPanelSlots, U - u0);
            if (u0 > 0) {  // the first pass's table was cleared before the union
                for (int i = tid; i < uc * R; i += 256) s_blk[i] = -1;
                __syncthreads();
            }
            for (int e = tid; e < T; e += 256) {
                const int xe = e < 256 ? x : a.col_idx[e0 + e];
                int u = e - u0;
                if (!identity) {
                    u = s_pre[xe >> 5] +
                        __builtin_popcount(s_bits[xe >> 5] & ((1u << (xe & 31)) - 1u)) - u0;
                }
                if (u >= 0 && u < uc) {
                    s_blk[u * R + list_of(e)] = e0 + e;
                    s_ucol[u] = xe;
                }
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int u = 64 * k + lane;
                tcol[k] = u < uc ? s_ucol[u] : -1;
#pragma unroll
                for (int i = 0; i < TR; ++i) tblk[i][k] = u < uc ? s_blk[u * R + wr * TR + i] : -1;
            }
            if (uc <= 63) {
                pipeline(uc, std::integral_constant<bool, false>());
            } else {
                pipeline(uc, std::integral_constant<bool, true>());
            }
            __syncthreads();  // the next pass rewrites the tables and the stages
        }
    }


    // D layout: lane holds rows 4*g + i, column t of each 16-column tile.
#pragma unroll
    for (int i = 0; i < TR; ++i) {
        const int br = br0 + wr * TR + i;
#pragma unroll
        for (int j = 0; j < TC; ++j) {
            const int col = n0 + (wc * TC + j) * 16 + t;
            if (col >= a.N) continue;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int row = br * 16 + 4 * g + k;
                if (row < a.M) store_c(a.C + static_cast<size_t>(row) * a.N + col, acc[i][j][k]);
            }
        }
    }
    // A block-row's pair is multiplied with the B rows of both its slots, those
    // of a block that it has not by an A of zeros: an infinity or a NaN there, of
    // another block-row's, would be in its sums.  Looked for behind the stores,
    // which the lanes then write again.
    f32x4 z = f32x4(0.0f);
#pragma unroll
    for (int i = 0; i < TR; ++i) {
#pragma unroll
        for (int j = 0; j < TC; ++j) {
#pragma unroll
            for (int k = 0; k < 4; ++k) z[k] = __builtin_fmaf(acc[i][j][k], 0.0f, z[k]);
        }
    }
    if (__builtin_expect(__any((z[0] + z[1]) + (z[2] + z[3]) != 0.0f), 0)) {
        bsr_tiles_apart(a, br0 + wr * TR, TR, n0 + wc * TC * 16, TC, lane);
    }
    return true;
}

// The stages and tables are separate LDS objects passed as restrict pointers
// (as in the record kernel): the wait-count pass then sees that reading one
// stage does not depend on buffer-to-LDS writes still going into another.
template <int R, int J, int WR, int D>
__global__ __launch_bounds__(256) void bsr_panel_kernel(BsrArgs a) {
    constexpr int TILE = 32 * 16 * J;
    __shared__ __attribute__((aligned(16))) _Float16 s_b0[TILE];
    __shared__ __attribute__((aligned(16))) _Float16 s_b1[TILE];
    __shared__ __attribute__((aligned(16))) _Float16 s_b2[D >= 3 ? TILE : 8];
    __shared__ __attribute__((aligned(16))) _Float16 s_b3[D >= 4 ? TILE : 8];
    __shared__ uint32_t s_bits[kPanelMaxWords];
    __shared__ int s_pre[kPanelMaxWords];
    __shared__ int s_ucol[kPanelSlots];
    __shared__ int s_blk[kPanelSlots * R];
    __shared__ uint64_t s_mask[4 * R];
    __shared__ int s_misc[8];
    bsr_panel_body<R, J, WR, D>(a, s_b0, s_b1, s_b2, s_b3, s_bits, s_pre, s_ucol, s_blk, s_mask,
                                s_misc);
}

// The waves of bsr_wide_kernel: the record kernel's work of four 16-column tiles,
// with single blocks (not pairs) following each other through three slots.  A
// block's loads go out two blocks ahead, about as far ahead as of pairs in two
// slots, in 6 KiB a wave instead of eight: five of these workgroups fit a CU, as
// of the panel kernel's, where 32 KiB would hold four (LDS is given out in 1280
// bytes).
__device__ __forceinline__ void bsr_wide_waves(const BsrArgs& a, int slices,
                                               _Float16* __restrict__ s0,
                                               _Float16* __restrict__ s1,
                                               _Float16* __restrict__ s2) {
    constexpr int BLOCK = 16 * 64;  // fp16 of a slot: 16 B rows x 64 columns
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g    = lane >> 4;
    const int t    = lane & 15;
    int bx, by;
    wave_tile_of(a, slices, bx, by);
    const int br = bx * 4 + wave;
    const int n0 = by * 64;
    if (br >= a.block_rows) return;  // waves are independent: no barrier anywhere
    auto slot = [&](int i) -> _Float16* { return (i == 0 ? s0 : i == 1 ? s1 : s2) + wave * BLOCK; };

    const __amdgpu_buffer_rsrc_t rec_b = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16*>(a.B), static_cast<short>(a.N * 2), a.K, kBufWord3);
    const __amdgpu_buffer_rsrc_t rec_a = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16*>(a.vals), static_cast<short>(512), a.num_blocks, kBufWord3);

    // Load c of a block fills rows 8c .. 8c+7 of the slot, lane l row l / 8 of
    // them and 16-byte position l % 8, which holds chunk l % 8 ^ swz (rows 8
    // apart swizzle alike): the eight rows that half a wave reads at once then
    // lie on all banks.  Columns past N read a valid chunk and are not stored.
    auto swz = [](int r) { return 2 * ((r >> 1) & 3); };
    const int srow  = lane >> 3;
    const int n     = n0 + ((lane & 7) ^ swz(srow)) * 8;
    const int nbyte = (n < a.N ? n : 0) * 2;
    // B operand: rows 4g .. 4g+3, column t of each tile; A operand: row t,
    // columns 4g .. 4g+3.
    const int brow = 4 * g + (t >> 2);
    const int h    = swz(brow) >> 1;
    const int in   = brow * 64 + ((t & 3) >> 1) * 8 + (t & 1) * 4;  // fp16 units
    const int a_off = t * 32 + 8 * g;

    const int bs = a.row_ptr[br];
    const int be = a.row_ptr[br + 1];
    f32x4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] = f32x4(0.0f);
    u32x2 af[3];

    for (int c0 = bs; c0 < be; c0 += 64) {  // 64 blocks per column-index chunk
        const int cnt = min(64, be - c0);
        const int ci  = lane < cnt ? a.col_idx[c0 + lane] : 0;
        auto load = [&](int q, int k) {  // block c0 + q into slot k
            const int bc  = __builtin_amdgcn_readlane(ci, q);
            _Float16* dst = slot(k);
            sbuf_load_lds(rec_b, (spmm_lds_ptr)dst, 16, bc * 16 + srow, nbyte, 0, 0, 0);
            sbuf_load_lds(rec_b, (spmm_lds_ptr)(dst + 512), 16, bc * 16 + 8 + srow, nbyte, 0, 0, 0);
            af[k] = sbuf_load_u32x2(rec_a, c0 + q, a_off, 0, 0);
        };
        auto multiply = [&](int k) {
            const f16x4 afv = __builtin_bit_cast(f16x4, af[k]);
            const _Float16* st = slot(k);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const s16x4 b = lds_read_tr16(st + in + (j ^ h) * 16);
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x16f16(afv, __builtin_bit_cast(f16x4, b),
                                                               acc[j], 0, 0, 0);
            }
        };
        // The loads of the two blocks after q, three each, may still be under
        // way when q is multiplied (loads retire in issue order).
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (k < cnt) load(k, k);
        }
        int q0 = 0;
        for (; q0 + 5 < cnt; q0 += 3) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                wait_vmcnt<6>();
                multiply(k);
                load(q0 + k + 3, k);
            }
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) {  // the last 1 .. 5 blocks
            if (q0 + k < cnt) {
                if (q0 + k + 2 < cnt) wait_vmcnt<6>();
                else if (q0 + k + 1 < cnt) wait_vmcnt<3>();
                else wait_vmcnt<0>();
                multiply(k % 3);
                if (q0 + k + 3 < cnt) load(q0 + k + 3, k % 3);
            }
        }
    }

    // D layout: lane holds rows 4*g + i, column t of each 16-column tile.
    const int rows_here = min(16, a.M - br * 16);
    if (a.c_vec_ok) {
        // As in the record kernel, two tiles through a slot at a time: 16 rows of
        // 32 floats, stored as 128-byte row pieces.
        const __amdgpu_buffer_rsrc_t c_rows = __builtin_amdgcn_make_buffer_rsrc(
            a.C + static_cast<size_t>(br) * 16 * a.N, static_cast<short>(0),
            rows_here * a.N * 4, kBufWord3);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float* ct = reinterpret_cast<float*>(slot(h));
#pragma unroll
            for (int j = 0; j < 2; ++j) {
#pragma unroll
                for (int i = 0; i < 4; ++i) ct[(4 * g + i) * 32 + 16 * j + t] = acc[2 * h + j][i];
            }
            const int col = n0 + 32 * h + (lane & 7) * 4;  // N % 8 == 0: all in or all out
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int r   = s * 8 + (lane >> 3);
                const f32x4 v = *reinterpret_cast<const f32x4*>(ct + r * 32 + (lane & 7) * 4);
                if (r < rows_here && col < a.N) {
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), c_rows,
                                                           (r * a.N + col) * 4, 0, kStoreDevice);
                }
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int col = n0 + 16 * j + t;
        if (col >= a.N) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = br * 16 + 4 * g + i;
            if (row < a.M) store_c(a.C + static_cast<size_t>(row) * a.N + col, acc[j][i]);
        }
    }
}

// One launch for wide B and 24 - 64 blocks per block-row: the shared panel
// where A's blocks lie in runs, and waves (the same 4 block-rows x 64 columns a
// workgroup, in column slices) where they lie all over: a panel's union then
// nears the sum of its lists, and its lockstep pairs bound it.  The panel's
// stages lie in the waves' slots.  PAIRS: the waves are the record kernel's, whose
// 32 KiB of slots leave a CU four workgroups; else bsr_wide_waves and five.
constexpr int kWideTables = 4 * (2 * kPanelMaxWords + kPanelSlots * 5 + 8) + 8 * 16;  // bytes
constexpr bool cu_holds(int workgroups, int lds_bytes) {  // LDS: 160 KiB, given out in 1280 bytes
    return workgroups * ((lds_bytes + 1279) / 1280) <= 128;
}
static_assert(cu_holds(4, 4 * 2 * 4096 + kWideTables + 16) && cu_holds(5, 4 * 3 * 2048 + kWideTables),
              "resident workgroups of the two forms of bsr_wide_kernel");

template <bool PAIRS>
__global__ __launch_bounds__(256) void bsr_wide_kernel(BsrArgs a) {
    constexpr int R = 4, J = 4, STAGE = 32 * 16 * J, SLOT = PAIRS ? 4 * STAGE : 2 * STAGE;
    __shared__ __attribute__((aligned(16))) _Float16 s_b0[SLOT];
    __shared__ __attribute__((aligned(16))) _Float16 s_b1[SLOT];
    __shared__ __attribute__((aligned(16))) _Float16 s_b2[PAIRS ? 8 : SLOT];
    __shared__ uint32_t s_bits[kPanelMaxWords];
    __shared__ int s_pre[kPanelMaxWords];
    __shared__ int s_ucol[kPanelSlots];
    __shared__ int s_blk[kPanelSlots * R];
    __shared__ uint64_t s_mask[4 * R];
    __shared__ int s_misc[8];
    // two stages: the other two are never touched
    if (!bsr_panel_body<R, J, 4, 2, true>(a, s_b0, s_b1, s_b2, s_b2, s_bits, s_pre, s_ucol, s_blk,
                                          s_mask, s_misc)) {
        if constexpr (PAIRS) {
            bsr_record_body<J, 2>(a, a.slices, s_b0, s_b1, s_b2, s_b2);
        } else {
            bsr_wide_waves(a, a.slices, s_b0, s_b1, s_b2);
        }
    }
}

Error fail(int status, std::string msg) { return Error{status, std::move(msg)}; }

Error from_hip(hipError_t e, const char* what) {
    if (e == hipSuccess) return Error{};
    return fail(kHipError, std::string(what) + ": " + hipGetErrorString(e));
}

// Workgroups of 256 threads: HIP 7.0 takes a launch of 2^32 threads and more without
// an error and runs none or a part of it.
constexpr long kMaxGroups = 0xffffffffL / 256;

// B rows and A blocks fit structured-buffer records: the record stride field
// holds at most 16383 bytes and each buffer must stay within 2 GiB.
bool records_fit(const BsrArgs& a) {
    return a.b_vec_ok && static_cast<long long>(a.N) * 2 <= 16383 &&
           static_cast<long long>(a.K) * a.N * 2 <= 0x7fffffffLL &&
           static_cast<long long>(a.num_blocks) * 512 <= 0x7fffffffLL;
}

// Column slices for blocks that lie in no runs: as many (a power of two, at
// most 8, splitting the tiles to within 15%) as bring an XCD's share of B to
// about 3 MiB, which leaves its L2 room for A and C.  Each slice reads A again,
// which costs little next to B's rows from 8 blocks per block-row on; up to 5
// MiB B mostly stays in the L2s whole.  Below one block in 64 A is more likely a
// band, which gains nothing and would pay for looking (32768 rows of 15 blocks, N
// = 512: 31 -> 33 us).
// 12288^2 at 2%: N = 512 28.2 -> 20.0 us, N = 1024 57 -> 33 us.
int record_slices(const BsrArgs& a) {
    const long long b_bytes = 2LL * a.K * a.N;
    if (a.xcd_order == 0 || b_bytes <= (5LL << 20) || a.num_blocks < 8LL * a.block_rows ||
        64LL * a.num_blocks < static_cast<long long>(a.block_rows) * a.block_cols) {
        return 1;
    }
    int s = 1;
    while (s < 8 && b_bytes > s * (3LL << 20)) s *= 2;
    while (s > 1 && 100L * ceil_div(a.tiles_n, s) * s > 115L * a.tiles_n) s /= 2;
    return s;
}

// Workgroups of a grid that takes either of wave_tile_of's orders.
unsigned grid_size(const BsrArgs& a) {
    if (a.slices == 1) return static_cast<unsigned>(a.wg_total);
    const int rows = ceil_div(ceil_div(a.block_rows, 4), 8 / a.slices);
    const unsigned sliced = 8u * static_cast<unsigned>(rows) * ceil_div(a.tiles_n, a.slices);
    return std::max(sliced, static_cast<unsigned>(a.wg_total));
}

// Sets the column slices of tiles_n and wg_total and returns the grid.
unsigned slice_grid(BsrArgs& a) {
    a.slices = record_slices(a);
    if (grid_size(a) > kMaxGroups) a.slices = 1;
    return grid_size(a);
}

template <int J, int D>
hipError_t run_wave(BsrArgs args, hipStream_t stream, bool pointer_addressing) {
    args.tiles_n = ceil_div(args.N, 16 * J);
    const long total = static_cast<long>(ceil_div(args.block_rows, 4)) * args.tiles_n;
    if (total > kMaxGroups) return hipErrorInvalidConfiguration;
    args.wg_total = static_cast<int>(total);
    const unsigned tiles = slice_grid(args);
    if (!pointer_addressing && records_fit(args)) {
        constexpr int DEPTH = D == 1 ? 2 : D;
        if (args.slices > 1) {
            hipLaunchKernelGGL((bsr_record_kernel<J, DEPTH, true>), dim3(tiles), dim3(256), 0,
                               stream, args);
        } else {
            hipLaunchKernelGGL((bsr_record_kernel<J, DEPTH, false>), dim3(tiles), dim3(256), 0,
                               stream, args);
        }
        return hipGetLastError();
    }
    if (args.b_vec_ok) {
        hipLaunchKernelGGL((bsr_wave_kernel<J, D, Chunks::Aligned>), dim3(args.wg_total), dim3(256),
                           0, stream, args);
    } else if (static_cast<long long>(args.K) * args.N >= 8) {
        hipLaunchKernelGGL((bsr_wave_kernel<J, D, Chunks::Any>), dim3(args.wg_total), dim3(256), 0,
                           stream, args);
    } else {  // B is smaller than one chunk
        args.tiles_n  = 1;
        args.wg_total = ceil_div(args.block_rows, 4);
        hipLaunchKernelGGL((bsr_wave_kernel<1, 1, Chunks::Elements>), dim3(args.wg_total), dim3(256), 0,
                           stream, args);
    }
    return hipGetLastError();
}

template <int J>
hipError_t dispatch_wave(int depth, bool pointer_addressing, const BsrArgs& args,
                         hipStream_t stream) {
    return depth == 1 ? run_wave<J, 1>(args, stream, pointer_addressing)
                      : (depth == 2 ? run_wave<J, 2>(args, stream, pointer_addressing)
                                    : run_wave<J, 4>(args, stream, pointer_addressing));
}

template <int R, int J, int WR, int D>
hipError_t run_panel(BsrArgs args, hipStream_t stream) {
    args.tiles_n = ceil_div(args.N, 16 * J);
    const long total = static_cast<long>(ceil_div(args.block_rows, R)) * args.tiles_n;
    if (total > kMaxGroups) return hipErrorInvalidConfiguration;
    args.wg_total = static_cast<int>(total);
    hipLaunchKernelGGL((bsr_panel_kernel<R, J, WR, D>), dim3(args.wg_total), dim3(256), 0, stream,
                       args);
    return hipGetLastError();
}

// Workgroups up to which the wide kernel's waves take pairs: four per CU.  The
// panel loses nothing to 32 KiB of slots then and the waves gain (MI355X, blocks
// at 12.5% of 8192^2, N = 512 40.3 -> 37.0 us; 3000 x 6997 at 10%, N = 512 15.5 -> 13.8);
// beyond, the panel of five workgroups a CU would lose up to 1.55x to four (bands
// of 8192 rows, half-bandwidth 480, N = 640 22.5 against 34.5 us, the waves gain 1.17x
// at most: 16384 x 8192 at 6%, N = 512 43.2 against 36.9).
constexpr int kPairsMaxGroups = 1024;

hipError_t run_wide(BsrArgs args, hipStream_t stream) {
    args.tiles_n = ceil_div(args.N, 64);
    const long total = static_cast<long>(ceil_div(args.block_rows, 4)) * args.tiles_n;
    if (total > kMaxGroups) return hipErrorInvalidConfiguration;
    args.wg_total = static_cast<int>(total);
    const unsigned grid = slice_grid(args);
    if (args.wg_total <= kPairsMaxGroups) {
        hipLaunchKernelGGL(bsr_wide_kernel<true>, dim3(grid), dim3(256), 0, stream, args);
    } else {
        hipLaunchKernelGGL(bsr_wide_kernel<false>, dim3(grid), dim3(256), 0, stream, args);
    }
    return hipGetLastError();
}

// Panel shapes: R block-rows x 16J columns per workgroup, each wave four
// 16-column tiles (waves 4 x 1 for J = 4, 2 x 2 for J = 8).
// Stages in flight: 2 or 4.
template <int R, int J>
hipError_t dispatch_panel(int depth, const BsrArgs& args, hipStream_t stream) {
    constexpr int WR = J == 4 ? 4 : 2;
    return depth <= 2 ? run_panel<R, J, WR, 2>(args, stream) : run_panel<R, J, WR, 4>(args, stream);
}

}  // namespace

Error launch_float_to_half(const float* src, half* dst, long n, hipStream_t stream) {
    if (n < 0) return fail(kInvalid, "negative element count");
    if (n == 0) return Error{};
    if (src == nullptr || dst == nullptr) return fail(kInvalid, "null device pointer");
    const bool vec = (reinterpret_cast<uintptr_t>(src) % 16 == 0) &&
                     (reinterpret_cast<uintptr_t>(dst) % 16 == 0);
    const long threads = vec ? (n + 7) / 8 : n;
    const long blocks = (threads + 255) / 256;
    if (blocks > 0x7fffffffL) return fail(kInvalid, "element count too large");
    hipLaunchKernelGGL(f32_to_f16_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                       stream, src, reinterpret_cast<_Float16*>(dst), n, vec ? 1 : 0);
    return from_hip(hipGetLastError(), "float_to_half launch");
}

Error launch_bsr(const BSR& A, const half* B, float* C, int N, hipStream_t stream,
                 const BsrOpts* opts) {
    if (A.num_rows < 0 || A.num_cols < 0 || A.num_blocks < 0 || N < 0) {
        return fail(kInvalid, "negative matrix dimension");
    }
    if (A.block_rows != (A.num_rows + 15) / 16 || A.block_cols != (A.num_cols + 15) / 16) {
        return fail(kInvalid, "BSR block dimensions do not match num_rows / num_cols");
    }
    if (A.num_rows == 0 || N == 0) return Error{};
    if (A.row_ptr == nullptr || C == nullptr || B == nullptr) {
        return fail(kInvalid, "null device pointer");
    }
    if (A.num_blocks > 0 && (A.col_idx == nullptr || A.values == nullptr)) {
        return fail(kInvalid, "null device pointer");
    }
    if (reinterpret_cast<uintptr_t>(A.values) % 16 != 0) {
        return fail(kInvalid, "BSR values must be 16-byte aligned");
    }
    BsrArgs args{A.row_ptr,
                 A.col_idx,
                 reinterpret_cast<const _Float16*>(A.values),
                 reinterpret_cast<const _Float16*>(B),
                 C,
                 A.num_rows,
                 A.num_cols,
                 N,
                 A.block_rows,
                 (N % 8 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0) ? 1 : 0,
                 A.block_cols,
                 0,
                 0,
                 0,
                 std::max(A.num_blocks - 8, 0) / 7,
                 1,
                 A.num_blocks,
                 reinterpret_cast<uintptr_t>(C) % 16 == 0 ? 1 : 0};
    const BsrOpts o = opts ? *opts : BsrOpts{};
    if (o.row_group != 0 && o.row_group != 1 && o.row_group != 4 && o.row_group != 8) {
        return fail(kInvalid, "row_group must be 0, 1, 4 or 8");
    }
    // Option values no kernel has are refused; with the kernel chosen
    // explicitly (row_group 1 / per_wave, row_group 4 / 8) so are the values
    // that kernel lacks.  Under the automatic choice a value the chosen kernel
    // lacks takes that kernel's default.
    const auto one_of = [](int v, std::initializer_list<int> ok) {
        for (int x : ok) {
            if (v == x) return true;
        }
        return false;
    };
    if (!one_of(o.tiles, {0, 1, 2, 4, 8}) || !one_of(o.depth, {0, 1, 2, 4})) {
        return fail(kInvalid, "tiles must be 0, 1, 2, 4 or 8 and depth 0, 1, 2 or 4");
    }
    const bool panel_forced = !o.per_wave && (o.row_group == 4 || o.row_group == 8);
    const bool wave_forced = o.per_wave || o.row_group == 1;
    if (panel_forced && (!one_of(o.tiles, {0, 4, 8}) || !one_of(o.depth, {0, 2, 4}))) {
        return fail(kInvalid, "shared-panel kernel: tiles must be 0, 4 or 8 and depth 0, 2 or 4");
    }
    if (wave_forced && o.tiles == 8) {
        return fail(kInvalid, "wave kernel: tiles must be 0, 1, 2 or 4");
    }
    args.xcd_order = o.xcd_order == 2 ? 0 : 1;
    hipError_t e;
    const bool rec = o.addressing != 1 && records_fit(args);
    const double bpr = A.block_rows > 0 ? static_cast<double>(A.num_blocks) / A.block_rows : 0.0;
    // Shared-panel kernel (R = 4, 64 columns, 2 stages): automatic on wide B
    // with long block-rows, where it measured faster than the wave kernel on
    // structured inputs (N >= 256, 24 - 64 blocks per block-row: 1.03 - 1.31x
    // over 36 block-diagonal and banded inputs); explicit row_group 4 / 8
    // forces it.  From one block in 24 on A may as well have no structure, and
    // then the panel takes 1.6 - 3.4 times the waves' time, so each launch looks
    // (bsr_wide_kernel; against the panel: blocks at 12.5% of 8192^2, N = 512 61 ->
    // 38 us and N = 1024 119 -> 77; 3000 x 6997 at 10%, N = 512 42 -> 14; bands and
    // diagonal blocks 0 - 0.3 us more), except on up to one workgroup a CU: there
    // the waves win on structured A too (bands of 4096 rows, N = 256 7.2 -> 5.0 us,
    // diagonal blocks of 1024 11.2 -> 7.7; at 320 workgroups 12.0 against 12.5).
    // Sparser A keeps the panel: bands of 16384 rows, N = 256 take 15.0 us there,
    // 16.8 with waves.
    const bool panel_auto = rec && N >= 256 && A.block_cols <= kPanelMaxWords * 32 &&
                            bpr >= 24.0 && bpr <= 64.0;
    const bool dense = 24.0 * bpr >= A.block_cols;
    const bool defaults = !o.per_wave && o.row_group == 0 && o.tiles == 0 && o.depth == 0;
    const long panel_groups = static_cast<long>(ceil_div(A.block_rows, 4)) * ceil_div(N, 64);
    if (panel_auto && dense && defaults && panel_groups > 256) {
        return from_hip(run_wide(args, stream), "spmm_wmma launch");
    }
    const bool panel = !o.per_wave && rec &&
                       (o.row_group == 4 || o.row_group == 8 ||
                        (o.row_group == 0 && panel_auto && !(dense && defaults)));
    if (panel) {
        const int R = o.row_group == 8 ? 8 : 4;
        const int j = o.tiles == 8 ? 8 : 4;
        const int d = o.depth == 4 ? 4 : 2;  // 0 (or a wave-only 1 when automatic): 2
        if (R == 4) {
            e = j == 4 ? dispatch_panel<4, 4>(d, args, stream) : dispatch_panel<4, 8>(d, args, stream);
        } else {
            e = j == 4 ? dispatch_panel<8, 4>(d, args, stream) : dispatch_panel<8, 8>(d, args, stream);
        }
        return from_hip(e, "spmm_wmma launch");
    }
    // Defaults of the wave kernel, from a sweep of 92 MI355X runs (uniform,
    // banded, block-diagonal and power-law, M = 4096 .. 16384, N = 64 .. 512).
    // Four 16-column tiles per wave halve the A-block re-reads of two tiles
    // and win once the grid still has >= 1024 waves at four tiles, unless
    // block-rows are short (< 12 blocks) and the grid is under 2048 waves:
    // then the extra waves of two tiles hide more latency (e.g. uniform
    // 8192^2 density 0.01 N=128: 67 -> 48 us).  Four pairs in flight pay on
    // long block-rows: >= 30 blocks at two tiles, >= 96 at four (uniform
    // 4096^2 density 0.01 N=128: 26.4 -> 20.3 us).  The pointer-arithmetic form
    // (widths that are no multiple of 8, B off 16 bytes, buffers past 2 GiB)
    // stages through registers: four tiles pay from 2048 waves on, with one
    // pair in flight (8192^2 blocks at 12.5%, N = 500: 46 us against 75 with two
    // tiles and 52 with two pairs; at 1024 waves 52 against 35), and one tile
    // below 512 waves of two (2000^2, N = 36: 4.1 against 5.1 us).  Where its chunks
    // are aligned four tiles need N >= 256 and 12 blocks per block-row besides
    // (8192^2 at 12.5%, N = 512 73 -> 42 us; N = 128 15.2 against 24, bands of 5 blocks,
    // N = 256 6.4 against 7.1).
    const long waves4 = static_cast<long>(A.block_rows) * ((N + 63) / 64);
    const long waves2 = static_cast<long>(A.block_rows) * ((N + 31) / 32);
    const bool ptr4 = waves4 >= 2048 && (!args.b_vec_ok || (N >= 256 && bpr >= 12.0));
    const int j_auto =
        N <= 16 ? 1
        : rec   ? ((waves4 >= 1024 && (bpr >= 12.0 || waves4 >= 2048)) ? 4 : 2)
                : (ptr4 ? 4 : (waves2 >= 512 ? 2 : 1));
    const int j = (o.tiles == 1 || o.tiles == 2 || o.tiles == 4) ? o.tiles : j_auto;
    const int d_auto = rec ? (bpr >= (j == 4 ? 96.0 : 30.0) ? 4 : 2) : (j == 4 ? 1 : 2);
    const int d = (o.depth == 1 || o.depth == 2 || o.depth == 4) ? o.depth : d_auto;
    const bool ptr = o.addressing == 1;
    e = j == 1 ? dispatch_wave<1>(d, ptr, args, stream)
               : (j == 2 ? dispatch_wave<2>(d, ptr, args, stream)
                         : dispatch_wave<4>(d, ptr, args, stream));
    return from_hip(e, "spmm_wmma launch");
}

}  // namespace engine
}  // namespace spmm
