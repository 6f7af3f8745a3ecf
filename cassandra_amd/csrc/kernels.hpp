// HIP kernels of the pattern-evaluator fit (gfx950 / CDNA4).
//
// Layout of a stored matrix (fixed k entries per row, implicit value 1):
//   slot-major: idx[s * ld + r], r < rows, s < k, column = sys_base + base[s] + idx
//   (u16 when every slot's column range is narrower than 65536, else u32).
// Every row-parallel kernel walks a RowWork list, every column-parallel kernel a
// ColWork list and the scatter kernels ScatterWork / ReduceWork lists, so one
// launch covers any number of independent systems (block-diagonal batches).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "board.hpp"
#include "device.hpp"

namespace cad {
// Kernels have internal linkage: every translation unit instantiates the ones
// it launches.
namespace {

constexpr int kRowBlock = 256;   // threads of the row / column kernels
constexpr int kRowsPerThread = 4;  // rows per thread of the generic row work
constexpr int kScatterBlock = 1024;

// ------------------------------------------------------------ index views --
template <class IdxT>
struct SlotMajor {
    using index_type = IdxT;
    const IdxT* __restrict__ idx;
    int64_t ld;
    const uint32_t* __restrict__ base;  // per slot
    __device__ __forceinline__ uint32_t col(int s, int64_t r) const
    {
        return base[s] + uint32_t(idx[int64_t(s) * ld + r]);
    }
    // Slot s's entries, for a loop over rows (s the same for the whole wave:
    // the pointer and base stay in scalar registers, and the rows' loads of
    // several slots can all be in flight together).
    struct Slot {
        const IdxT* __restrict__ p;
        uint32_t base;
        __device__ __forceinline__ uint32_t col(int64_t r) const { return base + uint32_t(p[r]); }
    };
    __device__ __forceinline__ Slot slot(int s) const
    {
        return Slot{idx + int64_t(s) * ld, uint32_t(__builtin_amdgcn_readfirstlane(base[s]))};
    }
};

template <class View>
struct is_slot_major : std::false_type {};
template <class IdxT>
struct is_slot_major<SlotMajor<IdxT>> : std::true_type {};
template <class View>
struct SlotRefOf {
    using type = int;
};
template <class IdxT>
struct SlotRefOf<SlotMajor<IdxT>> {
    using type = typename SlotMajor<IdxT>::Slot;
};

// ------------------------------------------------------------ reductions ---
__device__ __forceinline__ double wave_sum(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Sum over the block; the result is valid in thread 0.
template <int BS>
__device__ __forceinline__ double block_sum(double v, double* sh)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) sh[wid] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < BS / 64; i++) t += sh[i];
    return t;
}

// Single-pass grid reduction: every block of a system stores its partial, the
// last block to arrive (ticket on the system's counter) sees all partials and
// returns true.  The counter is re-armed by that last block, so the kernel can
// be replayed (graphs) without clearing it.
__device__ __forceinline__ bool arrive_last(unsigned* counter, unsigned nblocks)
{
    __shared__ bool last;
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        unsigned t = atomicAdd(counter, 1u);
        last = (t == nblocks - 1);
        if (last) atomicExch(counter, 0u);
    }
    __syncthreads();
    if (last) __threadfence();
    return last;
}

// Sum of one system's block partials (slot 0), returned to every thread:
// each thread adds its strided share in block order, then the block's fixed
// reduction tree, so every block that forms the sum gets the same value.
template <int BS>
__device__ __forceinline__ double system_sum(const GridSys& g, int sys, double* sh)
{
    double s = 0.0;
    const int first = g.blk_first[sys], n = g.blk_count[sys];
    for (int i = threadIdx.x; i < n; i += BS) s += g.partials[2 * (first + i)];
    s = block_sum<BS>(s, sh);
    if (threadIdx.x == 0) sh[0] = s;
    __syncthreads();
    return sh[0];
}

// The same for both slots of the partials.
template <int BS>
__device__ __forceinline__ void system_sum2(const GridSys& g, int sys, double* sh, double& s0, double& s1)
{
    double a0 = 0.0, a1 = 0.0;
    const int first = g.blk_first[sys], n = g.blk_count[sys];
    for (int i = threadIdx.x; i < n; i += BS) {
        a0 += g.partials[2 * (first + i)];
        a1 += g.partials[2 * (first + i) + 1];
    }
    a0 = block_sum<BS>(a0, sh);
    a1 = block_sum<BS>(a1, sh);
    if (threadIdx.x == 0) {
        sh[0] = a0;
        sh[1] = a1;
    }
    __syncthreads();
    s0 = sh[0];
    s1 = sh[1];
}

// ------------------------------------------------------------ fill --------
template <class T>
__global__ void k_fill(T* __restrict__ p, int64_t n, T v)
{
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        p[i] = v;
}

template <class TO, class TI>
__global__ void k_convert(TO* __restrict__ out, const TI* __restrict__ in, int64_t n)
{
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        out[i] = TO(in[i]);
}

// ------------------------------------------------------------ index --------
// Pattern/Indexer.cpp InsertIndices for every row: one thread per position.
// out[s * slot_stride + r * row_stride] = (local ? 0 : col_offset) + index.
__device__ __forceinline__ uint32_t list_value(const uint8_t* __restrict__ sq, int off, int len,
                                               uint64_t P, uint64_t O)
{
    // the square numbers are the same for the whole wave: read them as 32-bit
    // words (scalar loads; the array is padded to whole words) and take the
    // byte, rather than one vector byte load per square
    const uint32_t* __restrict__ w = reinterpret_cast<const uint32_t*>(sq);
    uint32_t v = 0;
    for (int j = len - 1; j >= 0; --j) {
        const int b = off + j;
        const int q = int((w[b >> 2] >> (8 * (b & 3))) & 0xFFu);
        v = v * 3u + uint32_t((P >> q) & 1u) + 2u * uint32_t((O >> q) & 1u);
    }
    return v;
}

__device__ __forceinline__ uint32_t slot_index(const DevSlot& s, const uint8_t* __restrict__ sq,
                                               const uint32_t* __restrict__ dense, uint64_t P, uint64_t O)
{
    const uint32_t a = list_value(sq, s.off[0], s.len[0], P, O);
    if (s.kind == 0) return a;
    if (s.kind == 3) return dense[s.dense_offset + a];
    const uint32_t b = list_value(sq, s.off[1], s.len[1], P, O);
    const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
    uint32_t idx = lo * s.hs + hi - lo * (lo + 1u) / 2u;
    if (s.kind == 2) idx = idx * s.ds + list_value(sq, s.off[2], s.len[2], P, O);
    return idx;
}

// The four ternary words of a position: square q's digit P_q + 2 O_q in bits
// 2 (q mod 16) of word q / 16 (each 16-bit half-board's bits spread to every
// other bit).
__device__ __forceinline__ uint32_t spread16(uint32_t x)
{
    x &= 0xFFFFu;
    x = (x | (x << 8)) & 0x00FF00FFu;
    x = (x | (x << 4)) & 0x0F0F0F0Fu;
    x = (x | (x << 2)) & 0x33333333u;
    x = (x | (x << 1)) & 0x55555555u;
    return x;
}

__device__ __forceinline__ void ternary_words(uint64_t P, uint64_t O, uint32_t (&T)[4])
{
#pragma unroll
    for (int w = 0; w < 4; w++)
        T[w] = spread16(uint32_t(P >> (16 * w))) | (spread16(uint32_t(O >> (16 * w))) << 1);
}

// Read-only memory at a wave-uniform address through the constant address
// space: scalar loads into scalar registers.  Only for arrays no kernel
// writes (programs uploaded before the launch).  Scalar loads and LDS
// operations share one wait counter, so a wait for one waits for the other.
typedef const __attribute__((address_space(4))) uint32_t* ConstWords;

// A descriptor that is the same for the whole wave, read as whole 32-bit
// words into scalar registers (a struct with byte or half-word fields would
// otherwise be read with vector loads and full waits).  Vector loads and
// lane-to-scalar moves: their wait does not also wait for the LDS operations
// in flight, as a scalar load's would.
template <class T>
__device__ __forceinline__ T uniform_load(const T* p)
{
    static_assert(sizeof(T) % 4 == 0, "whole words");
    const uint32_t* __restrict__ w = reinterpret_cast<const uint32_t*>(p);
    uint32_t r[sizeof(T) / 4];
#pragma unroll
    for (int i = 0; i < int(sizeof(T) / 4); i++) r[i] = __builtin_amdgcn_readfirstlane(w[i]);
    T t;
    __builtin_memcpy(&t, r, sizeof(T));
    return t;
}

// A descriptor through the constant address space (scalar loads): for arrays
// no kernel writes, in kernels without LDS traffic to wait for.
template <class T>
__device__ __forceinline__ T constant_load(const T* p)
{
    static_assert(sizeof(T) % 4 == 0, "whole words");
    const ConstWords c = (ConstWords)(reinterpret_cast<const uint32_t*>(p));
    uint32_t r[sizeof(T) / 4];
#pragma unroll
    for (int i = 0; i < int(sizeof(T) / 4); i++) r[i] = c[i];
    T t;
    __builtin_memcpy(&t, r, sizeof(T));
    return t;
}

// Element i of a uint16 array the whole wave reads (the array is padded to
// whole 32-bit words).
__device__ __forceinline__ int uniform_u16(const uint16_t* p, int i)
{
    const uint32_t w = __builtin_amdgcn_readfirstlane(reinterpret_cast<const uint32_t*>(p)[i >> 1]);
    return int((w >> (16 * (i & 1))) & 0xFFFFu);
}

// The ternary words of n positions (a matrix-free matrix keeps them, so the
// products need not recompute them).
__global__ void k_ternary_rows(const uint64_t* __restrict__ pos, int64_t n, uint4* __restrict__ tw)
{
    for (int64_t r = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; r < n; r += int64_t(gridDim.x) * blockDim.x) {
        uint32_t T[4];
        ternary_words(pos[2 * r], pos[2 * r + 1], T);
        tw[r] = make_uint4(T[0], T[1], T[2], T[3]);
    }
}

// ------------------------------------------------------ index tiles --------
// A wave computes a tile's columns (IndexTile) for 64 rows with four matrix
// products of 16 positions each: lane (n, g) = (lane % 16, lane / 16) feeds
// the 16 digits of word g of position n (four registers, byte m of register v
// the digit of square 16 g + v + 4 m) and receives the four roles of slot g
// for position n.  Evaluating the square lists digit by digit took two vector
// instructions per square and about as many scalar ones (FIT12: 444 squares a
// row, 36 vector instructions per column); the products leave about 10.
typedef int Int4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ Int4 expand_digits(uint32_t t)
{
    return Int4{int(t & 0x03030303u), int((t >> 2) & 0x03030303u), int((t >> 4) & 0x03030303u),
                int((t >> 6) & 0x03030303u)};
}

// Lane (n, g)'s digits of row r, from the rows' ternary words tw[r] (word g).
__device__ __forceinline__ Int4 digits_of_words(const uint4* __restrict__ tw, int64_t r)
{
    return expand_digits(reinterpret_cast<const uint32_t*>(tw + r)[(threadIdx.x >> 4) & 3]);
}

// Four registers of 16-lane groups, transposed: register p
// holding slot g of position set p in lane group g becomes register j holding
// slot j of position set p in lane group p (lane = position).
__device__ __forceinline__ void transpose_groups(uint32_t (&r)[4])
{
    auto s01 = __builtin_amdgcn_permlane16_swap(r[0], r[1], false, false);
    auto s23 = __builtin_amdgcn_permlane16_swap(r[2], r[3], false, false);
    auto a = __builtin_amdgcn_permlane32_swap(s01[0], s23[0], false, false);
    auto b = __builtin_amdgcn_permlane32_swap(s01[1], s23[1], false, false);
    r[0] = a[0];
    r[1] = b[0];
    r[2] = a[1];
    r[3] = b[1];
}

// The digits of the wave's 64 rows, lane l's row r: every lane loads its own
// position, and the transposition hands word g of lane 16 p + n's row to lane (n, g)
// of set p (each lane loading the 16 bits of its words: extraction of 5M rows of
// FIT8 156 µs against 124, of 4 slots 79 against 30; 300,000 positions scored
// with 4 slots 7.6 against 5.3, with 18 slots 19.0 against 16.3).
__device__ __forceinline__ void digits_of_rows(const uint64_t* __restrict__ pos, int64_t r, Int4 (&b)[4])
{
    uint32_t T[4];
    ternary_words(pos[2 * r], pos[2 * r + 1], T);
    transpose_groups(T);
#pragma unroll
    for (int p = 0; p < 4; p++) b[p] = expand_digits(T[p]);
}

// Tile t's weights (two blocks of 64 a tile, the second for wide pairs with a
// diagonal).
__device__ __forceinline__ const Int4* tile_weights(int t, const TileView& tv)
{
    return reinterpret_cast<const Int4*>(tv.weights) + (128 * t + int(threadIdx.x & 63));
}

// The pattern-local column of slot g of the tile for the four position sets
// b[0..4) (idx[p]: lane (n, g) holds slot g of position n of set p; lanes of
// slots past the tile's hold column 0 of some configuration).
__device__ __forceinline__ void tile_columns(const IndexTile& t, int number, const TileView& tv, const Int4& w,
                                             const Int4 (&b)[4], uint32_t (&idx)[4])
{
    const Int4 zero = {0, 0, 0, 0};
    Int4 d[4];
#pragma unroll
    for (int p = 0; p < 4; p++) d[p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, b[p], zero, 0, 0, 0);
    if (t.kind == 0 || t.kind == 3) {
#pragma unroll
        for (int p = 0; p < 4; p++) idx[p] = uint32_t(d[p][0]) + __umul24(uint32_t(d[p][1]), 243u);
        if (t.wide) {
#pragma unroll
            for (int p = 0; p < 4; p++)
                idx[p] += __umul24(uint32_t(d[p][2]), 59049u) + __umul24(uint32_t(d[p][3]), 14348907u);
        }
        if (t.kind == 3) {
#pragma unroll
            for (int p = 0; p < 4; p++) idx[p] = tv.dense[t.dense_offset + idx[p]];
        }
        return;
    }
    uint32_t a[4], c[4];
#pragma unroll
    for (int p = 0; p < 4; p++) {
        a[p] = uint32_t(d[p][0]);
        c[p] = uint32_t(d[p][1]);
    }
    if (t.wide) {
        if (t.kind == 1) {
#pragma unroll
            for (int p = 0; p < 4; p++) {
                a[p] += __umul24(uint32_t(d[p][2]), 243u);
                c[p] += __umul24(uint32_t(d[p][3]), 243u);
            }
        } else {
            const Int4 w2 = tile_weights(number, tv)[64];
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const Int4 e = __builtin_amdgcn_mfma_i32_16x16x64_i8(w2, b[p], zero, 0, 0, 0);
                a[p] += __umul24(uint32_t(e[0]), 243u);
                c[p] += __umul24(uint32_t(e[1]), 243u);
            }
        }
    }
    // the pair's number, from the smaller and the larger half (below 3^8)
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const uint32_t lo = min(a[p], c[p]), hi = max(a[p], c[p]);
        idx[p] = __umul24(lo, t.hs) + hi - (__umul24(lo, lo + 1u) >> 1);
    }
    if (t.kind == 2) {
#pragma unroll
        for (int p = 0; p < 4; p++)
            idx[p] = __umul24(idx[p], t.ds) + uint32_t(d[p][2]) + __umul24(uint32_t(d[p][3]), 243u);
    }
}

// A tile's descriptor and weights on their way from memory, in vector registers
// (the descriptor the same in every lane): loaded a tile ahead, they are in
// flight while the tile before is used, and their wait is not one for the LDS.
struct TileRegs {
    Int4 desc[2];
    Int4 weights;
    __device__ __forceinline__ IndexTile tile() const
    {
        uint32_t r[8];
#pragma unroll
        for (int i = 0; i < 8; i++) r[i] = __builtin_amdgcn_readfirstlane(uint32_t(desc[i >> 2][i & 3]));
        IndexTile t;
        __builtin_memcpy(&t, r, sizeof(t));
        return t;
    }
};

__device__ __forceinline__ TileRegs load_tile(const TileView& tv, int t)
{
    TileRegs r;
    int v = 0;
    asm volatile("" : "+v"(v));  // a vector load
    const Int4* __restrict__ d = reinterpret_cast<const Int4*>(tv.tiles + t) + v;
    r.desc[0] = d[0];
    r.desc[1] = d[1];
    r.weights = *tile_weights(t, tv);
    return r;
}

// Pattern/Indexer.cpp InsertIndices for every row, slot-major: out[s * ld + r]
// = (local ? 0 : col_offset) + column, rows [n, nstore) as zeros.  A wave takes
// 64 C rows: where 2-byte entries are aligned in runs of C (vec), lane l has the
// C consecutive rows from its first + l C on, so that a slot's stores are C
// entries wide; else row l of each 64, a store's entries side by side (4-byte
// entries C apart or in runs took 1M rows of 4 slots 21 and 19 µs, 9.4 so).
// Bound by the stores: 5M rows of FIT8 as u16 take 124 µs for 420 MB, 240 (with
// the clear of the whole matrix that the padding rows cost) digit by digit;
// 100,000 rows of FIT4 8 against 36.
template <class OutT, int C>
__global__ __launch_bounds__(kRowBlock) void k_index_extract(const uint64_t* __restrict__ pos, int64_t n,
                                                             int64_t nstore, TileView tv, OutT* __restrict__ out,
                                                             int64_t ld, int local, int vec)
{
    const int lane = threadIdx.x & 63;
    const int64_t base = (blockIdx.x * int64_t(kRowBlock / 64) + (threadIdx.x >> 6)) * (64 * C);
    if (base >= nstore) return;
    // row c of lane l: l per_lane + c per_row from the wave's first
    const int per_lane = vec ? C : 1, per_row = vec ? 1 : 64;
    Int4 b[C][4];
    const int64_t r0 = base + int64_t(lane) * per_lane;
#pragma unroll
    for (int c = 0; c < C; c++) digits_of_rows(pos, min(r0 + c * per_row, n - 1), b[c]);
    for (int t = 0; t < tv.n; t++) {
        const IndexTile tl = constant_load(tv.tiles + t);
        const Int4 wt = *tile_weights(t, tv);
        const uint32_t off = local ? 0u : tl.col_offset;
        uint32_t v[C][4];
#pragma unroll
        for (int c = 0; c < C; c++) {
            tile_columns(tl, t, tv, wt, b[c], v[c]);
            transpose_groups(v[c]);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (j >= tl.nslots) break;
            OutT o[C];
#pragma unroll
            for (int c = 0; c < C; c++) o[c] = r0 + c * per_row < n ? OutT(off + v[c][j]) : OutT(0);
            OutT* __restrict__ dst = out + int64_t(tl.slot_first + j) * ld + r0;
            if (vec && r0 + C <= nstore) {
                struct alignas(sizeof(OutT) * C) Run {
                    OutT e[C];
                };
                Run run;
                __builtin_memcpy(&run, o, sizeof(run));
                *reinterpret_cast<Run*>(dst) = run;
            } else {
#pragma unroll
                for (int c = 0; c < C; c++)
                    if (r0 + c * per_row < nstore) dst[c * per_row] = o[c];
            }
        }
    }
}

// The same row-major (out[r * k + s], the global column).  A wave takes 64
// rows: the columns of a run of tiles (at most `chunk` slots) go into the
// wave's part of the LDS and from there to memory in row order, so that a
// store instruction writes consecutive words; one 4-byte store per column,
// rows apart, wrote partial lines.  With all slots in one chunk the 64 rows
// are one run of memory and leave in 16-byte stores (vec: out is aligned).
// 5M rows of FIT4: 117 µs for 440 MB (3.8 TB/s); 1,051 µs with the scattered
// stores.
__global__ __launch_bounds__(kRowBlock) void k_index_extract_rows(const uint64_t* __restrict__ pos, int64_t n,
                                                                  TileView tv, int k, int chunk, int pitch,
                                                                  uint32_t* __restrict__ out, int vec)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t* __restrict__ st = reinterpret_cast<uint32_t*>(smem_raw) + wave * 64 * pitch;
    const int64_t base = (blockIdx.x * int64_t(kRowBlock / 64) + wave) * 64;
    if (base >= n) return;
    const int rows = int(min<int64_t>(64, n - base));
    Int4 b[4];
    digits_of_rows(pos, min<int64_t>(base + lane, n - 1), b);
    uint32_t* __restrict__ dst = out + base * k;
    int first = 0;  // first slot of the chunk
    for (int t = 0; t < tv.n; t++) {
        const IndexTile tl = constant_load(tv.tiles + t);
        uint32_t v[4];
        tile_columns(tl, t, tv, *tile_weights(t, tv), b, v);
        const int g = lane >> 4;
        if (g < tl.nslots) {
#pragma unroll
            for (int p = 0; p < 4; p++)
                st[(16 * p + (lane & 15)) * pitch + (tl.slot_first - first) + g] = tl.col_offset + v[p];
        }
        const int end = tl.slot_first + tl.nslots;
        const int next = t + 1 < tv.n ? end + int(constant_load(tv.tiles + t + 1).nslots) : 0;
        if (t + 1 < tv.n && next - first <= chunk) continue;
        // the wave's LDS writes land before its reads (in order; the fence
        // keeps the compiler from moving them)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int nc = end - first;
        if (nc == k && pitch == k && vec) {
            const int total = rows * k, whole = total & ~3;
            for (int e = 4 * lane; e < whole; e += 256)
                *reinterpret_cast<uint4*>(dst + e) = *reinterpret_cast<const uint4*>(st + e);
            if (whole + lane < total) dst[whole + lane] = st[whole + lane];
        } else {
            // word e of the chunk is slot e % nc of row e / nc
            const int dr = 64 / nc, ds = 64 % nc;
            int r = lane / nc, s = lane % nc;
            while (r < rows) {
                dst[int64_t(r) * k + first + s] = st[r * pitch + s];
                r += dr;
                s += ds;
                if (s >= nc) {
                    s -= nc;
                    r++;
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        first = end;
    }
}

// Most slots a chunk of k_index_extract_rows holds in LDS (14 KB a wave), and
// the row pitch: the chunk itself where it holds all k slots (the LDS then has
// the layout of the memory), else odd.  (A chunk of 32 slots, whose rows start in
// the same LDS bank, takes 1M rows 41 µs, one of 34 slots 40.)
constexpr int kExtractChunk = 56;

// Matrix-free view of a pattern matrix: the column of slot s in row r is
// recomputed from the row's position (16 bytes) with the slot's program
// instead of being read from a stored index matrix.
struct PositionsView {
    using index_type = void;  // no stored indices
    const uint64_t* __restrict__ pos;
    const DevSlot* __restrict__ slots;
    const uint8_t* __restrict__ sq;
    const uint32_t* __restrict__ dense;
    const uint4* __restrict__ tw;        // every row's ternary words (computed once, at creation)
    TileView tiles;
    const uint32_t* __restrict__ slot_tiles;  // the index tile of every slot
    __device__ __forceinline__ int slot_tile(int s) const
    {
        return __builtin_amdgcn_readfirstlane(int(slot_tiles[s]));
    }
    __device__ __forceinline__ uint32_t col(int s, int64_t r) const
    {
        const DevSlot sl = slots[s];
        return sl.col_offset + slot_index(sl, sq, dense, pos[2 * r], pos[2 * r + 1]);
    }
};

// ------------------------------------------------------------ gathers ------
// y = A x with the in-row sum taken sequentially in slot order from zero, the
// order of Math/MatrixCSR.cpp:59-62 (bit-exact with it in FP32).  What is
// done with each row sum is an epilogue:
//   bool begin(sys)             per block; false skips the block (inactive system)
//   double row(r, acc)          store the row; returns its share of a reduction
//   void finish(sys, total)     last block of a system (kReduce only)
template <class VT>
struct EpiStore {
    VT* __restrict__ y;
    static constexpr bool kReduce = false;
    __device__ bool begin(int) { return true; }
    __device__ double row(int64_t r, VT a) { y[r] = a; return 0.0; }
    // RPT consecutive rows from a (a multiple of RPT), all of them valid:
    // 16-byte stores where y + a is 16-byte aligned
    template <int RPT>
    __device__ double rows(int64_t a, const VT (&acc)[RPT])
    {
        constexpr int Q = 16 / sizeof(VT);
        if constexpr (RPT % Q == 0) {
            if ((reinterpret_cast<uintptr_t>(y + a) & 15) == 0) {
                using V4 = std::conditional_t<sizeof(VT) == 4, float4, double2>;
#pragma unroll
                for (int i = 0; i < RPT; i += Q) {
                    V4 v;
                    __builtin_memcpy(&v, &acc[i], 16);
                    *reinterpret_cast<V4*>(y + a + i) = v;
                }
                return 0.0;
            }
        }
#pragma unroll
        for (int i = 0; i < RPT; i++) y[a + i] = acc[i];
        return 0.0;
    }
    __device__ void finish(int, double) {}
};

// LSQR step 1 (Math/Solver.h:161): u <- A v - alpha u.  u is kept unnormalised
// as u_raw with u = u_raw / beta; the gather source is vd = D v.  The new beta
// is |u_raw| (FP64 reduction).
template <class VT>
struct EpiLsqrU {
    VT* __restrict__ u;
    LsqrScalars* scal;
    VT f;
    static constexpr bool kReduce = true;
    static constexpr bool kFinishKernel = true;
    __device__ bool begin(int sys)
    {
        const LsqrScalars* st = &scal[sys];
        if (!st->active || st->stop) return false;
        const double beta = st->beta;
        f = VT(beta != 0.0 ? st->alpha / beta : 0.0);
        return true;
    }
    __device__ double row(int64_t r, VT a)
    {
        const VT v = a - f * u[r];
        u[r] = v;
        return double(v) * double(v);
    }
    // RPT consecutive valid rows from a: 16-byte loads and stores of u where
    // aligned; the squares add up in row order, as row() would
    template <int RPT>
    __device__ double rows(int64_t a, const VT (&acc)[RPT])
    {
        VT o[RPT];
        constexpr int Q = 16 / sizeof(VT);
        bool vec = false;
        if constexpr (RPT % Q == 0) vec = (reinterpret_cast<uintptr_t>(u + a) & 15) == 0;
        using V4 = std::conditional_t<sizeof(VT) == 4, float4, double2>;
        if constexpr (RPT % Q == 0) {
            if (vec) {
#pragma unroll
                for (int i = 0; i < RPT; i += Q) {
                    const V4 t = *reinterpret_cast<const V4*>(u + a + i);
                    __builtin_memcpy(&o[i], &t, 16);
                }
            }
        }
        if (!vec) {
#pragma unroll
            for (int i = 0; i < RPT; i++) o[i] = u[a + i];
        }
        double red = 0.0;
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            o[i] = acc[i] - f * o[i];
            red += double(o[i]) * double(o[i]);
        }
        if constexpr (RPT % Q == 0) {
            if (vec) {
#pragma unroll
                for (int i = 0; i < RPT; i += Q) {
                    V4 t;
                    __builtin_memcpy(&t, &o[i], 16);
                    *reinterpret_cast<V4*>(u + a + i) = t;
                }
                return red;
            }
        }
#pragma unroll
        for (int i = 0; i < RPT; i++) u[a + i] = o[i];
        return red;
    }
    // beta = |u_raw|; its square is kept for the rotation, which adds it to
    // the Frobenius estimate (as the scatter that forms beta itself does)
    __device__ void finish(int sys, double s)
    {
        scal[sys].beta = sqrt(s);
        scal[sys].beta2 = s;
    }
};

// FP64 residual of the original system: r = b - A x into r64, |r|^2 into
// reduce_a and beta = |r|; when u is given it also receives r converted to VT
// (the start vector of a refinement solve).
template <class VT>
struct EpiResidual {
    const double* __restrict__ b;
    double* __restrict__ r64;
    VT* __restrict__ u;
    LsqrScalars* scal;
    static constexpr bool kReduce = true;
    static constexpr bool kFinishKernel = true;
    __device__ bool begin(int sys) { return scal[sys].active != 0 && scal[sys].restart != 0; }
    __device__ double row(int64_t r, double a)
    {
        const double v = b[r] - a;
        r64[r] = v;
        if (u) u[r] = VT(v);
        return v * v;
    }
    template <int RPT>
    __device__ double rows(int64_t a, const double (&acc)[RPT])
    {
        double red = 0.0;
#pragma unroll
        for (int i = 0; i < RPT; i++) red += row(a + i, acc[i]);
        return red;
    }
    __device__ void finish(int sys, double s)
    {
        scal[sys].reduce_a = s;
        scal[sys].beta = sqrt(s);
        scal[sys].anorm2 = 0.0;
    }
};

// b = clip(2 * floor((A x_true + sn * N) / 2 + 1/2), -64, 64)
struct EpiTargets {
    double* __restrict__ b;
    uint64_t seed;
    double sn;
    static constexpr bool kReduce = false;
    __device__ bool begin(int) { return true; }
    __device__ double row(int64_t r, double a)
    {
        Stream rng(seed, uint64_t(r));
        const double v = __dadd_rn(a, __dmul_rn(sn, rng.ih12()));
        const double e = 2.0 * floor(v * 0.5 + 0.5);
        b[r] = fmin(64.0, fmax(-64.0, e));
        return 0.0;
    }
    template <int RPT>
    __device__ double rows(int64_t a, const double (&acc)[RPT])
    {
        double red = 0.0;
#pragma unroll
        for (int i = 0; i < RPT; i++) red += row(a + i, acc[i]);
        return red;
    }
    __device__ void finish(int, double) {}
};

// Block reduction of the epilogue shares, then the per-system grid finish.
// An epilogue with kFinishKernel only stores its block partials; the
// per-system finish runs in k_epi_finish, the next launch.  That avoids the
// device-scope fences of the last-block ticket (on gfx950 an L2 write-back
// and invalidate in every block), which the tile gather pays once per tile.
template <class Epi>
constexpr bool finish_kernel()
{
    if constexpr (Epi::kReduce)
        return Epi::kFinishKernel;
    else
        return false;
}

template <int BS, class Epi>
__device__ __forceinline__ void reduce_tail(Epi& epi, double acc, int sys, const GridSys& g)
{
    if constexpr (Epi::kReduce) {
        __shared__ double sh[BS / 64];
        acc = block_sum<BS>(acc, sh);
        if (threadIdx.x == 0) g.partials[2 * blockIdx.x] = acc;
        if constexpr (finish_kernel<Epi>()) return;
        if (arrive_last(&g.counters[sys], g.blk_count[sys])) {
            double s = 0.0;
            for (int i = threadIdx.x; i < g.blk_count[sys]; i += BS) s += g.partials[2 * (g.blk_first[sys] + i)];
            s = block_sum<BS>(s, sh);
            if (threadIdx.x == 0) epi.finish(sys, s);
        }
    }
}

// One block per system: the sum of the system's block partials (the order
// of the last-block ticket's sum) handed to the epilogue's finish.  Systems
// whose gather blocks returned early (begin() false) are skipped the same way.
template <class Epi>
__global__ __launch_bounds__(kRowBlock) void k_epi_finish(Epi epi, GridSys g)
{
    __shared__ double sh[kRowBlock / 64];
    const int sys = blockIdx.x;
    if (!epi.begin(sys)) return;
    double s = 0.0;
    for (int i = threadIdx.x; i < g.blk_count[sys]; i += kRowBlock) s += g.partials[2 * (g.blk_first[sys] + i)];
    s = block_sum<kRowBlock>(s, sh);
    if (threadIdx.x == 0) epi.finish(sys, s);
}

// One block per system: the sums of both slots of the system's block partials
// handed to f, in the order of the last-block ticket's sums.  For the column
// kernels at a solve's start and end, whose tickets' fences (an L2 write-back
// and invalidate a block) took most of their time: 16 systems of 102,222
// columns, |z|^2 76 -> 6 + 5 µs, the start of PCG 130 -> 12 + 5; one such
// system 8.6 -> 3 + 3.
template <class F>
__global__ __launch_bounds__(kRowBlock) void k_system_finish(F f, GridSys g)
{
    __shared__ double sh[kRowBlock / 64];
    if (!f.begin(blockIdx.x)) return;
    double s0, s1;
    system_sum2<kRowBlock>(g, blockIdx.x, sh, s0, s1);
    if (threadIdx.x == 0) f.finish(blockIdx.x, s0, s1);
}

template <class VT, class View>
__device__ __forceinline__ VT row_sum(const View& m, int k, int64_t r, uint32_t cb, const VT* __restrict__ x)
{
    VT acc = VT(0);
#pragma unroll 8
    for (int s = 0; s < k; s++) acc += x[cb + m.col(s, r)];
    return acc;
}

// Generic gather: one row per thread, x read straight from global memory
// (any matrix).
template <class VT, class View, class Epi>
__global__ __launch_bounds__(kRowBlock) void k_gather_rows(View m, int k, const RowWork* __restrict__ work,
                                                           const uint32_t* __restrict__ sys_col,
                                                           const VT* __restrict__ x, Epi epi, GridSys g)
{
    const RowWork w = work[blockIdx.x];
    if (!epi.begin(w.sys)) return;
    const uint32_t cb = sys_col[w.sys];
    double acc = 0.0;
    for (int64_t r = w.row_begin + threadIdx.x; r < w.row_end; r += kRowBlock)
        acc += epi.row(r, row_sum<VT>(m, k, r, cb, x));
    reduce_tail<kRowBlock>(epi, acc, w.sys, g);
}

// RPT consecutive entries of one slot column in one aligned vector load.
template <class IdxT, int RPT>
struct IdxVec;
template <>
struct IdxVec<uint16_t, 1> {
    using T = uint16_t;
    static __device__ __forceinline__ uint32_t get(T v, int) { return v; }
};
template <>
struct IdxVec<uint32_t, 1> {
    using T = uint32_t;
    static __device__ __forceinline__ uint32_t get(T v, int) { return v; }
};
template <>
struct IdxVec<uint16_t, 2> {
    using T = uint32_t;
    static __device__ __forceinline__ uint32_t get(T v, int i) { return (v >> (16 * i)) & 0xFFFFu; }
};
template <>
struct IdxVec<uint16_t, 4> {
    using T = uint2;
    static __device__ __forceinline__ uint32_t get(T v, int i)
    {
        const uint32_t w = i < 2 ? v.x : v.y;
        return (w >> (16 * (i & 1))) & 0xFFFFu;
    }
};
template <>
struct IdxVec<uint16_t, 8> {
    using T = uint4;
    static __device__ __forceinline__ uint32_t get(T v, int i)
    {
        const uint32_t w = i < 2 ? v.x : i < 4 ? v.y : i < 6 ? v.z : v.w;
        return (w >> (16 * (i & 1))) & 0xFFFFu;
    }
};
template <>
struct IdxVec<uint32_t, 2> {
    using T = uint2;
    static __device__ __forceinline__ uint32_t get(T v, int i) { return i == 0 ? v.x : v.y; }
};
template <>
struct IdxVec<uint32_t, 4> {
    using T = uint4;
    static __device__ __forceinline__ uint32_t get(T v, int i)
    {
        return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
    }
};

// One 16-byte line from global memory into LDS: lane i of the wave writes
// lds + 16 i (lds is the same for the whole wave).  Issued as an instruction
// the compiler does not see as an LDS write, so its own waits for LDS reads
// do not wait for this load -- nor for every vector load issued after it
// (vmcnt counts in order); the caller waits for it (s_waitcnt vmcnt(0)) and
// synchronises the block before any thread reads those bytes, and the block
// barriers before and after a staging keep the LDS accesses in order around
// it.  Declared without a memory clobber: one would mark every later load of
// the kernel's read-only tables as possibly overwritten and turn their scalar
// loads into vector loads with full vmcnt waits.  M0 (the LDS address of
// the load) is declared clobbered, so the compiler assumes no value of its
// own survives in it across the asm (clang warns that a reserved register is
// not saved for the caller, which is not wanted here).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void load_line_to_lds(const void* src, void* lds)
{
    const uint32_t la = __builtin_amdgcn_readfirstlane(
        uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)lds)));
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(la), "v"(src) : "m0");
}
#pragma clang diagnostic pop

// Copies the W elements at src into LDS at dst + h, h = the element offset of
// src inside its 16-byte line (dst is 16-byte aligned), and returns h: the
// 16-byte lines wholly inside [src, src + W) go from memory straight into LDS
// (global_load_lds_dwordx4: a wave's 64 lanes fill 1 KB of consecutive LDS,
// no registers held, every load of the thread in flight at once), the ragged
// head and tail through registers.  Reads nothing outside [src, src + W).
// The caller waits for the loads (vmcnt) and synchronises the block before
// the LDS is read.
template <class VT, int BS>
__device__ __forceinline__ uint32_t stage_direct(VT* __restrict__ dst, const VT* __restrict__ src, uint32_t W)
{
    constexpr uint32_t Q = 16 / sizeof(VT);
    const uint32_t h = uint32_t(reinterpret_cast<uintptr_t>(src) / sizeof(VT)) & (Q - 1);
    const uint32_t j0 = min(W, (Q - h) & (Q - 1));  // first element of a whole line
    const uint32_t nq = (W - j0) / Q;               // whole lines
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const VT* g = src + j0;
    VT* l = dst + h + j0;  // 16-byte aligned
    for (uint32_t t0 = wave * 64; t0 < nq; t0 += BS) {
        if (t0 + lane < nq) load_line_to_lds(g + (t0 + lane) * Q, l + t0 * Q);
    }
    if (threadIdx.x < Q) {
        const uint32_t a = threadIdx.x, b = j0 + nq * Q + threadIdx.x;
        if (a < j0) dst[h + a] = src[a];
        if (b < W) dst[h + b] = src[b];
    }
    return h;
}

// LDS-staged gather for pattern matrices.  A block owns a tile of rows and
// walks the plan's steps (runs of at most kMaxSegSlots slots of one segment,
// a segment being a run of slots over one column block) in slot order.  The
// columns of consecutive segments that fit the LDS together are staged in one
// phase, and the random reads of x then hit LDS instead of pulling an L2 line
// per element.  Thread t owns the RPT consecutive rows starting at the tile's
// first row rounded down to RPT plus RPT * t, so one aligned vector load brings
// a slot's entries of all its rows; the next step's entry loads go out once a
// step's staging has landed, so they are in flight during its sums.  Segments wider than the LDS (windows of
// wmax columns) are staged window by window: each slot's value is kept in
// registers until every window was seen, then the segment's slots are added
// in slot order, so every row is the sequential sum in slot order
// (Math/MatrixCSR.cpp:59-62).
// Threads of a tile-gather block: kTileBlock (one block and the whole LDS per
// CU), or half of it, with two blocks of half the LDS per CU whose staging
// and sums overlap each other.
constexpr int kTileBlock = 1024;

// Step k's descriptor in scalar registers (the same for the whole block).
__device__ __forceinline__ GatherStep step_at(const GatherStep* __restrict__ steps, int k)
{
    const uint32_t* __restrict__ w = reinterpret_cast<const uint32_t*>(steps + k);
    uint32_t r[sizeof(GatherStep) / 4];
#pragma unroll
    for (int i = 0; i < int(sizeof(GatherStep) / 4); i++) r[i] = __builtin_amdgcn_readfirstlane(w[i]);
    GatherStep st;
    __builtin_memcpy(&st, r, sizeof(st));
    return st;
}

// A step's entries of this thread's rows (threads past the tile read row 0
// through vec; the sums ignore them).  With Uncond every slot up to
// kMaxSegSlots is loaded (slots past the step's last repeat it): no branch
// around the loads, so the compiler can count them and need not wait for all
// loads in flight before a use; otherwise only the step's slots.
template <class IdxT, int RPT, bool Uncond>
__device__ __forceinline__ void load_step(typename IdxVec<IdxT, RPT>::T (&q)[kMaxSegSlots],
                                          const typename IdxVec<IdxT, RPT>::T* __restrict__ vec, int64_t vld,
                                          const GatherStep& st)
{
    const int last = st.nslots - 1;
#pragma unroll
    for (int j = 0; j < kMaxSegSlots; j++) {
        if (Uncond)
            q[j] = vec[int64_t(st.slot_first + min(j, last)) * vld];
        else if (j <= last)
            q[j] = vec[int64_t(st.slot_first + j) * vld];
    }
}

// element offset of p inside its 16-byte line
template <class VT>
__device__ __forceinline__ uint32_t line_head(const VT* p)
{
    return uint32_t(reinterpret_cast<uintptr_t>(p) / sizeof(VT)) & (16 / sizeof(VT) - 1);
}

// One tile per block (no sub-tiles): the body of k_gather_tile<..., 1>.
template <class VT, int RPT, class IdxT, class Epi, int BS>
__device__ __forceinline__ void gather_tile_single(const SlotMajor<IdxT>& m, const RowWork* __restrict__ work,
                                                   const uint32_t* __restrict__ sys_col,
                                                   const GatherStep* __restrict__ steps, int nsteps,
                                                   const PhaseSeg* __restrict__ phases, uint32_t wmax,
                                                   const VT* __restrict__ x, Epi& epi, const GridSys& g)
{
    using V = IdxVec<IdxT, RPT>;
    using VecT = typename V::T;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    VT* xs = reinterpret_cast<VT*>(smem_raw);
    const RowWork w = work[blockIdx.x];
    if (!epi.begin(w.sys)) return;
    const VT* __restrict__ xb = x + sys_col[w.sys];
    const int64_t a = (w.row_begin & ~int64_t(RPT - 1)) + int64_t(RPT) * threadIdx.x;
    const bool live = a < w.row_end;
    bool ok[RPT];
    VT acc[RPT];
#pragma unroll
    for (int i = 0; i < RPT; i++) {
        ok[i] = live && a + i >= w.row_begin && a + i < w.row_end;
        acc[i] = VT(0);
    }
    // slot s of this thread's rows: vec[s * vld]
    const VecT* __restrict__ vec = reinterpret_cast<const VecT*>(m.idx + (live ? a : 0));
    const int64_t vld = m.ld / RPT;
    // The next step's entries are loaded once this step's staging has landed,
    // so they are in flight while this step's sums run.  A segment wider than
    // the LDS holds its slots' values of every row until its last window; with
    // more than 8 bytes of entries per slot the registers do not allow holding
    // the next step's entries too, and the step after it loads its own.
    constexpr bool kPrefetchWide = sizeof(VecT) <= 8;
    constexpr int kWide = wide_step_slots(int(sizeof(VecT)));  // slots of a wide step (the plan's split)
    VecT q[kMaxSegSlots], qn[kMaxSegSlots];
    GatherStep st = nsteps > 0 ? step_at(steps, 0) : GatherStep{};
    bool have = false;  // q holds this step's entries (loaded by the step before)
    for (int k = 0; k < nsteps; k++) {
        const bool more = k + 1 < nsteps;
        const GatherStep nx = step_at(steps, more ? k + 1 : k);
        if (!have) load_step<IdxT, RPT, true>(q, vec, vld, st);
        have = false;
        if (st.nwin > 1) {
            // a segment wider than the LDS, at most kWide slots per step
            VT v[RPT][kWide];
#pragma unroll
            for (int j = 0; j < kWide; j++)
#pragma unroll
                for (int i = 0; i < RPT; i++) v[i][j] = VT(0);
            const bool rev = st.wflags & kWideReverse;
            for (uint32_t n = 0; n < st.nwin; n++) {
                const uint32_t wl = (rev ? st.nwin - 1 - n : n) * wmax;
                const uint32_t W = min(wmax, st.width - wl);
                // the next step's entries load with the last window's staging
                if constexpr (kPrefetchWide)
                    if (more && n + 1 == st.nwin) {
                        load_step<IdxT, RPT, true>(qn, vec, vld, nx);
                        have = true;
                    }
                uint32_t h;
                if (n == 0 && (st.wflags & kWideStaged)) {
                    // staged by the step before (same segment, same window)
                    h = line_head(xb + st.col_lo + wl);
                } else {
                    __syncthreads();
                    h = stage_direct<VT, BS>(xs, xb + st.col_lo + wl, W);
                    __builtin_amdgcn_s_waitcnt(0);
                    __syncthreads();
                }
#pragma unroll
                for (int j = 0; j < kWide; j++) {
                    if (j < st.nslots) {
                        // 32-bit offset: base - col_lo wraps for u32 storage
                        // (base 0) and the sum with the entry unwraps it
                        const uint32_t off = st.off[j] - wl;
#pragma unroll
                        for (int i = 0; i < RPT; i++) {
                            const uint32_t c = off + V::get(q[j], i);
                            const bool in = ok[i] && c < W;
                            const VT t = xs[h + (in ? c : 0u)];
                            v[i][j] = in ? t : v[i][j];
                        }
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < kWide; j++)
                if (j < st.nslots) {
#pragma unroll
                    for (int i = 0; i < RPT; i++) acc[i] += v[i][j];
                }
            if constexpr (kPrefetchWide)
                if (have) {
#pragma unroll
                    for (int j = 0; j < kMaxSegSlots; j++) q[j] = qn[j];
                }
        } else {
            if (st.phase_count > 0) {
                __syncthreads();
                for (int p = st.phase_first; p < st.phase_first + st.phase_count; p++) {
                    const PhaseSeg ps = phases[p];
                    stage_direct<VT, BS>(xs + ps.lds_off, xb + ps.col_lo, ps.width);
                }
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
            } else {
                // this step's entries must be in before the next step's loads
                // go out: the compiler's own wait for them would be a vmcnt(0)
                // after those
                __builtin_amdgcn_s_waitcnt(0);
            }
            if (more) {
                load_step<IdxT, RPT, true>(qn, vec, vld, nx);
                have = true;
            }
            const uint32_t h = line_head(xb + st.col_lo);
#pragma unroll
            for (int j = 0; j < kMaxSegSlots; j++) {
                if (j < st.nslots) {
                    const uint32_t off = st.off[j] + h;
#pragma unroll
                    for (int i = 0; i < RPT; i++)
                    {
                        const VT t = xs[ok[i] ? off + V::get(q[j], i) : 0u];
                        acc[i] += ok[i] ? t : VT(0);
                    }
                }
            }
            // (the copy in each branch: qn is not live across a wide step
            // that does not load it)
            if (have) {
#pragma unroll
                for (int j = 0; j < kMaxSegSlots; j++) q[j] = qn[j];
            }
        }
        st = nx;
    }
    // all RPT rows valid (every thread but the tile's first and last): the
    // epilogue's vector form; else row by row
    bool all = true;
#pragma unroll
    for (int i = 0; i < RPT; i++) all = all && ok[i];
    double red = 0.0;
    if (all) {
        red = epi.template rows<RPT>(a, acc);
    } else {
#pragma unroll
        for (int i = 0; i < RPT; i++)
            if (ok[i]) red += epi.row(a + i, acc[i]);
    }
    reduce_tail<BS>(epi, red, w.sys, g);
}

// S sub-tiles per block: the body of k_gather_tile<..., S > 1>.
template <class VT, int RPT, class IdxT, class Epi, int BS, int S>
__device__ __forceinline__ void gather_tile_sub(const SlotMajor<IdxT>& m, const RowWork* __restrict__ work,
                                                const uint32_t* __restrict__ sys_col,
                                                const GatherStep* __restrict__ steps, int nsteps,
                                                const PhaseSeg* __restrict__ phases, uint32_t wmax,
                                                const VT* __restrict__ x, Epi& epi, const GridSys& g)
{
    using V = IdxVec<IdxT, RPT>;
    using VecT = typename V::T;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    VT* xs = reinterpret_cast<VT*>(smem_raw);
    const RowWork w = work[blockIdx.x];
    if (!epi.begin(w.sys)) return;
    const VT* __restrict__ xb = x + sys_col[w.sys];
    // S sub-tiles of BS * RPT rows: in sub-tile u the thread owns rows
    // a0 + u * kSub + i, i < RPT; every staging serves all of them
    constexpr int64_t kSub = int64_t(RPT) * BS;
    const int64_t a0 = (w.row_begin & ~int64_t(RPT - 1)) + int64_t(RPT) * threadIdx.x;
    bool okr[S][RPT];  // that row is in the tile
    VT acc[S][RPT];
#pragma unroll
    for (int u = 0; u < S; u++)
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            const int64_t r = a0 + u * kSub + i;
            okr[u][i] = r >= w.row_begin && r < w.row_end;
            acc[u][i] = VT(0);
        }
    auto ok = [&](int u, int i) { return okr[u][i]; };
    // slot s of sub-tile u's rows: vec_of(u)[s * vld] (rows past the tile read row 0)
    const int64_t vld = m.ld / RPT;
    auto vec_of = [&](int u) {
        const int64_t au = a0 + u * kSub;
        return reinterpret_cast<const VecT*>(m.idx + (au < w.row_end ? au : 0));
    };
    // Where the registers allow it (up to 8 bytes of entries per slot) the
    // entries of the next (step, sub-tile) are loaded while this one sums;
    // otherwise each sub-tile loads its own (the first ahead of the staging).
    constexpr bool kPrefetch = sizeof(VecT) <= 8;
    VecT q[kMaxSegSlots], qn[kPrefetch ? kMaxSegSlots : 1];
    GatherStep st = nsteps > 0 ? step_at(steps, 0) : GatherStep{};
    if (kPrefetch && nsteps > 0) load_step<IdxT, RPT, true>(q, vec_of(0), vld, st);
    for (int k = 0; k < nsteps; k++) {
        const bool more = k + 1 < nsteps;
        const GatherStep nx = step_at(steps, more ? k + 1 : k);
        // the pair after (k, u) is (k, u + 1), or (k + 1, 0)
        auto prefetch_after = [&](int u) {
            if constexpr (kPrefetch) {
                if (u + 1 < S)
                    load_step<IdxT, RPT, true>(qn, vec_of(u + 1), vld, st);
                else if (more)
                    load_step<IdxT, RPT, true>(qn, vec_of(0), vld, nx);
            }
        };
        auto advance = [&](int u) {
            if constexpr (kPrefetch)
                if (u + 1 < S || more) {
#pragma unroll
                    for (int j = 0; j < kMaxSegSlots; j++) q[j] = qn[j];
                }
        };
        if (st.nwin > 1) {
            // a segment wider than the LDS, at most kMaxSegSlots slots: each
            // sub-tile walks its windows
#pragma unroll
            for (int u = 0; u < S; u++) {
                if constexpr (!kPrefetch) load_step<IdxT, RPT, false>(q, vec_of(u), vld, st);
                VT v[RPT][kMaxSegSlots];
#pragma unroll
                for (int j = 0; j < kMaxSegSlots; j++)
#pragma unroll
                    for (int i = 0; i < RPT; i++) v[i][j] = VT(0);
                for (uint32_t wl = 0; wl < st.width; wl += wmax) {
                    const uint32_t W = min(wmax, st.width - wl);
                    // the next entries load with the last window's staging
                    if (wl + W >= st.width) prefetch_after(u);
                    __syncthreads();
                    const uint32_t h = stage_direct<VT, BS>(xs, xb + st.col_lo + wl, W);
                    __builtin_amdgcn_s_waitcnt(0);
                    __syncthreads();
#pragma unroll
                    for (int j = 0; j < kMaxSegSlots; j++) {
                        if (j < st.nslots) {
                            // 32-bit offset: base - col_lo wraps for u32 storage
                            // (base 0) and the sum with the entry unwraps it
                            const uint32_t off = st.off[j] - wl;
#pragma unroll
                            for (int i = 0; i < RPT; i++) {
                                const uint32_t c = off + V::get(q[j], i);
                                const bool in = ok(u, i) && c < W;
                                const VT t = xs[h + (in ? c : 0u)];
                                v[i][j] = in ? t : v[i][j];
                            }
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < kMaxSegSlots; j++)
                    if (j < st.nslots) {
#pragma unroll
                        for (int i = 0; i < RPT; i++) acc[u][i] += v[i][j];
                    }
                advance(u);
            }
        } else {
            if constexpr (!kPrefetch) load_step<IdxT, RPT, false>(q, vec_of(0), vld, st);
            if (st.phase_count > 0) {
                __syncthreads();
                for (int p = st.phase_first; p < st.phase_first + st.phase_count; p++) {
                    const PhaseSeg ps = phases[p];
                    stage_direct<VT, BS>(xs + ps.lds_off, xb + ps.col_lo, ps.width);
                }
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
            }
            const uint32_t h = line_head(xb + st.col_lo);
#pragma unroll
            for (int u = 0; u < S; u++) {
                if constexpr (!kPrefetch) {
                    if (u > 0) load_step<IdxT, RPT, false>(q, vec_of(u), vld, st);
                } else if (u > 0 || st.phase_count == 0) {
                    // this pair's entries (loaded during the last pair's sums)
                    // must be in before the next pair's loads go out: the
                    // compiler's own wait for them would be a vmcnt(0) after
                    __builtin_amdgcn_s_waitcnt(0);
                }
                prefetch_after(u);
#pragma unroll
                for (int j = 0; j < kMaxSegSlots; j++) {
                    if (j < st.nslots) {
                        const uint32_t off = st.off[j] + h;
#pragma unroll
                        for (int i = 0; i < RPT; i++) {
                            const VT t = xs[ok(u, i) ? off + V::get(q[j], i) : 0u];
                            acc[u][i] += ok(u, i) ? t : VT(0);
                        }
                    }
                }
                advance(u);
            }
        }
        st = nx;
    }
    // a sub-tile's RPT rows all in the tile (every thread but the tile's first
    // and last): the epilogue's vector form; else row by row
    double red = 0.0;
#pragma unroll
    for (int u = 0; u < S; u++) {
        const int64_t au = a0 + u * kSub;
        bool all = true;
#pragma unroll
        for (int i = 0; i < RPT; i++) all = all && okr[u][i];
        if (all) {
            red += epi.template rows<RPT>(au, acc[u]);
        } else {
#pragma unroll
            for (int i = 0; i < RPT; i++)
                if (ok(u, i)) red += epi.row(au + i, acc[u][i]);
        }
    }
    reduce_tail<BS>(epi, red, w.sys, g);
}

// The stored gather over long tiles: as gather_tile_single, with R runs of
// kTileBlock * RPT rows a tile that share every staging, wide segments too
// (their windows are walked once for all runs, in steps of kWide slots whose
// values stay in registers).  A staging (160 KB through the L2, two barriers,
// the latency) costs a CU the same whatever the rows it serves, and a block its
// start and end; so a CU's rows are one tile where the registers allow it.  (5M rows of FIT8: FP64 165 µs against 334 with 2,048 rows a tile, FP32
// 95 against 121 with three tiles a CU; 1.2M rows of edax in FP64 46 against
// 102.)  Steps hold at most kLongStep slots; the entries of the next (step, run)
// load while this one sums.  Entries of rows outside the tile are read like
// the others (they are valid columns) and their sums dropped.
template <class VT, int RPT, class IdxT, class Epi, int R, int kWide>
__device__ __forceinline__ double gather_long(const SlotMajor<IdxT>& m, const RowWork& w,
                                              const GatherStep* __restrict__ steps, int nsteps,
                                              const PhaseSeg* __restrict__ phases, uint32_t wmax,
                                              const VT* __restrict__ xb, VT* __restrict__ xs, Epi& epi)
{
    using V = IdxVec<IdxT, RPT>;
    using VecT = typename V::T;
    constexpr int kSub = RPT * kTileBlock;
    const int64_t a0 = (w.row_begin & ~int64_t(RPT - 1)) + int64_t(RPT) * threadIdx.x;
    const int64_t vld = m.ld / RPT;
    VT acc[R][RPT];
#pragma unroll
    for (int u = 0; u < R; u++)
#pragma unroll
        for (int i = 0; i < RPT; i++) acc[u][i] = VT(0);
    // up to N slots of step st of run u (threads past the tile read its first
    // rows; slots past the step's last repeat it)
    auto load = [&](auto& q, const GatherStep& st, int u) {
        const int64_t a = a0 + u * kSub;
        const VecT* __restrict__ v = reinterpret_cast<const VecT*>(m.idx + (a < w.row_end ? a : (w.row_begin & ~int64_t(RPT - 1))));
        constexpr int N = sizeof(q) / sizeof(q[0]);
#pragma unroll
        for (int j = 0; j < N; j++) q[j] = v[int64_t(st.slot_first + min(j, st.nslots - 1)) * vld];
    };
    VecT q[kLongStep];
    GatherStep st = step_at(steps, 0);
    bool have = false;  // q holds run 0's entries of this step
    for (int k = 0; k < nsteps; k++) {
        const bool more = k + 1 < nsteps;
        const GatherStep nx = step_at(steps, more ? k + 1 : k);
        if (st.nwin > 1) {
            VecT qw[R][kWide];
            VT v[R][RPT][kWide];
#pragma unroll
            for (int u = 0; u < R; u++) {
                load(qw[u], st, u);
#pragma unroll
                for (int i = 0; i < RPT; i++)
#pragma unroll
                    for (int j = 0; j < kWide; j++) v[u][i][j] = VT(0);
            }
            const bool rev = st.wflags & kWideReverse;
            for (uint32_t n = 0; n < st.nwin; n++) {
                const uint32_t wl = (rev ? st.nwin - 1 - n : n) * wmax;
                const uint32_t W = min(wmax, st.width - wl);
                const uint32_t h = line_head(xb + st.col_lo + wl);
                if (n > 0 || !(st.wflags & kWideStaged)) {  // (else staged by the step before)
                    __syncthreads();
                    stage_direct<VT, kTileBlock>(xs, xb + st.col_lo + wl, W);
                    __builtin_amdgcn_s_waitcnt(0);
                    __syncthreads();
                }
#pragma unroll
                for (int u = 0; u < R; u++) {
#pragma unroll
                    for (int j = 0; j < kWide; j++) {
                        if (j < st.nslots) {
                            // 32-bit offset: base - col_lo wraps for u32
                            // storage (base 0) and the sum with the entry
                            // unwraps it
                            const uint32_t off = st.off[j] - wl;
#pragma unroll
                            for (int i = 0; i < RPT; i++) {
                                const uint32_t c = off + V::get(qw[u][j], i);
                                const VT t = xs[h + (c < W ? c : 0u)];
                                v[u][i][j] = c < W ? t : v[u][i][j];
                            }
                        }
                    }
                }
            }
            // the next step's entries, unless it is a step of this kind
            have = more && nx.nwin <= 1;
            if (have) load(q, nx, 0);
#pragma unroll
            for (int j = 0; j < kWide; j++)
                if (j < st.nslots) {
#pragma unroll
                    for (int u = 0; u < R; u++)
#pragma unroll
                        for (int i = 0; i < RPT; i++) acc[u][i] += v[u][i][j];
                }
        } else {
            if (!have) load(q, st, 0);
            if (st.phase_count > 0) {
                __syncthreads();
                for (int p = st.phase_first; p < st.phase_first + st.phase_count; p++) {
                    const PhaseSeg ps = phases[p];
                    stage_direct<VT, kTileBlock>(xs + ps.lds_off, xb + ps.col_lo, ps.width);
                }
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
            }
            const uint32_t h = line_head(xb + st.col_lo);
            have = more && nx.nwin <= 1;
#pragma unroll
            for (int u = 0; u < R; u++) {
                // this run's entries must be in before the next loads go out:
                // the compiler's own wait for them would be one for all
                __builtin_amdgcn_s_waitcnt(0);
                VecT qn[kLongStep];
                if (u + 1 < R) load(qn, st, u + 1);
                else if (have) load(qn, nx, 0);
#pragma unroll
                for (int j = 0; j < kLongStep; j++) {
                    if (j < st.nslots) {
                        const uint32_t off = st.off[j] + h;
#pragma unroll
                        for (int i = 0; i < RPT; i++) acc[u][i] += xs[off + V::get(q[j], i)];
                    }
                }
                if (u + 1 < R || have) {
#pragma unroll
                    for (int j = 0; j < kLongStep; j++) q[j] = qn[j];
                }
            }
        }
        st = nx;
    }
    // a run's RPT rows all in the tile (every thread but the tile's first and
    // last): the epilogue's vector form; else row by row
    double red = 0.0;
#pragma unroll
    for (int u = 0; u < R; u++) {
        const int64_t a = a0 + u * kSub;
        if (a >= w.row_begin && a + RPT <= w.row_end) {
            red += epi.template rows<RPT>(a, acc[u]);
        } else {
#pragma unroll
            for (int i = 0; i < RPT; i++)
                if (a + i >= w.row_begin && a + i < w.row_end) red += epi.row(a + i, acc[u][i]);
        }
    }
    return red;
}

// (a tile with fewer runs of rows than R -- a batch's small systems, the last
// tile of a system -- runs the body for those)
template <class VT, int RPT, class IdxT, class Epi, int R, int kWide>
__global__ __launch_bounds__(kTileBlock) void k_gather_long(SlotMajor<IdxT> m, const RowWork* __restrict__ work,
                                                            const uint32_t* __restrict__ sys_col,
                                                            const GatherStep* __restrict__ steps, int nsteps,
                                                            const PhaseSeg* __restrict__ phases, uint32_t wmax,
                                                            const VT* __restrict__ x, Epi epi, GridSys g)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    VT* xs = reinterpret_cast<VT*>(smem_raw);
    const RowWork w = work[blockIdx.x];
    if (!epi.begin(w.sys)) return;
    const VT* __restrict__ xb = x + sys_col[w.sys];
    const int64_t rows = w.row_end - (w.row_begin & ~int64_t(RPT - 1));
    double red;
    if (R > 1 && rows <= RPT * kTileBlock)
        red = gather_long<VT, RPT, IdxT, Epi, 1, kWide>(m, w, steps, nsteps, phases, wmax, xb, xs, epi);
    else if (R > 2 && rows <= 2 * RPT * kTileBlock)
        red = gather_long<VT, RPT, IdxT, Epi, R < 2 ? R : 2, kWide>(m, w, steps, nsteps, phases, wmax, xb, xs, epi);
    else
        red = gather_long<VT, RPT, IdxT, Epi, R, kWide>(m, w, steps, nsteps, phases, wmax, xb, xs, epi);
    reduce_tail<kTileBlock>(epi, red, w.sys, g);
}

template <class VT, int RPT, class IdxT, class Epi, int BS, int S>
__global__ __launch_bounds__(BS) void k_gather_tile(SlotMajor<IdxT> m, const RowWork* __restrict__ work,
                                                    const uint32_t* __restrict__ sys_col,
                                                    const GatherStep* __restrict__ steps, int nsteps,
                                                    const PhaseSeg* __restrict__ phases, uint32_t wmax,
                                                    const VT* __restrict__ x, Epi epi, GridSys g)
{
    if constexpr (S == 1)
        gather_tile_single<VT, RPT, IdxT, Epi, BS>(m, work, sys_col, steps, nsteps, phases, wmax, x, epi, g);
    else
        gather_tile_sub<VT, RPT, IdxT, Epi, BS, S>(m, work, sys_col, steps, nsteps, phases, wmax, x, epi, g);
}

// The LDS-staged gather of a matrix-free pattern matrix: the stored tile
// kernel's plan (steps over the slots, narrow segments staged side by side in
// one phase, wide segments window by window), with every slot's column
// computed by its index tile where the stored kernel loads it.  A wave owns
// 64 rows of each of the block's RPT runs of kTileBlock rows and keeps their
// digits in registers (16 a run); each tile's columns turn from one slot per
// 16-lane group to one row per lane, and the row sums run in slot order.  A
// wide step holds one tile (four slots), its columns computed once, before
// the window loop.
// 20M rows of FIT12: 998 µs (digit by digit 1,764): 54 % of the cycles issue
// vector instructions, and staging with its barriers takes about a third (26
// µs a tile of 4,096 rows when nothing else is done).  Four runs are what the
// registers hold: with two it takes 1,336 µs; a loop over more rows a block,
// computing during the staging, and taking the digits anew in every phase so
// that eight runs fit all spilled or took longer (1,180 to 1,450 µs).
template <class VT, int RPT, class Epi>
__global__ __launch_bounds__(kTileBlock) void k_gather_tile_mf(PositionsView m, const RowWork* __restrict__ work,
                                                               const uint32_t* __restrict__ sys_col,
                                                               const GatherStep* __restrict__ steps, int nsteps,
                                                               const PhaseSeg* __restrict__ phases, uint32_t wmax,
                                                               const VT* __restrict__ x, Epi epi, GridSys g)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    VT* xs = reinterpret_cast<VT*>(smem_raw);
    const RowWork w = work[blockIdx.x];
    if (!epi.begin(w.sys)) return;
    const VT* __restrict__ xb = x + sys_col[w.sys];
    const int64_t r0 = w.row_begin + threadIdx.x;
    const int nval = int(max<int64_t>(0, min<int64_t>(w.row_end - r0, int64_t(RPT) * kTileBlock)));
    // the wave's first row of run c: wave0 + c kTileBlock (rows past the tile's
    // end repeat its last)
    const int64_t wave0 = w.row_begin + (threadIdx.x & ~63u);
    Int4 b[RPT][4];
    VT acc[RPT];
#pragma unroll
    for (int c = 0; c < RPT; c++) {
        acc[c] = VT(0);
#pragma unroll
        for (int p = 0; p < 4; p++)
            b[c][p] = digits_of_words(m.tw, min(wave0 + int64_t(c) * kTileBlock + 16 * p + int(threadIdx.x & 15),
                                                w.row_end - 1));
    }
    for (int k = 0; k < nsteps; k++) {
        const GatherStep st = step_at(steps, k);
        if (st.nwin > 1) {
            // a segment wider than the LDS: the tile's columns
            // (segment-local), then the windows, each slot's value kept until
            // the last window
            const IndexTile tl = uniform_load(m.tiles.tiles + st.tile_first);
            const Int4 wt = *tile_weights(int(st.tile_first), m.tiles);
            const uint32_t off = st.off[0] + tl.col_offset;
            uint32_t ci[RPT][4];
            VT v[RPT][4];
#pragma unroll
            for (int c = 0; c < RPT; c++) {
                tile_columns(tl, int(st.tile_first), m.tiles, wt, b[c], ci[c]);
                transpose_groups(ci[c]);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    ci[c][j] += off;
                    v[c][j] = VT(0);
                }
            }
            const bool rev = st.wflags & kWideReverse;
            for (uint32_t n = 0; n < st.nwin; n++) {
                const uint32_t wl = (rev ? st.nwin - 1 - n : n) * wmax;
                const uint32_t W = min(wmax, st.width - wl);
                const uint32_t h = line_head(xb + st.col_lo + wl);
                if (n > 0 || !(st.wflags & kWideStaged)) {  // (else staged by the step before)
                    __syncthreads();
                    stage_direct<VT, kTileBlock>(xs, xb + st.col_lo + wl, W);
                    __builtin_amdgcn_s_waitcnt(0);
                    __syncthreads();
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    if (j < st.nslots) {
#pragma unroll
                        for (int c = 0; c < RPT; c++) {
                            const uint32_t cl = ci[c][j] - wl;
                            if (cl < W) v[c][j] = xs[h + cl];
                        }
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (j < st.nslots) {
#pragma unroll
                    for (int c = 0; c < RPT; c++) acc[c] += v[c][j];
                }
        } else {
            if (st.phase_count > 0) {
                __syncthreads();
                for (int p = st.phase_first; p < st.phase_first + st.phase_count; p++) {
                    const PhaseSeg ps = uniform_load(phases + p);
                    stage_direct<VT, kTileBlock>(xs + ps.lds_off, xb + ps.col_lo, ps.width);
                }
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
            }
            const uint32_t h = line_head(xb + st.col_lo);
            for (int t = 0; 4 * t < st.nslots; t++) {
                const int number = int(st.tile_first) + t;
                const IndexTile tl = uniform_load(m.tiles.tiles + number);
                const Int4 wt = *tile_weights(number, m.tiles);
                const uint32_t off = st.off[0] + h + tl.col_offset;
#pragma unroll
                for (int c = 0; c < RPT; c++) {
                    uint32_t ci[4];
                    tile_columns(tl, number, m.tiles, wt, b[c], ci);
                    transpose_groups(ci);
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        if (j < tl.nslots) acc[c] += xs[off + ci[j]];
                }
            }
        }
    }
    double red = 0.0;
#pragma unroll
    for (int c = 0; c < RPT; c++)
        if (c * kTileBlock < nval) red += epi.row(r0 + int64_t(c) * kTileBlock, acc[c]);
    reduce_tail<kTileBlock>(epi, red, w.sys, g);
}

// ------------------------------------------------------------ scatter ------
// Which systems a scatter serves, and its scale:
//   kScatterAll      every system, scale 1 (plain products)
//   kScatterLsqr     the systems iterating (active, not stopped), y scaled by 1 / beta
//   kScatterRestart  the systems being (re)started (active, restart), scale 1
constexpr int kScatterAll = 0, kScatterLsqr = 1, kScatterRestart = 2;

__device__ __forceinline__ bool scatter_selected(const LsqrScalars* div, int mode, int sys)
{
    if (mode == kScatterAll) return true;
    const LsqrScalars& d = div[sys];
    if (!d.active) return false;
    return mode == kScatterLsqr ? d.stop == 0 : d.restart != 0;
}

template <class VT>
__device__ __forceinline__ VT scatter_scale(const LsqrScalars* div, int mode, int sys)
{
    if (mode != kScatterLsqr) return VT(1);
    const double d = div[sys].beta;
    return VT(d != 0.0 ? 1.0 / d : 0.0);
}

// The same, where an LSQR iteration hands over its gather's |u_raw|^2 block
// partials (bsum.partials non-null): beta = sqrt of their sum is formed here,
// by every block from the same partials in the same order (so all blocks
// agree), and stored with its square for the kernels after; the scatter then
// reads no beta from the state.  Only the kBeta instantiations of the scatter
// kernels carry this code (the others compile as if it did not exist).
template <class VT, int BS, bool kBeta>
__device__ __forceinline__ VT scatter_scale(LsqrScalars* div, int mode, int sys, const GridSys& bsum)
{
    if constexpr (!kBeta) return scatter_scale<VT>(div, mode, sys);
    if (mode != kScatterLsqr || !bsum.partials) return scatter_scale<VT>(div, mode, sys);
    __shared__ double sh[BS / 64];
    const double s = system_sum<BS>(bsum, sys, sh);
    const double d = sqrt(s);
    if (threadIdx.x == 0) {
        div[sys].beta = d;
        div[sys].beta2 = s;
    }
    return VT(d != 0.0 ? 1.0 / d : 0.0);
}

// Integer accumulation of an FP32 scatter window.  Each term y * scale is
// rounded to a multiple of 2^-s and the window adds the int64 multiples with
// LDS integer atomics (ds_add_u64), which run about 1.8 times as fast as the
// FP64 ones on gfx950 and make the sums independent of the atomics' order
// (the FP32 A^T y is bit-reproducible).  s is chosen so that no column sum
// can overflow: |term| < 2^ey and fewer than 2^cbits terms per column and
// work item, so every sum stays below 2^(62 - 1); each term keeps at least 32
// bits (rounding error <= 2^(ey - 33) of the largest term, far below FP32
// rounding of the sums where y is of one size; a column that only terms of
// 2^-15 of the largest or less reach keeps fewer bits than FP32 has).  Outside
// an LSQR iteration, where |u_r / beta| < 2 by construction, the kYmax
// instantiation takes the bits of each system's max |y| (a non-negative float,
// NaN and inf above every finite value) from the row blocks' maxima that
// k_absmax_blocks left (ypart, the system's blocks at yfirst[sys], ycount[sys]).
struct FixedScale {
    int cbits;
    const unsigned* ypart;
    const int32_t* yfirst;
    const int32_t* ycount;
};

// 2^s for a system whose max |y| has float bits b (bounded: b is given; else
// |y * sc| < 2), or 0 where the FP64 window must be used (non-finite values,
// or fewer than 32 bits left for the largest term).
__device__ __forceinline__ double fixed_scale_bits(int cbits, bool bounded, unsigned b, double sc)
{
    int ey;
    if (bounded) {
        if (b >= 0x7f800000u) return 0.0;
        ey = b == 0 ? -126 : ilogbf(__uint_as_float(b)) + 1;
    } else {
        if (!isfinite(sc)) return 0.0;
        ey = 1;
    }
    const int sh = 62 - cbits - ey;
    if (sh + ey < 32) return 0.0;
    return ldexp(1.0, sh);
}

// The max of a system's row-block maxima (float bits), in every thread.
template <int BS>
__device__ __forceinline__ unsigned system_max(const FixedScale& fx, int sys, unsigned* sh)
{
    unsigned mb = 0;
    const int first = fx.yfirst[sys], n = fx.ycount[sys];
    for (int i = threadIdx.x; i < n; i += BS) mb = max(mb, fx.ypart[first + i]);
    for (int o = 32; o > 0; o >>= 1) mb = max(mb, unsigned(__shfl_xor(int(mb), o, 64)));
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = mb;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < BS / 64; i++) mb = max(mb, sh[i]);
        sh[0] = mb;
    }
    __syncthreads();
    return sh[0];
}

template <class WT>
__device__ __forceinline__ WT window_term(double v, double fscale)
{
    if constexpr (std::is_same_v<WT, double>)
        return v;
    else
        return WT(__double2ll_rn(v * fscale));
}

// The fixed-point scale of a block's window (0: the FP64 window): of FP32
// windows, from the system's max |y| -- formed here from the row blocks' maxima
// where the instantiation says so -- or LSQR's bound.
template <class VT, int BS, bool kYmax>
__device__ __forceinline__ double window_scale(const FixedScale& fx, int sys, VT sc, bool allowed = true)
{
    if constexpr (!std::is_same_v<VT, float>) {
        return 0.0;
    } else if constexpr (kYmax) {
        __shared__ unsigned shm[BS / 64];
        const unsigned b = system_max<BS>(fx, sys, shm);
        return allowed ? fixed_scale_bits(fx.cbits, true, b, double(sc)) : 0.0;
    } else {
        return allowed ? fixed_scale_bits(fx.cbits, false, 0u, double(sc)) : 0.0;
    }
}

// A finished window as a partial slice.
template <class VT>
__device__ __forceinline__ void store_window(const double* __restrict__ win, uint32_t W, double fscale,
                                             VT* __restrict__ out)
{
    if (fscale > 0.0) {
        const unsigned long long* wu = reinterpret_cast<const unsigned long long*>(win);
        const double inv = 1.0 / fscale;  // a power of two: exact
        for (uint32_t i = threadIdx.x; i < W; i += kScatterBlock) out[i] = VT(double((long long)wu[i]) * inv);
    } else {
        for (uint32_t i = threadIdx.x; i < W; i += kScatterBlock) out[i] = VT(win[i]);
    }
}

// max |y| of each row block as float bits (non-negative floats order as unsigned
// integers; NaN and inf above every finite value): the ypart of FixedScale.
// 5M rows: 7.1 µs, 10.5 with one row a thread at a time.
template <class YT>
__global__ __launch_bounds__(kRowBlock) void k_absmax_blocks(const RowWork* __restrict__ work,
                                                             const YT* __restrict__ y, unsigned* __restrict__ part)
{
    __shared__ unsigned sh[kRowBlock / 64];
    const RowWork w = work[blockIdx.x];
    unsigned mb = 0;
    // four rows a thread in flight (the last row again past the end)
    for (int64_t r = w.row_begin + threadIdx.x; r < w.row_end; r += 4 * kRowBlock) {
        YT t[4];
#pragma unroll
        for (int i = 0; i < 4; i++) t[i] = y[min(r + i * kRowBlock, w.row_end - 1)];
#pragma unroll
        for (int i = 0; i < 4; i++) mb = max(mb, __float_as_uint(fabsf(float(t[i]))));
    }
    for (int o = 32; o > 0; o >>= 1) mb = max(mb, unsigned(__shfl_xor(int(mb), o, 64)));
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = mb;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < kRowBlock / 64; i++) mb = max(mb, sh[i]);
        part[blockIdx.x] = mb;
    }
}

// The evaluator's A^T g, stage 1: each block owns a column window of one slot
// group in LDS, adds a chunk of the minibatch's rows into it (FP64: LDS atomic
// adds on doubles run several times faster than on floats on this GPU, and the
// sums are exact for integer data either way) and stores the window to its
// slice of the partial buffer -- no global atomics.  Entry (r, s) is
// idx[r row_stride + s slot_stride].  A chunk is one or two rows a thread, so
// the kernel is a chain of latencies: the first two rows' entries and g are on
// their way before the window is cleared, all of a row's entries together -- as
// many as a group of up to four slots or of up to eight has, and no second row
// where there is none (4,096 rows of 4 slots 8.3 µs with eight loads for each of
// two rows, 7.0 so, both with the column sums; 65,536 rows of FIT4 21.1 and 17.5).
// 65,536 rows of FIT4 alone 9.9 µs slot-major and 12.4 row-major, where every
// lane's entries lie in lines of their own.
// Groups are runs of at most kMaxSegSlots consecutive slots.
template <class VT>
__global__ __launch_bounds__(kScatterBlock) void k_scatter_part(const int32_t* __restrict__ idx, int64_t row_stride,
                                                                int64_t slot_stride,
                                                                const ScatterWork* __restrict__ work,
                                                                const SlotGroup* __restrict__ groups,
                                                                const uint16_t* __restrict__ slot_list,
                                                                const VT* __restrict__ g, VT* __restrict__ part)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double* win = reinterpret_cast<double*>(smem_raw);
    const ScatterWork w = constant_load(work + blockIdx.x);
    const SlotGroup gr = constant_load(groups + w.group);
    const int ns = gr.nslots, s0 = uniform_u16(slot_list, gr.first);
    const uint32_t W = w.win_hi - w.win_lo;
    auto rows = [&](auto slots) {
        constexpr int NS = decltype(slots)::value, kRows = 2;
        int32_t c[kRows][NS];
        VT y[kRows];
        // rows a + threadIdx.x and, if the chunk has any, the kScatterBlock rows after
        auto load = [&](int64_t a) {
#pragma unroll
            for (int u = 0; u < kRows; u++) {
                if (a + u * kScatterBlock >= w.row_end) break;
                const int64_t r = min(a + u * kScatterBlock + threadIdx.x, w.row_end - 1);
                const int32_t* __restrict__ row = idx + r * row_stride + s0 * slot_stride;
#pragma unroll
                for (int j = 0; j < NS; j++) c[u][j] = row[min(j, ns - 1) * slot_stride];
                y[u] = g[r];
            }
        };
        load(w.row_begin);
        for (uint32_t i = threadIdx.x; i < W; i += kScatterBlock) win[i] = 0.0;
        __syncthreads();
        for (int64_t a = w.row_begin; a < w.row_end; a += kRows * kScatterBlock) {
#pragma unroll
            for (int u = 0; u < kRows; u++) {
                if (a + u * kScatterBlock >= w.row_end) break;
                const bool ok = a + u * kScatterBlock + threadIdx.x < w.row_end;
#pragma unroll
                for (int j = 0; j < NS; j++) {
                    const uint32_t uc = uint32_t(c[u][j]) - w.win_lo;
                    if (j < ns && ok && uc < W) atomicAdd(&win[uc], double(y[u]));
                }
            }
            load(a + kRows * kScatterBlock);
        }
    };
    if (ns <= kMaxSegSlots / 2)
        rows(std::integral_constant<int, kMaxSegSlots / 2>{});
    else
        rows(std::integral_constant<int, kMaxSegSlots>{});
    __syncthreads();
    store_window<VT>(win, W, 0.0, part + w.part_off);
}

// The rows of one scatter work item for a group of at most NS slots (slot j
// of the group at vec + slot[j], its window offset off[j]; slots ns..NS-1
// repeat slot 0's loads and add nothing).  Every load is unconditional (rows
// clamped into the chunk), and the next step's y and entries are loaded
// before this step's atomics, so their latency overlaps the LDS work.
template <int NS, class WT, bool VY, class VT, class YT, class IdxT, int RPT>
__device__ __forceinline__ void scatter_rows(const SlotMajor<IdxT>& m, const ScatterWork& w, int ns,
                                             const int64_t (&slot)[kMaxSegSlots],
                                             const uint32_t (&off)[kMaxSegSlots], const YT* __restrict__ y,
                                             VT sc, double fscale, uint32_t W, bool full, WT* win)
{
    using V = IdxVec<IdxT, RPT>;
    using VecT = typename V::T;
    if (w.row_end <= w.row_begin) return;
    const int64_t last = w.row_end - 1, alast = last & ~int64_t(RPT - 1);
    const int64_t stride = int64_t(RPT) * kScatterBlock;
    auto fetch = [&](int64_t at, VecT (&q)[NS], YT (&yy)[RPT]) {
        const VecT* __restrict__ vec = reinterpret_cast<const VecT*>(m.idx + min(at, alast));
#pragma unroll
        for (int j = 0; j < NS; j++) q[j] = vec[slot[j]];
        if constexpr (VY) {
            // y readable through the padding to a multiple of 64 rows: the
            // RPT values in 16-byte loads (rows past the chunk are masked)
            constexpr int kPer = 16 / int(sizeof(YT));
            using Y16 = std::conditional_t<sizeof(YT) == 4, float4, double2>;
            const Y16* __restrict__ yv = reinterpret_cast<const Y16*>(y + min(at, alast));
#pragma unroll
            for (int i = 0; i < RPT; i += kPer) {
                const Y16 t = yv[i / kPer];
                __builtin_memcpy(&yy[i], &t, 16);
            }
        } else {
#pragma unroll
            for (int i = 0; i < RPT; i++) yy[i] = y[min(at + i, last)];
        }
    };
    int64_t a = (w.row_begin & ~int64_t(RPT - 1)) + int64_t(RPT) * threadIdx.x;
    VecT q[NS];
    YT yr[RPT];
    fetch(a, q, yr);
    for (; a < w.row_end; a += stride) {
        VecT qn[NS];
        YT yn[RPT];
        fetch(a + stride, qn, yn);
        WT yv[RPT];
        bool ok[RPT];
#pragma unroll
        for (int i = 0; i < RPT; i++) {
            ok[i] = a + i >= w.row_begin && a + i < w.row_end;
            yv[i] = window_term<WT>(double(VT(yr[i]) * sc), fscale);
        }
        // A wave whose rows all lie inside the chunk, over a group whose
        // columns all lie in the window, adds without per-lane conditions
        // (entries past the window, which valid data never holds, are held
        // inside it rather than skipped)
        if (__all(full && a >= w.row_begin && a + RPT <= w.row_end)) {
#pragma unroll
            for (int j = 0; j < NS; j++) {
                if (j < ns) {
#pragma unroll
                    for (int i = 0; i < RPT; i++) atomicAdd(&win[min(off[j] + V::get(q[j], i), W - 1)], yv[i]);
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < NS; j++) {
                if (j < ns) {
#pragma unroll
                    for (int i = 0; i < RPT; i++) {
                        const uint32_t uc = off[j] + V::get(q[j], i);
                        if (ok[i] && uc < W) atomicAdd(&win[uc], yv[i]);
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < NS; j++) q[j] = qn[j];
#pragma unroll
        for (int i = 0; i < RPT; i++) yr[i] = yn[i];
    }
}

// Stage 1 for stored indices: as k_scatter_part, with each thread taking RPT
// consecutive rows per step (counted from the chunk's first row rounded down
// to RPT) so one aligned vector load brings a slot's entries of all of them.
// For groups of up to kMaxSegSlots slots the slot numbers and window offsets
// are hoisted out of the row loop and the loads are software-pipelined
// (scatter_rows).
template <class VT, class YT, class IdxT, int RPT, bool kBeta = false, bool kYmax = false>
__global__ __launch_bounds__(kScatterBlock) void k_scatter_tile(SlotMajor<IdxT> m,
                                                                const ScatterWork* __restrict__ work,
                                                                const SlotGroup* __restrict__ groups,
                                                                const uint16_t* __restrict__ slot_list,
                                                                const uint32_t* __restrict__ sys_col,
                                                                const YT* __restrict__ y, LsqrScalars* div,
                                                                int mode, FixedScale fx, int y_padded,
                                                                VT* __restrict__ part, GridSys bsum)
{
    using V = IdxVec<IdxT, RPT>;
    using VecT = typename V::T;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double* win = reinterpret_cast<double*>(smem_raw);  // 8-byte window words (FP64 or fixed point)
    const ScatterWork w = work[blockIdx.x];
    if (!scatter_selected(div, mode, w.sys)) return;
    const uint32_t W = w.win_hi - w.win_lo;
    for (uint32_t i = threadIdx.x; i < W; i += kScatterBlock) win[i] = 0.0;
    __syncthreads();
    const SlotGroup gr = groups[w.group];
    const int ns = gr.nslots;
    const uint32_t cb = sys_col[w.sys];
    const VT sc = scatter_scale<VT, kScatterBlock, kBeta>(div, mode, w.sys, bsum);
    const int64_t vld = m.ld / RPT;
    // FP32 windows accumulate in fixed point where the scale allows it
    const double fscale = window_scale<VT, kScatterBlock, kYmax>(fx, w.sys, sc, ns <= kMaxSegSlots);
    if (ns <= kMaxSegSlots) {
        int64_t slot[kMaxSegSlots];
        uint32_t off[kMaxSegSlots];
        const int s0 = slot_list[gr.first];
#pragma unroll
        for (int j = 0; j < kMaxSegSlots; j++) {
            const int sj = j < ns ? int(slot_list[gr.first + j]) : s0;
            slot[j] = int64_t(sj) * vld;
            off[j] = cb + m.base[sj] - w.win_lo;
        }
        // every column of the group inside this window
        const bool full = w.win_lo == cb + gr.col_lo && gr.col_hi - gr.col_lo <= W;
        auto rows_y = [&](auto* wn, auto vy) {
            using WT = std::remove_pointer_t<decltype(wn)>;
            constexpr bool VY = decltype(vy)::value;
            if (ns == 4)
                scatter_rows<4, WT, VY, VT, YT, IdxT, RPT>(m, w, ns, slot, off, y, sc, fscale, W, full, wn);
            else if (ns == 8)
                scatter_rows<8, WT, VY, VT, YT, IdxT, RPT>(m, w, ns, slot, off, y, sc, fscale, W, full, wn);
            else if (ns <= 2)
                scatter_rows<2, WT, VY, VT, YT, IdxT, RPT>(m, w, ns, slot, off, y, sc, fscale, W, full, wn);
            else if (ns <= 4)
                scatter_rows<4, WT, VY, VT, YT, IdxT, RPT>(m, w, ns, slot, off, y, sc, fscale, W, full, wn);
            else
                scatter_rows<8, WT, VY, VT, YT, IdxT, RPT>(m, w, ns, slot, off, y, sc, fscale, W, full, wn);
        };
        // 16-byte y loads need RPT values to fill them and y padded
        constexpr bool kVecY = RPT * sizeof(YT) % 16 == 0;
        auto rows = [&](auto* wn) {
            if constexpr (kVecY) {
                if (y_padded) {
                    rows_y(wn, std::true_type{});
                    return;
                }
            }
            rows_y(wn, std::false_type{});
        };
        if constexpr (std::is_same_v<VT, float>) {
            if (fscale > 0.0)
                rows(reinterpret_cast<unsigned long long*>(win));
            else
                rows(win);
        } else {
            rows(win);
        }
    } else {
        for (int64_t a = (w.row_begin & ~int64_t(RPT - 1)) + int64_t(RPT) * threadIdx.x; a < w.row_end;
             a += int64_t(RPT) * kScatterBlock) {
            bool ok[RPT];
            double yv[RPT];
#pragma unroll
            for (int i = 0; i < RPT; i++) {
                ok[i] = a + i >= w.row_begin && a + i < w.row_end;
                const double t = double(VT(y[min(a + i, w.row_end - 1)]) * sc);
                yv[i] = ok[i] ? t : 0.0;
            }
            const VecT* __restrict__ vec = reinterpret_cast<const VecT*>(m.idx + a);
            for (int j = 0; j < ns; j++) {
                const int sj = slot_list[gr.first + j];
                const VecT q = vec[int64_t(sj) * vld];
                const uint32_t o = cb + m.base[sj] - w.win_lo;
#pragma unroll
                for (int i = 0; i < RPT; i++) {
                    const uint32_t uc = o + V::get(q, i);
                    if (ok[i] && uc < W) atomicAdd(&win[uc], yv[i]);
                }
            }
        }
    }
    __syncthreads();
    store_window<VT>(win, W, fscale, part + w.part_off);
}

// Stage 1 for a matrix-free matrix: as k_scatter_tile, with every slot's column
// computed by its index tile.  A wave takes RPT runs of 64 rows a step; the
// columns turn from one slot per 16-lane group to one row per lane.  A group's
// slots are runs of whole patterns, so its tiles follow each other.  The windows
// are FP64 whatever VT is: the terms of up to 32 slots and a million rows meet
// in one window, and a fixed-point word with room for that many terms resolves
// no more than 2^-39 of max |y|.  20M rows of FIT12: 1,694 µs (2,570 with the
// lists evaluated digit by digit): 48 % of the cycles issue vector instructions,
// and the LDS is busy 48 % of them.  A window of 32 slots takes 1,099 cycles per
// 64 rows, where fixed point, whose adds are faster, took 790.
template <class VT, class YT, int RPT, bool kBeta = false>
__global__ __launch_bounds__(kScatterBlock) void k_scatter_tile_mf(PositionsView m,
                                                                   const ScatterWork* __restrict__ work,
                                                                   const SlotGroup* __restrict__ groups,
                                                                   const uint16_t* __restrict__ slot_list,
                                                                   const uint32_t* __restrict__ sys_col,
                                                                   const YT* __restrict__ y, LsqrScalars* div,
                                                                   int mode, FixedScale, int,
                                                                   VT* __restrict__ part, GridSys bsum)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double* win = reinterpret_cast<double*>(smem_raw);
    const ScatterWork w = uniform_load(work + blockIdx.x);
    if (!scatter_selected(div, mode, w.sys)) return;
    const uint32_t W = w.win_hi - w.win_lo;
    for (uint32_t i = threadIdx.x; i < W; i += kScatterBlock) win[i] = 0.0;
    __syncthreads();
    const SlotGroup gr = uniform_load(groups + w.group);
    const uint32_t cb = sys_col[w.sys];
    const VT sc = scatter_scale<VT, kScatterBlock, kBeta>(div, mode, w.sys, bsum);
    // the group's tiles: ntile of them, gr.nslots slots in all
    const int first = uniform_u16(slot_list, gr.first);
    const int tile0 = m.slot_tile(first), ntile = m.slot_tile(first + gr.nslots - 1) - tile0 + 1;
    const int lane = threadIdx.x & 63;
    // Run c of a step: the wave's rows a + c kScatterBlock + [0, 64).  The
    // next step's words and y load while this one is added.
    uint32_t tn[RPT][4];
    YT yn[RPT];
    auto load = [&](int64_t a) {
        const uint32_t* __restrict__ tw = reinterpret_cast<const uint32_t*>(m.tw + a);
        const YT* __restrict__ ya = y + a;
        const int last = int(min<int64_t>(w.row_end - a, int64_t(RPT) * kScatterBlock)) - 1;
        if (last >= (RPT - 1) * kScatterBlock + 63) {
#pragma unroll
            for (int c = 0; c < RPT; c++) {
#pragma unroll
                for (int p = 0; p < 4; p++)
                    tn[c][p] = tw[uint32_t(4 * (lane & 15) + (lane >> 4)) + uint32_t(4 * (c * kScatterBlock + 16 * p))];
                yn[c] = ya[uint32_t(lane) + uint32_t(c * kScatterBlock)];
            }
        } else {
#pragma unroll
            for (int c = 0; c < RPT; c++) {
#pragma unroll
                for (int p = 0; p < 4; p++)
                    tn[c][p] = tw[4 * min(c * kScatterBlock + 16 * p + (lane & 15), last) + (lane >> 4)];
                yn[c] = ya[min(c * kScatterBlock + lane, last)];
            }
        }
    };
    // (the wave's rows through scalar registers: its addresses are a
    // scalar base and one offset)
    int64_t a = w.row_begin + __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u);
    if (a < w.row_end) load(a);
    TileRegs tr = load_tile(m.tiles, tile0);
    int at = 0;
    for (; a < w.row_end; a += RPT * kScatterBlock) {
        Int4 b[RPT][4];
        double yv[RPT];
        bool ok[RPT];
#pragma unroll
        for (int c = 0; c < RPT; c++) {
#pragma unroll
            for (int p = 0; p < 4; p++) b[c][p] = expand_digits(tn[c][p]);
            ok[c] = a + c * kScatterBlock + lane < w.row_end;
            yv[c] = double(VT(yn[c]) * sc);
        }
        if (a + RPT * kScatterBlock < w.row_end) load(a + RPT * kScatterBlock);
        for (int t = 0; t < ntile; t++) {
            const IndexTile tl = tr.tile();
            const Int4 wt = tr.weights;
            const int number = tile0 + at;
            at = at + 1 < ntile ? at + 1 : 0;
            tr = load_tile(m.tiles, tile0 + at);
            const uint32_t off = cb + tl.col_offset - w.win_lo;
#pragma unroll
            for (int c = 0; c < RPT; c++) {
                uint32_t ci[4];
                tile_columns(tl, number, m.tiles, wt, b[c], ci);
                transpose_groups(ci);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const uint32_t uc = off + ci[j];
                    if (j < tl.nslots && ok[c] && uc < W) atomicAdd(&win[uc], yv[c]);
                }
            }
        }
    }
    __syncthreads();
    store_window<VT>(win, W, 0.0, part + w.part_off);
}

// Stage 2: z[c] = sum of the window's chunk slices, in chunk order
// (the order of the slices is fixed; the sums inside a slice took the LDS
// atomics' arrival order); columns outside every window get 0.
// Column c's sum over the slices of its window: integer counts stay
// integer; real sums add up in FP64, in chunk order, up to sixteen slices
// loaded ahead of their additions (a load's latency, not the bytes, is what a
// column of 20 to 60 slices waits for).  Whole sixteens, then the smallest step
// that holds the rest: a batch's columns have one slice or a few, and sixteen
// loads (with a 64-bit multiply each for the address) for those took 17.8 µs
// where one takes 7.3 (30 systems of 102,222 columns); 100,000 rows, 25 to 38
// slices a column, 4.5 -> 2.7, 1M rows 5.0 -> 3.3.
template <class T>
__device__ __forceinline__ std::conditional_t<std::is_integral_v<T>, T, double>
reduce_column(const T* __restrict__ part, const ReduceWork& w, int64_t c)
{
    using AccT = std::conditional_t<std::is_integral_v<T>, T, double>;
    const T* __restrict__ p = part + w.part_off + (c - w.col_begin);
    AccT s = AccT(0);
    int left = w.nchunk;
    if (left == 1) return s + AccT(*p);
    // the next `ahead` slices (the last one again past the end)
    auto step = [&](auto ahead, auto whole) {
        constexpr int kAhead = decltype(ahead)::value;
        T t[kAhead];
#pragma unroll
        for (int q = 0; q < kAhead; q++) {
            t[q] = *p;
            if (decltype(whole)::value || q + 1 < left) p += w.stride;
        }
#pragma unroll
        for (int q = 0; q < kAhead; q++)
            if (decltype(whole)::value || q < left) s += AccT(t[q]);
        left -= kAhead;
    };
    while (left >= 16) step(std::integral_constant<int, 16>{}, std::true_type{});
    if (left > 8) step(std::integral_constant<int, 16>{}, std::false_type{});
    else if (left > 4) step(std::integral_constant<int, 8>{}, std::false_type{});
    else if (left > 2) step(std::integral_constant<int, 4>{}, std::false_type{});
    else if (left > 0) step(std::integral_constant<int, 2>{}, std::false_type{});
    return s;
}

template <class T, class ZT>
__global__ __launch_bounds__(kRowBlock) void k_scatter_reduce(const ReduceWork* __restrict__ work,
                                                              const T* __restrict__ part, ZT* __restrict__ z,
                                                              const LsqrScalars* div, int mode)
{
    const ReduceWork w = work[blockIdx.x];
    if (!scatter_selected(div, mode, w.sys)) return;
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) z[c] = ZT(reduce_column(part, w, c));
}

// Jacobi of A^T A (Math/MatrixCSR.cpp:21-47): diag_c = sum over rows of the
// squared multiplicity of c in the row.  A row's columns of one slot group
// (repeats can only occur within a group, of at most kMaxSegSlots slots) are
// loaded once into registers, and the occurrences of a column add up to its
// mult^2.  Counts are exact 32-bit integers.
template <class View>
__global__ __launch_bounds__(kScatterBlock) void k_jacobi_part(View m, const ScatterWork* __restrict__ work,
                                                               const SlotGroup* __restrict__ groups,
                                                               const uint16_t* __restrict__ slot_list,
                                                               const uint32_t* __restrict__ sys_col,
                                                               uint32_t* __restrict__ part)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    uint32_t* win = reinterpret_cast<uint32_t*>(smem_raw);
    const ScatterWork w = work[blockIdx.x];
    const uint32_t W = w.win_hi - w.win_lo;
    for (uint32_t i = threadIdx.x; i < W; i += kScatterBlock) win[i] = 0u;
    __syncthreads();
    const SlotGroup gr = uniform_load(groups + w.group);
    const uint32_t cb = sys_col[w.sys];
    const int ns = gr.nslots;
    // four rows a thread per step, all their entries loaded before any add
    constexpr int kRows = 4;
    // stored indices: the group's slots are looked up once, outside the row
    // loop (slots past the group's end repeat its first, unused)
    using SlotRef = std::conditional_t<is_slot_major<View>::value, typename SlotRefOf<View>::type, int>;
    SlotRef sref[kMaxSegSlots];
    if constexpr (is_slot_major<View>::value) {
#pragma unroll
        for (int j = 0; j < kMaxSegSlots; j++) sref[j] = m.slot(uniform_u16(slot_list, gr.first + (j < ns ? j : 0)));
    }
    const int64_t last = w.row_end - 1;
    for (int64_t r0 = w.row_begin + threadIdx.x; r0 < w.row_end; r0 += kRows * kScatterBlock) {
        uint32_t c[kRows][kMaxSegSlots];
#pragma unroll
        for (int u = 0; u < kRows; u++) {
            const int64_t r = r0 + int64_t(u) * kScatterBlock;
            const bool valid = r < w.row_end;
#pragma unroll
            for (int j = 0; j < kMaxSegSlots; j++) {
                if constexpr (is_slot_major<View>::value) {
                    // every load issued (a clamped row, the group's first slot
                    // past its end), then the unused ones dropped: no branch
                    // around a load, so all of them are in flight together
                    const uint32_t v = cb + sref[j].col(min(r, last));
                    c[u][j] = (valid && j < ns) ? v : 0xFFFFFFFFu;
                } else {
                    c[u][j] = (valid && j < ns) ? cb + m.col(slot_list[gr.first + j], r) : 0xFFFFFFFFu;
                }
            }
        }
        // a column that m slots of the row hold must gain m^2 = 1 + 3 + ...
        // + (2m - 1): its k-th occurrence adds 2k - 1, i.e. one plus twice
        // the number of earlier slots holding it
#pragma unroll
        for (int u = 0; u < kRows; u++) {
#pragma unroll
            for (int j = 0; j < kMaxSegSlots; j++) {
                const uint32_t uc = c[u][j] - w.win_lo;
                if (c[u][j] == 0xFFFFFFFFu || uc >= W) continue;
                uint32_t before = 0;
#pragma unroll
                for (int t = 0; t < j; t++) before += c[u][t] == c[u][j] ? 1u : 0u;
                atomicAdd(&win[uc], 2u * before + 1u);
            }
        }
    }
    __syncthreads();
    uint32_t* __restrict__ out = part + w.part_off;
    for (uint32_t i = threadIdx.x; i < W; i += kScatterBlock) out[i] = win[i];
}

// 1 / diag in float, exactly as inv() of the reference (1/0 = inf).
__global__ void k_jacobi_finish(const uint32_t* __restrict__ cnt, int64_t n, float* __restrict__ d)
{
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        d[i] = 1.0f / float(cnt[i]);
}

// Column scaling of LSQR: D = 1/|a_c| = sqrt(jacobi), 1 for empty columns.
__global__ void k_colscale(const uint32_t* __restrict__ cnt, int64_t n, double* __restrict__ D)
{
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        D[i] = cnt[i] ? 1.0 / sqrt(double(cnt[i])) : 1.0;
}

// ------------------------------------------------------------ LSQR cols ----
// LSQR step 2 (Math/Solver.h:162), fused with the column reduction of
// A^T (u / beta): per column z = the slices' sum rounded to VT (as
// k_scatter_reduce writes it), then vbar = D z - beta v and the block
// partials of |vbar|^2, one block per reduce item (g: the reduce items of
// each system); k_lsqr_step (LSQR) or k_lsmr_rot (LSMR) finishes alpha.  The
// system's first block also keeps rhobar, phibar and stop aside for
// k_lsqr_step, whose blocks read them while its first block updates them.
// (A grid-wide last-block ticket here would cost every block an L2
// write-back and invalidate on gfx950.)
template <class VT>
__global__ __launch_bounds__(kRowBlock) void k_lsqr_reduce_v(const ReduceWork* __restrict__ work,
                                                             const VT* __restrict__ part,
                                                             const double* __restrict__ D, double* __restrict__ v,
                                                             GridSys g, LsqrScalars* scal)
{
    __shared__ double sh[kRowBlock / 64];
    const ReduceWork w = work[blockIdx.x];
    LsqrScalars* st = &scal[w.sys];
    if (!st->active) return;
    if (threadIdx.x == 0 && int(blockIdx.x) == g.blk_first[w.sys]) {
        st->rhobar0 = st->rhobar;
        st->phibar0 = st->phibar;
        st->stop0 = st->stop;
    }
    const double beta = st->beta;
    double acc = 0.0;
    if (st->stop == 0)
        for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) {
            const double zc = double(VT(reduce_column(part, w, c)));
            const double vb = D[c] * zc - beta * v[c];
            v[c] = vb;
            acc += vb * vb;
        }
    acc = block_sum<kRowBlock>(acc, sh);
    if (threadIdx.x == 0) g.partials[2 * blockIdx.x] = acc;
}

// The LSQR rotation and update in one launch (Math/Solver.h:165-175).  Every
// block of a system forms alpha = |vbar| from k_lsqr_reduce_v's partials and
// the rotation (rho, c, s, theta, phi, phibar) from the rhobar, phibar and
// stop that k_lsqr_reduce_v kept aside -- the same values in every block --
// and updates its columns: v = vbar / alpha, vd = D v, y += (phi/rho) w,
// w = v - (theta/rho) w.  The system's first column block stores the new
// state, with the device-side stop; the fields it writes are read by no
// block of this launch.
template <class VT>
__global__ __launch_bounds__(kRowBlock) void k_lsqr_step(const ColWork* __restrict__ work, GridSys g,
                                                         const double* __restrict__ D, double* __restrict__ v,
                                                         VT* __restrict__ vd, double* __restrict__ w_,
                                                         double* __restrict__ y, LsqrScalars* scal)
{
    __shared__ double sh[kRowBlock / 64];
    const ColWork w = work[blockIdx.x];
    LsqrScalars* st = &scal[w.sys];
    if (!st->active) return;
    const double s = system_sum<kRowBlock>(g, w.sys, sh);
    const bool writer = w.first != 0 && threadIdx.x == 0;
    if (st->stop0 != 0) {
        // the iteration after the stop: no further step
        if (writer) {
            st->stop = 2;
            st->step_x = 0.0;
            st->step_w = 0.0;
        }
        return;
    }
    const double beta = st->beta, rhobar = st->rhobar0, phibar = st->phibar0;
    const double alpha = sqrt(s);
    const double rho = sqrt(rhobar * rhobar + beta * beta);
    const double c = rho != 0.0 ? rhobar / rho : 0.0;
    const double sn = rho != 0.0 ? beta / rho : 0.0;
    const double theta = sn * alpha;
    const double phi = c * phibar;
    const double sx = rho != 0.0 ? phi / rho : 0.0;
    const double sw = rho != 0.0 ? theta / rho : 0.0;
    if (writer) {
        const double phibar_new = sn * phibar;
        st->rhobar = -c * alpha;
        st->phibar = phibar_new;
        st->step_x = sx;
        st->step_w = sw;
        st->alpha = alpha;
        st->nres = phibar_new * alpha * fabs(c);
        st->rnorm = phibar_new;
        st->anorm2 += st->beta2;
        st->anorm2 += s;
        st->iters += 1;
        // met the target: this iteration's step is the last (a rank-deficient
        // system that continued would iterate on rounding noise)
        if (st->target > 0.0 && st->nres <= st->target * st->nres0) st->stop = 1;
    }
    const double ia = alpha != 0.0 ? 1.0 / alpha : 0.0;
    for (int64_t c0 = w.col_begin + threadIdx.x; c0 < w.col_end; c0 += kRowBlock) {
        const double vn = v[c0] * ia;
        v[c0] = vn;
        vd[c0] = VT(D[c0] * vn);
        const double wc = w_[c0];
        y[c0] += sx * wc;
        w_[c0] = vn - sw * wc;
    }
}

// LSQR start on the columns (Math/Solver.h:146-150), from an FP64 A^T u_raw:
//   vbar = D z / beta, alpha = |vbar|; also |z|^2 = |A^T src|^2 into reduce_b.
template <class ZT>
__global__ __launch_bounds__(kRowBlock) void k_lsqr_init_v(const ColWork* __restrict__ work,
                                                           const double* __restrict__ D, const ZT* __restrict__ z,
                                                           double* __restrict__ v, GridSys g, const LsqrScalars* scal)
{
    __shared__ double sh[kRowBlock / 64];
    const ColWork w = work[blockIdx.x];
    const LsqrScalars* st = &scal[w.sys];
    if (!st->active || !st->restart) return;
    const double ib = st->beta != 0.0 ? 1.0 / st->beta : 0.0;
    double a0 = 0.0, a1 = 0.0;
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) {
        const double zc = double(z[c]);
        const double vb = D[c] * zc * ib;
        v[c] = vb;
        a0 += vb * vb;
        a1 += zc * zc;
    }
    a0 = block_sum<kRowBlock>(a0, sh);
    a1 = block_sum<kRowBlock>(a1, sh);
    if (threadIdx.x == 0) {
        g.partials[2 * blockIdx.x] = a0;
        g.partials[2 * blockIdx.x + 1] = a1;
    }
}

struct FinishLsqrInit {
    LsqrScalars* scal;
    __device__ bool begin(int sys) const { return scal[sys].active && scal[sys].restart; }
    __device__ void finish(int sys, double s0, double s1) const
    {
        LsqrScalars* st = &scal[sys];
        const double alpha = sqrt(s0);
        st->alpha = alpha;
        st->rhobar = alpha;
        st->phibar = st->beta;
        st->nres0 = alpha * st->beta;
        st->nres = st->nres0;
        st->rnorm = st->beta;
        st->anorm2 = s0 + st->beta * 0.0;
        st->reduce_b = s1;
        st->iters = 0;
        st->stop = 0;
    }
};

// v = vbar/alpha, vd = D v, w = v, y = 0.
template <class VT>
__global__ __launch_bounds__(kRowBlock) void k_lsqr_init_w(const ColWork* __restrict__ work,
                                                           const double* __restrict__ D, double* __restrict__ v,
                                                           VT* __restrict__ vd, double* __restrict__ w_,
                                                           double* __restrict__ y, const LsqrScalars* scal)
{
    const ColWork w = work[blockIdx.x];
    const LsqrScalars* st = &scal[w.sys];
    if (!st->active || !st->restart) return;
    const double ia = st->alpha != 0.0 ? 1.0 / st->alpha : 0.0;
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) {
        const double vn = v[c] * ia;
        v[c] = vn;
        vd[c] = VT(D[c] * vn);
        w_[c] = vn;
        y[c] = 0.0;
    }
}

// x += D y (back to the unscaled space), y = 0, keeping the x before in
// xprev; for the selected systems (active and restart).
__global__ __launch_bounds__(kRowBlock) void k_lsqr_apply(const ColWork* __restrict__ work,
                                                          const double* __restrict__ D, double* __restrict__ y,
                                                          double* __restrict__ x, double* __restrict__ xprev,
                                                          const LsqrScalars* scal)
{
    const ColWork w = work[blockIdx.x];
    if (!scal[w.sys].active || !scal[w.sys].restart) return;
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) {
        const double xc = x[c];
        xprev[c] = xc;
        x[c] = xc + D[c] * y[c];
        y[c] = 0.0;
    }
}

// Undoes the last k_lsqr_apply of the selected systems: x = xprev.
__global__ __launch_bounds__(kRowBlock) void k_lsqr_undo(const ColWork* __restrict__ work,
                                                         const double* __restrict__ D, double* __restrict__ y,
                                                         double* __restrict__ x, double* __restrict__ xprev,
                                                         const LsqrScalars* scal)
{
    (void)D;
    (void)y;
    const ColWork w = work[blockIdx.x];
    if (!scal[w.sys].active || !scal[w.sys].restart) return;
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) x[c] = xprev[c];
}

// ------------------------------------------------------------ LSMR ------
// The symmetric Givens rotation of Math/Solver.h:193-217 (scipy's sym_ortho).
__device__ __forceinline__ void sym_ortho(double a, double b, double& c, double& s, double& r)
{
    const double sa = a < 0 ? -1.0 : (a > 0 ? 1.0 : 0.0), sb = b < 0 ? -1.0 : (b > 0 ? 1.0 : 0.0);
    if (b == 0.0) {
        c = sa;
        s = 0.0;
        r = fabs(a);
    } else if (a == 0.0) {
        c = 0.0;
        s = sb;
        r = fabs(b);
    } else if (fabs(b) > fabs(a)) {
        const double tau = a / b;
        s = sb / sqrt(1.0 + tau * tau);
        c = s * tau;
        r = b / s;
    } else {
        const double tau = b / a;
        c = sa / sqrt(1.0 + tau * tau);
        s = c * tau;
        r = a / c;
    }
}

// LSMR's rotations (Math/Solver.h:255-275), one block per system: alpha =
// |vbar| from k_lsqr_reduce_v's partials, then the two rotations, zeta and
// the update coefficients; nres = |zetabar| (= |A^T r_k|) and the device-side
// stop as in k_lsqr_step.
__global__ __launch_bounds__(kRowBlock) void k_lsmr_rot(GridSys g, LsqrScalars* scal, LsmrState* lsmr)
{
    __shared__ double sh[kRowBlock / 64];
    const int sys = blockIdx.x;
    LsqrScalars* st = &scal[sys];
    if (!st->active) return;
    double sum = 0.0;
    for (int i = threadIdx.x; i < g.blk_count[sys]; i += kRowBlock) sum += g.partials[2 * (g.blk_first[sys] + i)];
    sum = block_sum<kRowBlock>(sum, sh);
    if (threadIdx.x != 0) return;
    LsmrState* ls = &lsmr[sys];
    if (st->stop != 0) {
        st->stop = 2;
        return;
    }
    const double beta = st->beta, alpha = sqrt(sum);
    const double rho_old = ls->rho, rhobar_old = ls->rhobar;
    double c, s, rho;
    sym_ortho(ls->alphabar, beta, c, s, rho);
    const double theta_new = s * alpha;
    ls->alphabar = c * alpha;
    const double thetabar = ls->sbar * rho;
    double cbar, sbar, rhobar;
    sym_ortho(ls->cbar * rho, theta_new, cbar, sbar, rhobar);
    const double zeta = cbar * ls->zetabar;
    ls->zetabar = -sbar * ls->zetabar;
    ls->cbar = cbar;
    ls->sbar = sbar;
    ls->rho = rho;
    ls->rhobar = rhobar;
    ls->k_hb = -thetabar * rho / (rho_old * rhobar_old);
    ls->k_x = zeta / (rho * rhobar);
    ls->k_h = rho != 0.0 ? -theta_new / rho : 0.0;
    st->alpha = alpha;
    st->nres = fabs(ls->zetabar);
    st->anorm2 += st->beta2;
    st->anorm2 += sum;
    st->iters += 1;
    if (st->target > 0.0 && st->nres <= st->target * st->nres0) st->stop = 1;
}

// LSMR's vector updates (Math/Solver.h:277-283): v = vbar / alpha, vd = D v,
// hbar = h + k_hb hbar, x += k_x hbar, h = v + k_h h.
template <class VT>
__global__ __launch_bounds__(kRowBlock) void k_lsmr_update(const ColWork* __restrict__ work,
                                                           const double* __restrict__ D, double* __restrict__ v,
                                                           VT* __restrict__ vd, double* __restrict__ h,
                                                           double* __restrict__ hb, double* __restrict__ x,
                                                           const LsqrScalars* scal, const LsmrState* lsmr)
{
    const ColWork w = work[blockIdx.x];
    const LsqrScalars* st = &scal[w.sys];
    if (!st->active || st->stop > 1) return;
    const LsmrState* ls = &lsmr[w.sys];
    const double ia = st->alpha != 0.0 ? 1.0 / st->alpha : 0.0;
    const double khb = ls->k_hb, kx = ls->k_x, kh = ls->k_h;
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) {
        const double vn = v[c] * ia;
        v[c] = vn;
        vd[c] = VT(D[c] * vn);
        const double hc = h[c];
        const double hbn = hc + khb * hb[c];
        hb[c] = hbn;
        x[c] += kx * hbn;
        h[c] = vn + kh * hc;
    }
}

// LSMR's start after the LSQR start of each system (x = 0): the rotation
// state alphabar = alpha, zetabar = alpha beta, rho = rhobar = cbar = 1,
// sbar = 0 (Math/Solver.h:238-252).
__global__ void k_lsmr_init(int nsys, const LsqrScalars* scal, LsmrState* lsmr)
{
    const int sys = blockIdx.x * blockDim.x + threadIdx.x;
    if (sys >= nsys) return;
    LsmrState* ls = &lsmr[sys];
    ls->alphabar = scal[sys].alpha;
    ls->zetabar = scal[sys].alpha * scal[sys].beta;
    ls->rho = ls->rhobar = ls->cbar = 1.0;
    ls->sbar = 0.0;
    ls->k_hb = ls->k_x = ls->k_h = 0.0;
}

// |z|^2 per system into reduce_b (used for |A^T b| and |A^T r|): the block
// partials (slot 0; slot 1 is cleared), summed by FinishNorm2.
template <class ZT>
__global__ __launch_bounds__(kRowBlock) void k_cols_norm2(const ColWork* __restrict__ work, const ZT* __restrict__ z,
                                                          GridSys g, const LsqrScalars* scal)
{
    __shared__ double sh[kRowBlock / 64];
    const ColWork w = work[blockIdx.x];
    if (!scal[w.sys].active) return;
    double acc = 0.0;
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) {
        const double zc = double(z[c]);
        acc += zc * zc;
    }
    acc = block_sum<kRowBlock>(acc, sh);
    if (threadIdx.x == 0) {
        g.partials[2 * blockIdx.x] = acc;
        g.partials[2 * blockIdx.x + 1] = 0.0;
    }
}

struct FinishNorm2 {
    LsqrScalars* scal;
    __device__ bool begin(int sys) const { return scal[sys].active; }
    __device__ void finish(int sys, double s0, double) const { scal[sys].reduce_b = s0; }
};

// out = D y (the unscaled solution of a column-scaled LSQR).
__global__ void k_scale_mul(const double* __restrict__ D, const double* __restrict__ y, int64_t n,
                            double* __restrict__ out)
{
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        out[i] = D[i] * y[i];
}

// ------------------------------------------------------------ PCG ---------
// PCG on A^T A with a diagonal preconditioner (Math/Solver.h:78-117); the
// FP64 scalars live on the device.  An iteration is five launches: the gather
// t = A p, the window tiles of A^T t, then
//   k_pcg_reduce_q  q = A^T t (the slices' sum per column) and the block
//                   partials of p.q, one block per reduce item;
//   k_pcg_update    alpha = rz / pq, formed by every block from those partials
//                   (the same value in each), then x, r, zz = P r and the
//                   partials of r.zz and r.r;
//   k_pcg_p         beta = rz' / rz formed the same way, then p = zz + beta p.
// A system's first column block stores the scalars.  k_pcg_update keeps rz
// aside as rz0, so that k_pcg_p's blocks read the old rz while its first
// block stores the new one.  faithful: the scalars are rounded to VT before
// use, as in the float solver.
template <class VT>
__global__ __launch_bounds__(kRowBlock) void k_pcg_reduce_q(const ReduceWork* __restrict__ work,
                                                            const VT* __restrict__ part, const VT* __restrict__ p,
                                                            VT* __restrict__ q, GridSys g, const PcgScalars* scal)
{
    __shared__ double sh[kRowBlock / 64];
    const ReduceWork w = work[blockIdx.x];
    if (!scal[w.sys].active) return;
    double acc = 0.0;
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) {
        const VT qc = VT(reduce_column(part, w, c));
        q[c] = qc;
        acc += double(p[c]) * double(qc);
    }
    acc = block_sum<kRowBlock>(acc, sh);
    if (threadIdx.x == 0) g.partials[2 * blockIdx.x] = acc;
}

// gq: k_pcg_reduce_q's partials; g: this launch's
template <class VT>
__global__ __launch_bounds__(kRowBlock) void k_pcg_update(const ColWork* __restrict__ work, const VT* __restrict__ P,
                                                          const VT* __restrict__ p, const VT* __restrict__ q,
                                                          VT* __restrict__ x, VT* __restrict__ r, VT* __restrict__ zz,
                                                          GridSys gq, GridSys g, PcgScalars* scal)
{
    __shared__ double sh[kRowBlock / 64];
    const ColWork w = work[blockIdx.x];
    PcgScalars* st = &scal[w.sys];
    if (!st->active) return;
    const double pq = system_sum<kRowBlock>(gq, w.sys, sh);
    const double alpha = pq != 0.0 ? st->rz / pq : 0.0;
    if (w.first && threadIdx.x == 0) {
        st->pq = pq;
        st->alpha = alpha;
        st->rz0 = st->rz;
    }
    const VT a = VT(alpha);
    double a0 = 0.0, a1 = 0.0;
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) {
        x[c] += a * p[c];
        const VT rc = r[c] - a * q[c];
        r[c] = rc;
        const VT zc = P[c] * rc;
        zz[c] = zc;
        a0 += double(rc) * double(zc);
        a1 += double(rc) * double(rc);
    }
    a0 = block_sum<kRowBlock>(a0, sh);
    a1 = block_sum<kRowBlock>(a1, sh);
    if (threadIdx.x == 0) {
        g.partials[2 * blockIdx.x] = a0;
        g.partials[2 * blockIdx.x + 1] = a1;
    }
}

// rz' (slot 0 of k_pcg_update's partials), rr (slot 1), beta = rz' / rz;
// p = zz + beta p (k_pcg_reduce_q writes every column of q).
template <class VT>
__global__ __launch_bounds__(kRowBlock) void k_pcg_p(const ColWork* __restrict__ work, const VT* __restrict__ zz,
                                                     VT* __restrict__ p, GridSys g, PcgScalars* scal)
{
    __shared__ double sh[kRowBlock / 64];
    const ColWork w = work[blockIdx.x];
    PcgScalars* st = &scal[w.sys];
    if (!st->active) return;
    double rz, rr;
    system_sum2<kRowBlock>(g, w.sys, sh, rz, rr);
    const double beta = st->rz0 != 0.0 ? rz / st->rz0 : 0.0;
    if (w.first && threadIdx.x == 0) {
        st->beta = beta;
        st->rz = rz;
        st->rr = rr;
        st->iters += 1;
    }
    const VT b = VT(beta);
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) {
        p[c] = zz[c] + b * p[c];
    }
}

// PCG start: r = rhs (A^T b, x0 = 0), zz = P r, p = zz, the partials of
// rz = r.zz and r.r (FinishPcgInit).
template <class VT>
__global__ __launch_bounds__(kRowBlock) void k_pcg_init(const ColWork* __restrict__ work, const VT* __restrict__ P,
                                                        const VT* __restrict__ rhs_r, VT* __restrict__ zz, VT* __restrict__ p,
                                                        VT* __restrict__ x, GridSys g, const PcgScalars* scal)
{
    __shared__ double sh[kRowBlock / 64];
    const ColWork w = work[blockIdx.x];
    if (!scal[w.sys].active) return;
    double a0 = 0.0, a1 = 0.0;
    for (int64_t c = w.col_begin + threadIdx.x; c < w.col_end; c += kRowBlock) {
        const VT rc = rhs_r[c];
        const VT zc = P[c] * rc;
        zz[c] = zc;
        p[c] = zc;
        x[c] = VT(0);
        a0 += double(rc) * double(zc);
        a1 += double(rc) * double(rc);
    }
    a0 = block_sum<kRowBlock>(a0, sh);
    a1 = block_sum<kRowBlock>(a1, sh);
    if (threadIdx.x == 0) {
        g.partials[2 * blockIdx.x] = a0;
        g.partials[2 * blockIdx.x + 1] = a1;
    }
}

struct FinishPcgInit {
    PcgScalars* scal;
    __device__ bool begin(int sys) const { return scal[sys].active; }
    __device__ void finish(int sys, double s0, double s1) const
    {
        scal[sys].rz = s0;
        scal[sys].rr = s1;
        scal[sys].iters = 0;
    }
};

// DiagonalPreconditioner (Math/Solver.h:29-34): non-normal entries become 1.
template <class VT>
__global__ void k_precond_from_jacobi(const float* __restrict__ jac, int64_t n, VT* __restrict__ P)
{
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x) {
        const float d = jac[i];
        P[i] = VT(__builtin_isnormal(d) ? d : 1.0f);
    }
}

// ------------------------------------------------------------ evaluator ----
// sum_s w[idx[s]] of one row's k consecutive entries, in slot order from zero
// (Pattern/Evaluator.cpp:48-54 sums the same terms in the same order; entries
// outside [0, cols) add nothing).  A thread takes a row: up to twenty entries and
// then their weights are loaded together (V = 2: pairs, for an even k and rows
// aligned to 8 bytes), in steps of twenty and then the smallest that holds the
// rest: 262,144 rows of 4 slots 3.9 µs, of 12 slots 9.5, of 54 slots 37 (8.2, 11.7
// and 50 with twenty loads a step whatever is left).
template <class VT, int V>
__device__ __forceinline__ VT row_gather(const int32_t* __restrict__ row, int k, const VT* __restrict__ w,
                                         uint32_t cols)
{
    VT acc = VT(0);
    int s0 = 0;
    // (the last entries again past the row's end)
    auto step = [&](auto ahead, auto whole) {
        constexpr int kAhead = decltype(ahead)::value;
        constexpr bool kWhole = decltype(whole)::value;
        int32_t c[kAhead];
        VT x[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; j += V) {
            const int32_t* __restrict__ p = row + (kWhole ? s0 + j : min(s0 + j, k - V));
            if constexpr (V == 2) {
                const int2 t = *reinterpret_cast<const int2*>(p);
                c[j] = t.x;
                c[j + 1] = t.y;
            } else {
                c[j] = p[0];
            }
        }
#pragma unroll
        for (int j = 0; j < kAhead; j++) x[j] = w[min(uint32_t(c[j]), cols - 1)];
#pragma unroll
        for (int j = 0; j < kAhead; j++) {
            if (kWhole || s0 + j < k) acc = uint32_t(c[j]) < cols ? acc + x[j] : acc;
        }
        s0 += kAhead;
    };
    while (k - s0 >= 20) step(std::integral_constant<int, 20>{}, std::true_type{});
    const int left = k - s0;
    if (left > 12) step(std::integral_constant<int, 20>{}, std::false_type{});
    else if (left > 8) step(std::integral_constant<int, 12>{}, std::false_type{});
    else if (left > 4) step(std::integral_constant<int, 8>{}, std::false_type{});
    else if (left > 0) step(std::integral_constant<int, 4>{}, std::false_type{});
    return acc;
}

// Forward of the differentiable evaluator: out[r] = the sum of row r (65,536
// rows of FIT4: 6.0 µs, 9.6 with an entry, then its weight, at a time).
template <class VT, int V>
__global__ __launch_bounds__(kRowBlock) void k_eval_forward(const int32_t* __restrict__ idx, int64_t B, int k,
                                                            const VT* __restrict__ w, uint32_t cols,
                                                            VT* __restrict__ out)
{
    const int64_t r = blockIdx.x * int64_t(kRowBlock) + threadIdx.x;
    if (r >= B) return;
    out[r] = row_gather<VT, V>(idx + r * k, k, w, cols);
}

// The Huber loss of d = pred - target (0.5 d^2 inside [-delta, delta],
// delta (|d| - delta/2) outside) and the gradient of the batch mean,
// clamp(d, -delta, delta) / B.
__device__ __forceinline__ double huber_term(float d, float delta, int64_t B, float& grad)
{
    const float ad = fabsf(d);
    grad = fminf(fmaxf(d, -delta), delta) / float(B);
    return ad < delta ? 0.5 * double(d) * double(d) : double(delta) * (double(ad) - 0.5 * double(delta));
}

// One Huber-loss training step, forward half: for the minibatch rows sel[b]
// the prediction (the evaluator's gather-sum, slot order from zero), the loss
// and g[b] (huber_term); the block sums of the losses (FP64) go to
// part[blockIdx.x], and the entries to rows[s * B + b] -- slot-major, so that
// both these stores and the backward's loads are whole lines.
// A wave takes 64 rows, up to kTrainChunk slots at a time: its lanes load the
// entries as they lie in memory (row after row, so that a load touches the
// lines of a few rows and not of 64) into the wave's part of the LDS, from
// which each lane takes its row.  65,536 rows of FIT4 out of 5M: 11.4 µs (12.2
// with a lane loading its own row, 16.5 three pairs of entries at a time), with
// one wave a SIMD the latency of its loads one after the other: the shuffled
// order, the rows, the weights.
constexpr int kTrainChunk = 32;
__global__ __launch_bounds__(kRowBlock) void k_train_forward(const int32_t* __restrict__ idx,
                                                             const int64_t* __restrict__ sel, int64_t B, int k,
                                                             const float* __restrict__ w, uint32_t cols,
                                                             const float* __restrict__ target, float delta,
                                                             float* __restrict__ g, double* __restrict__ part,
                                                             int32_t* __restrict__ rows)
{
    constexpr int kWaves = kRowBlock / 64, kPitch = kTrainChunk + 1, kAhead = 16;
    __shared__ double sh[kWaves];
    __shared__ int64_t at[kWaves][64];            // first entry of each row
    __shared__ int32_t ent[kWaves][64 * kPitch];  // entry (row, slot of the chunk)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t b = blockIdx.x * int64_t(kRowBlock) + threadIdx.x, wave0 = b - lane;
    double loss = 0.0;
    if (wave0 < B) {
        const int64_t r = sel[min(b, B - 1)];
        const float t = target[r];
        at[wave][lane] = r * k;
        int32_t* __restrict__ dst = rows + b;
        float acc = 0.0f;
        for (int s0 = 0; s0 < k; s0 += kTrainChunk) {
            const int nc = min(kTrainChunk, k - s0);
            // e / nc for e < 64 nc, exact for nc <= 32
            const uint32_t inv = (65536u + uint32_t(nc) - 1u) / uint32_t(nc);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            for (int i0 = 0; i0 < nc; i0 += kAhead) {
                int32_t c[kAhead];
                int place[kAhead];
#pragma unroll
                for (int i = 0; i < kAhead; i++) {
                    const uint32_t e = uint32_t(lane + 64 * min(i0 + i, nc - 1));
                    const uint32_t row = (e * inv) >> 16, s = e - row * uint32_t(nc);
                    place[i] = int(row) * kPitch + int(s);
                    c[i] = idx[at[wave][row] + s0 + int(s)];
                }
#pragma unroll
                for (int i = 0; i < kAhead; i++) ent[wave][place[i]] = c[i];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            for (int j0 = 0; j0 < nc; j0 += kAhead) {
                int32_t c[kAhead];
                float x[kAhead];
#pragma unroll
                for (int j = 0; j < kAhead; j++) c[j] = ent[wave][lane * kPitch + min(j0 + j, nc - 1)];
#pragma unroll
                for (int j = 0; j < kAhead; j++) x[j] = w[min(uint32_t(c[j]), cols - 1)];
#pragma unroll
                for (int j = 0; j < kAhead; j++)
                    if (j0 + j < nc) {
                        acc = uint32_t(c[j]) < cols ? acc + x[j] : acc;
                        if (b < B) dst[(s0 + j0 + j) * B] = c[j];
                    }
            }
        }
        if (b < B) {
            float gr;
            loss = huber_term(acc - t, delta, B, gr);
            g[b] = gr;
        }
    }
    loss = block_sum<kRowBlock>(loss, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = loss;
}

// The step's Adam update (torch.optim.Adam without weight decay or amsgrad:
// m = b1 m + (1 - b1) g, v = b2 v + (1 - b2) g^2, w -= lr / (1 - b1^t) * m /
// (sqrt(v) / sqrt(1 - b2^t) + eps)); block 0 also adds the step's mean loss
// (the forward's block sums, reduced in a fixed order, / B) to *loss.
struct AdamStep {
    float lr, b1, b2, eps, bias1, bias2_sqrt;
};
__device__ __forceinline__ void adam_update(float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
                                            int64_t c, float gc, const AdamStep& a)
{
    const float mc = a.b1 * m[c] + (1.0f - a.b1) * gc;
    const float vc = a.b2 * v[c] + (1.0f - a.b2) * gc * gc;
    m[c] = mc;
    v[c] = vc;
    w[c] -= (a.lr / a.bias1) * mc / (sqrtf(vc) / a.bias2_sqrt + a.eps);
}

// The loss of the step: the forward's block partials, in a fixed order, / B.
__device__ __forceinline__ void add_loss(const double* __restrict__ part, int nparts, int64_t B,
                                         double* __restrict__ loss)
{
    __shared__ double sh[kRowBlock / 64];
    double s = 0.0;
    for (int i = threadIdx.x; i < nparts; i += kRowBlock) s += part[i];
    s = block_sum<kRowBlock>(s, sh);
    if (threadIdx.x == 0) *loss += s / double(B);
}

__global__ __launch_bounds__(kRowBlock) void k_adam(float* __restrict__ w, const float* __restrict__ grad,
                                                    float* __restrict__ m, float* __restrict__ v, int64_t n,
                                                    AdamStep a, const double* __restrict__ part, int nparts,
                                                    int64_t B, double* __restrict__ loss)
{
    for (int64_t c = blockIdx.x * int64_t(kRowBlock) + threadIdx.x; c < n; c += int64_t(gridDim.x) * kRowBlock)
        adam_update(w, m, v, c, grad[c], a);
    if (blockIdx.x == 0) add_loss(part, nparts, B, loss);
}

// The backward's column reduction with the Adam step fused: per column the
// gradient is the window slices' sum rounded to float (as k_scatter_reduce
// writes it), then the step of k_adam -- one launch fewer a step, the same
// values.  One block per reduce item (the items cover every column once).
__global__ __launch_bounds__(kRowBlock) void k_adam_reduce(const ReduceWork* __restrict__ work,
                                                           const float* __restrict__ gpart, float* __restrict__ w,
                                                           float* __restrict__ m, float* __restrict__ v, AdamStep a,
                                                           const double* __restrict__ part, int nparts, int64_t B,
                                                           double* __restrict__ loss)
{
    const ReduceWork rw = work[blockIdx.x];
    for (int64_t c = rw.col_begin + threadIdx.x; c < rw.col_end; c += kRowBlock)
        adam_update(w, m, v, c, float(reduce_column(gpart, rw, c)), a);
    if (blockIdx.x == 0) add_loss(part, nparts, B, loss);
}

// ------------------------------------------------------------ data ---------
__global__ __launch_bounds__(kRowBlock) void k_random_play(uint64_t seed, int64_t n, int e_lo, int e_hi,
                                                           uint64_t* __restrict__ out)
{
    const int64_t i = blockIdx.x * int64_t(kRowBlock) + threadIdx.x;
    if (i >= n) return;
    const Pos p = random_play(seed, uint64_t(i), e_lo, e_hi);
    out[2 * i] = p.P;
    out[2 * i + 1] = p.O;
}

__global__ void k_targets_x(uint64_t seed, int64_t cols, double sx, double* __restrict__ xt)
{
    for (int64_t c = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; c < cols; c += int64_t(gridDim.x) * blockDim.x) {
        Stream s(seed, uint64_t(c));
        xt[c] = __dmul_rn(sx, s.ih12());
    }
}

}  // namespace
}  // namespace cad
