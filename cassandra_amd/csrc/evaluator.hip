// The expanded-table evaluator on the device: expansion of compact weights
// into one table of 3^n floats per variation (ScoreEstimator's constructor,
// Pattern/Evaluator.cpp:11-29), compaction back (ScoreEstimator::Weights,
// Pattern/Evaluator.cpp:56-73), and a resident evaluator that keeps its
// weights in HBM and scores batches of positions (ScoreEstimator::Eval,
// Pattern/Evaluator.cpp:48-54, for the leaves of a search).
#include "evaluator.hpp"

#include <algorithm>
#include <cstring>

#include "kernels.hpp"

namespace cad {

namespace {

// w_i[t] = x[column of variation i for the configuration whose FastIndex over
// the variation's mask is t]: t's base-3 digits (least significant first) are
// the squares of the mask in ascending order, digit 1 = P, 2 = O.  One thread
// per table entry; blockIdx.y is the slot.
__global__ __launch_bounds__(256) void k_expand_tables(const EvalSlot* __restrict__ es,
                                                       const DevSlot* __restrict__ slots,
                                                       const uint8_t* __restrict__ sq,
                                                       const uint32_t* __restrict__ dense,
                                                       const float* __restrict__ w, float* __restrict__ tables)
{
    const EvalSlot s = es[blockIdx.y];
    const DevSlot sl = slots[blockIdx.y];
    const uint32_t n3 = s.n3;
    for (uint32_t t = blockIdx.x * 256u + threadIdx.x; t < n3; t += gridDim.x * 256u) {
        uint64_t P = 0, O = 0;
        uint32_t rest = t;
        for (int j = 0; j < int(s.n); j++) {
            const uint32_t d = rest % 3u;
            rest /= 3u;
            const uint64_t bit = uint64_t(1) << s.sq[j];
            if (d == 1u) P |= bit;
            else if (d == 2u) O |= bit;
        }
        tables[s.table_offset + t] = w[sl.col_offset + slot_index(sl, sq, dense, P, O)];
    }
}

// Compaction, pass 1: for every configuration (p, o) of a pattern's mask
// (p & o == 0 over the mask's n bits, enumerated p outer, o inner as
// Configurations does, Pattern/Helpers.cpp:81-102), the key p * 2^n + o + 1
// orders the configurations as the enumeration does; each compact column
// keeps the largest key of the configurations whose index it is (the last
// one the reference writes).  blockIdx.y is the pattern.
__device__ __forceinline__ void config_position(const EvalSlot& s, uint32_t pb, uint32_t ob, uint64_t& P,
                                                uint64_t& O)
{
    P = O = 0;
    for (int j = 0; j < int(s.n); j++) {
        const uint64_t bit = uint64_t(1) << s.sq[j];
        if ((pb >> j) & 1u) P |= bit;
        if ((ob >> j) & 1u) O |= bit;
    }
}

__global__ __launch_bounds__(256) void k_compact_keys(const EvalSlot* __restrict__ es,
                                                      const int32_t* __restrict__ first_slot,
                                                      const DevSlot* __restrict__ slots,
                                                      const uint8_t* __restrict__ sq,
                                                      const uint32_t* __restrict__ dense, uint32_t* __restrict__ key)
{
    const int s0 = first_slot[blockIdx.y];
    const EvalSlot s = es[s0];
    const DevSlot sl = slots[s0];
    const uint32_t n = s.n, nn = 1u << (2 * n);
    for (uint32_t c = blockIdx.x * 256u + threadIdx.x; c < nn; c += gridDim.x * 256u) {
        const uint32_t pb = c >> n, ob = c & ((1u << n) - 1u);
        if (pb & ob) continue;
        uint64_t P, O;
        config_position(s, pb, ob, P, O);
        atomicMax(&key[sl.col_offset + slot_index(sl, sq, dense, P, O)], c + 1u);
    }
}

// Compaction, pass 2: the configuration holding a column's key writes
// w[column] = table 0 of the pattern at its FastIndex.
__global__ __launch_bounds__(256) void k_compact_write(const EvalSlot* __restrict__ es,
                                                       const int32_t* __restrict__ first_slot,
                                                       const DevSlot* __restrict__ slots,
                                                       const uint8_t* __restrict__ sq,
                                                       const uint32_t* __restrict__ dense,
                                                       const uint32_t* __restrict__ key,
                                                       const float* __restrict__ tables, float* __restrict__ w)
{
    const int s0 = first_slot[blockIdx.y];
    const EvalSlot s = es[s0];
    const DevSlot sl = slots[s0];
    const uint32_t n = s.n, nn = 1u << (2 * n);
    for (uint32_t c = blockIdx.x * 256u + threadIdx.x; c < nn; c += gridDim.x * 256u) {
        const uint32_t pb = c >> n, ob = c & ((1u << n) - 1u);
        if (pb & ob) continue;
        uint64_t P, O;
        config_position(s, pb, ob, P, O);
        const uint32_t col = sl.col_offset + slot_index(sl, sq, dense, P, O);
        if (key[col] != c + 1u) continue;
        uint32_t t = 0;
        for (int j = int(n) - 1; j >= 0; --j) t = t * 3u + ((pb >> j) & 1u) + 2u * ((ob >> j) & 1u);
        w[col] = tables[s.table_offset + t];
    }
}

// Eval for every position: the sum over the variations of table_i[FastIndex(
// pos, mask_i)], in variation order from 0.0f (bit-identical to
// ScoreEstimator::Eval and to (A x)[row]).  The evaluator keeps the compact
// weights, not the expanded tables: every variation of a pattern reads the
// same columns, which an index tile computes for 64 positions and four
// variations with four matrix instructions; 52 slots of 12 patterns read 0.7 MB
// where their tables are 5.4 MB.
constexpr int kEvalBlock = 1024;

// Small batches: a block takes 64 positions, a wave of it one index tile, and
// the values meet in LDS, where wave 0 adds them in slot order (0.0f for the
// slots a tile does not have: no partial sum is -0.0f).  Walking the slots in
// one thread took a dependent chain of descriptor, program and table loads per
// slot: 64 positions x 52 slots 35 µs against 3.7 here, 65,536 43 against 11.4 (4
// patterns, 18 slots: 15.9 and 6.1).  Bound by latency, and above 30,000
// positions by the columns' lines in L1.  (The times of this kernel and the next
// are launches back to back.)
__global__ __launch_bounds__(kEvalBlock) void k_eval_block(const uint64_t* __restrict__ pos, int64_t n, TileView tv,
                                                           const float* __restrict__ w, uint32_t cols,
                                                           float* __restrict__ out)
{
    __shared__ uint32_t words[64 * 4];
    __shared__ float vals[kEvalBlock / 64][4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = int(blockDim.x) >> 6;
    const int64_t base = blockIdx.x * int64_t(64);
    TileRegs next = load_tile(tv, min(wave, tv.n - 1));
    if (wave == 0) {
        const int64_t r = min(base + lane, n - 1);
        uint32_t T[4];
        ternary_words(pos[2 * r], pos[2 * r + 1], T);
#pragma unroll
        for (int i = 0; i < 4; i++) words[4 * lane + i] = T[i];
    }
    __syncthreads();
    Int4 b[4];
#pragma unroll
    for (int p = 0; p < 4; p++) b[p] = expand_digits(words[4 * (16 * p + (lane & 15)) + (lane >> 4)]);
    float sum = 0.0f;
    for (int t0 = 0; t0 < tv.n; t0 += nw) {
        const int t = t0 + wave;
        if (t < tv.n) {
            const TileRegs cur = next;
            const IndexTile tl = cur.tile();
            next = load_tile(tv, min(t + nw, tv.n - 1));
            uint32_t ci[4];
            tile_columns(tl, t, tv, cur.weights, b, ci);
            transpose_groups(ci);
            float x[4];
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = w[min(tl.col_offset + ci[j], cols - 1)];
#pragma unroll
            for (int j = 0; j < 4; j++) vals[wave][j][lane] = j < tl.nslots ? x[j] : 0.0f;
        }
        __syncthreads();
        if (wave == 0) {
            const int m = min(nw, tv.n - t0);
            for (int i = 0; i < m; i++) {
#pragma unroll
                for (int j = 0; j < 4; j++) sum += vals[i][j][lane];
            }
        }
        if (t0 + nw < tv.n) __syncthreads();
    }
    if (wave == 0 && base + lane < n) out[base + lane] = sum;
}

// Large batches: one block a CU keeps the weights of the patterns with the
// most variations a column in LDS (EvalPlan) and its waves walk the positions,
// 64 C at a time; the other patterns' weights come through L1, where a wave's
// load of 64 columns takes as many lines, which bounds the kernel.
// 1M positions of 12 patterns (52 slots, 32 of them in LDS): 55 µs, 81 from the
// expanded tables, 134 in the block kernel; of 4 patterns 38, 40 and 53.  Two
// runs of positions a wave share a tile's weights and hide each other's latency
// (1M: 60 µs with one); where one run a wave covers the batch, one is faster
// (262,144: 20 against 26).  (Staging every pattern in phases, as
// k_gather_tile_mf does, was not tried.)
template <int C>
__global__ __launch_bounds__(kEvalBlock) void k_eval_staged(const uint64_t* __restrict__ pos, int64_t n, TileView tv,
                                                            const int32_t* __restrict__ tile_lds,
                                                            const PhaseSeg* __restrict__ segs, int nsegs,
                                                            const float* __restrict__ w, uint32_t cols,
                                                            float* __restrict__ out)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float* xs = reinterpret_cast<float*>(smem_raw);
    for (int s = 0; s < nsegs; s++) {
        const PhaseSeg ps = uniform_load(segs + s);
        stage_direct<float, kEvalBlock>(xs + ps.lds_off, w + ps.col_lo, ps.width);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t step = int64_t(gridDim.x) * (kEvalBlock * C);
    for (int64_t base = (blockIdx.x * int64_t(kEvalBlock / 64) + wave) * (64 * C); base < n; base += step) {
        Int4 b[C][4];
        float sum[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            sum[c] = 0.0f;
            digits_of_rows(pos, min(base + 64 * c + lane, n - 1), b[c]);
        }
        TileRegs next = load_tile(tv, 0);
        int next_lds = tile_lds[0];
        for (int t = 0; t < tv.n; t++) {
            const TileRegs cur = next;
            const IndexTile tl = cur.tile();
            const int at = __builtin_amdgcn_readfirstlane(next_lds);
            const int nt = min(t + 1, tv.n - 1);
            next = load_tile(tv, nt);
            next_lds = tile_lds[nt];
            float x[C][4];
#pragma unroll
            for (int c = 0; c < C; c++) {
                uint32_t ci[4];
                tile_columns(tl, t, tv, cur.weights, b[c], ci);
                transpose_groups(ci);
                if (at >= 0) {
#pragma unroll
                    for (int j = 0; j < 4; j++) x[c][j] = xs[uint32_t(at) + ci[j]];
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++) x[c][j] = w[min(tl.col_offset + ci[j], cols - 1)];
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (j < tl.nslots) {
#pragma unroll
                    for (int c = 0; c < C; c++) sum[c] += x[c][j];
                }
        }
#pragma unroll
        for (int c = 0; c < C; c++)
            if (base + 64 * c + lane < n) out[base + 64 * c + lane] = sum[c];
    }
}

int blocks_for(uint64_t n, int cap = 4096)
{
    return int(std::max<uint64_t>(1, std::min<uint64_t>((n + 255) / 256, uint64_t(cap))));
}

}  // namespace

// Positions a CU from which a batch is scored from LDS: the staging comes before
// the first position, and a pass of the staged block is long (131,072 positions
// on 256 CUs, block / staged: 18 slots 10.0 / 10.0 µs, 46 slots 15.1 / 15.0, 52
// slots 20.6 / 16.8, 54 slots 21.1 / 18.3; half as many 6.1 / 9.8, 8.4 / 14.7,
// 11.4 / 16.5, 12.0 / 17.9; twice as many 16.8 / 12.6, 27.0 / 15.9, 38.2 / 20.0,
// 37.7 / 21.2).  Sets of which nothing fits stay with the block kernel: 4M
// positions of three patterns of 11 and 12 squares (24 slots) 381 µs, from the
// expanded tables 413; of a single one of 10 squares (8 slots) 86 and 82.
constexpr int64_t kEvalStagedRows = 512;
// Most positions of one launch of the block kernel.
constexpr int64_t kEvalBlockRows = int64_t(1) << 26;

// Per-slot table layout of a pattern group (variation after variation, in
// slot order), uploaded once per pattern group.
const ExpandedLayout& expanded_layout(cad_patterns* p)
{
    if (p->layout) return *p->layout;
    std::unique_ptr<ExpandedLayout> L(new ExpandedLayout);
    const PatternGroup& g = *p->group;
    std::vector<EvalSlot> es;
    int slot = 0;
    uint64_t off = 0;
    for (const PatternInfo& pi : g.patterns) {
        L->first_slot.push_back(slot);
        for (uint64_t v : pi.variations) {
            EvalSlot e;
            std::memset(&e, 0, sizeof(e));
            int j = 0;
            for (int q = 0; q < 64; q++)
                if ((v >> q) & 1) e.sq[j++] = uint8_t(q);
            if (j > 16) throw Error(CAD_ERR_PATTERN, "expanded tables need patterns of at most 16 squares");
            e.n = uint8_t(j);
            e.n3 = pow3(j);
            e.table_offset = off;
            off += e.n3;
            es.push_back(e);
            slot++;
        }
    }
    if (slot != g.k()) throw Error(CAD_ERR_PATTERN, "variation count differs from the slot count");
    L->slots = es;
    L->size = int64_t(off);
    hipStream_t s = p->ctx->stream;
    L->d_slots = to_device(es, s);
    L->d_first_slot = to_device(L->first_slot, s);
    CAD_HIP(hipStreamSynchronize(s));  // the host vectors are uploaded
    p->layout = std::move(L);
    return *p->layout;
}

void weights_expand(cad_patterns* p, const float* w, float* tables)
{
    const ExpandedLayout& L = expanded_layout(p);
    uint32_t widest = 1;
    for (const EvalSlot& e : L.slots) widest = std::max(widest, e.n3);
    hipLaunchKernelGGL(k_expand_tables, dim3(unsigned(blocks_for(widest)), unsigned(L.slots.size())), dim3(256), 0,
                       p->ctx->stream, L.d_slots.as<EvalSlot>(), p->d_slots.as<DevSlot>(), p->d_sq.as<uint8_t>(),
                       p->d_dense.as<uint32_t>(), w, tables);
    CAD_HIP(hipGetLastError());
}

void weights_compact(cad_patterns* p, const float* tables, float* w)
{
    const ExpandedLayout& L = expanded_layout(p);
    const int64_t cols = int64_t(p->group->cols());
    hipStream_t s = p->ctx->stream;
    DBuf key(sizeof(uint32_t) * size_t(std::max<int64_t>(1, cols)));
    hipLaunchKernelGGL(k_fill<uint32_t>, dim3(unsigned(blocks_for(uint64_t(cols)))), dim3(256), 0, s,
                       key.as<uint32_t>(), cols, 0u);
    hipLaunchKernelGGL(k_fill<float>, dim3(unsigned(blocks_for(uint64_t(cols)))), dim3(256), 0, s, w, cols, 0.0f);
    uint32_t widest = 1;
    for (int f : L.first_slot) widest = std::max(widest, 1u << (2 * L.slots[size_t(f)].n));
    const dim3 grid(unsigned(blocks_for(widest)), unsigned(L.first_slot.size()));
    hipLaunchKernelGGL(k_compact_keys, grid, dim3(256), 0, s, L.d_slots.as<EvalSlot>(), L.d_first_slot.as<int32_t>(),
                       p->d_slots.as<DevSlot>(), p->d_sq.as<uint8_t>(), p->d_dense.as<uint32_t>(),
                       key.as<uint32_t>());
    hipLaunchKernelGGL(k_compact_write, grid, dim3(256), 0, s, L.d_slots.as<EvalSlot>(), L.d_first_slot.as<int32_t>(),
                       p->d_slots.as<DevSlot>(), p->d_sq.as<uint8_t>(), p->d_dense.as<uint32_t>(),
                       (const uint32_t*)key.as<uint32_t>(), tables, w);
    CAD_HIP(hipGetLastError());
    CAD_HIP(hipStreamSynchronize(s));  // the key buffer is freed on return
}

const EvalPlan& eval_weights_plan(cad_patterns* p)
{
    if (p->eval_plan) return *p->eval_plan;
    std::unique_ptr<EvalPlan> E(new EvalPlan);
    const PatternGroup& g = *p->group;
    // the patterns with the fewest columns a variation first
    std::vector<size_t> order(g.patterns.size());
    for (size_t i = 0; i < order.size(); i++) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) {
        const PatternInfo &x = g.patterns[a], &y = g.patterns[b];
        return uint64_t(x.size) * y.variations.size() < uint64_t(y.size) * x.variations.size();
    });
    const uint64_t room = std::min<size_t>(p->ctx->max_lds, 160 * 1024) / sizeof(float);
    std::vector<PhaseSeg> segs;
    std::vector<int32_t> pattern_lds(g.patterns.size(), -1), tile_lds(size_t(std::max(1, p->ntiles)), -1);
    uint64_t used = 0;
    for (size_t i : order) {
        // a segment keeps its columns' places within a 16-byte line
        const PatternInfo& pi = g.patterns[i];
        const uint32_t head = pi.offset & 3u;
        const uint64_t need = (uint64_t(head) + pi.size + 3) & ~uint64_t(3);
        if (used + need > room) continue;
        segs.push_back(PhaseSeg{pi.offset, pi.size, uint32_t(used), 0});
        pattern_lds[i] = int32_t(used + head);
        used += need;
    }
    int slot = 0;
    for (size_t i = 0; i < g.patterns.size(); i++)
        for (size_t v = 0; v < g.patterns[i].variations.size(); v++)
            tile_lds[p->slot_tile[size_t(slot++)]] = pattern_lds[i];
    if (slot != g.k()) throw Error(CAD_ERR_PATTERN, "variation count differs from the slot count");
    E->nsegs = int(segs.size());
    E->lds = size_t(used) * sizeof(float);
    // the kernels' LDS limit is set here, so that a launch is all a batch needs
    // (also while a stream is captured); the same limit for every pattern group
    for (auto kern : {k_eval_staged<1>, k_eval_staged<2>})
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  int(room * sizeof(float)));
    hipStream_t s = p->ctx->stream;
    E->d_segs = to_device(segs, s);
    E->d_tile_lds = to_device(tile_lds, s);
    CAD_HIP(hipStreamSynchronize(s));  // the host vectors are uploaded
    p->eval_plan = std::move(E);
    return *p->eval_plan;
}

void eval_weights(cad_patterns* p, const float* w, const uint64_t* pos, int64_t n, float* out)
{
    if (n <= 0) return;
    const EvalPlan& E = eval_weights_plan(p);
    const TileView tv = p->tiles();
    const uint32_t cols = uint32_t(p->group->cols());
    hipStream_t s = p->ctx->stream;
    if (tv.n == 0) {
        hipLaunchKernelGGL(k_fill<float>, dim3(unsigned(blocks_for(uint64_t(n)))), dim3(256), 0, s, out, n, 0.0f);
    } else if (E.nsegs > 0 && n >= kEvalStagedRows * p->ctx->cus) {
        const int C = n <= int64_t(p->ctx->cus) * kEvalBlock ? 1 : 2;
        auto kern = C == 1 ? k_eval_staged<1> : k_eval_staged<2>;
        const int64_t blocks = std::min<int64_t>(p->ctx->cus, (n + kEvalBlock * C - 1) / (kEvalBlock * C));
        hipLaunchKernelGGL(kern, dim3(unsigned(blocks)), dim3(kEvalBlock), E.lds, s, pos, n, tv,
                           E.d_tile_lds.as<int32_t>(), E.d_segs.as<PhaseSeg>(), E.nsegs, w, cols, out);
    } else {
        const int waves = std::min(kEvalBlock / 64, tv.n);
        // (a launch holds fewer than 2^32 threads: 2^28 positions of 16 waves)
        for (int64_t a = 0; a < n; a += kEvalBlockRows) {
            const int64_t m = std::min(kEvalBlockRows, n - a);
            hipLaunchKernelGGL(k_eval_block, dim3(unsigned((m + 63) / 64)), dim3(unsigned(64 * waves)), 0, s,
                               pos + 2 * a, m, tv, w, cols, out + a);
        }
    }
    CAD_HIP(hipGetLastError());
}

}  // namespace cad

void cad_evaluator::pin(int64_t n)
{
    if (n <= pinned) return;
    CAD_HIP(hipStreamSynchronize(ctx->stream));
    const int64_t m = std::max(n, 2 * pinned);  // (a search's batches grow in small steps)
    uint64_t* a = nullptr;
    float* b = nullptr;
    CAD_HIP(hipHostMalloc(reinterpret_cast<void**>(&a), sizeof(uint64_t) * 2 * size_t(m), hipHostMallocDefault));
    const hipError_t rc = hipHostMalloc(reinterpret_cast<void**>(&b), sizeof(float) * size_t(m), hipHostMallocDefault);
    if (rc != hipSuccess) (void)hipHostFree(a);
    CAD_HIP(rc);
    if (h_pos) (void)hipHostFree(h_pos);
    if (h_out) (void)hipHostFree(h_out);
    h_pos = a;
    h_out = b;
    pinned = m;
}

cad_evaluator::~cad_evaluator()
{
    if (h_pos) (void)hipHostFree(h_pos);
    if (h_out) (void)hipHostFree(h_out);
}
