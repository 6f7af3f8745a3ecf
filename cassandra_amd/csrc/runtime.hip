// Device buffers, contexts, pattern groups, matrices and their launch plans.
#include "runtime.hpp"

#include "../../include/cassandra_amd.h"

#include <algorithm>
#include <cstring>
#include <numeric>

#include "kernels.hpp"

namespace cad {

void hip_check(hipError_t e, const char* what)
{
    if (e != hipSuccess) {
        if (e == hipErrorOutOfMemory) throw Error(-5, std::string("out of device memory: ") + what);
        throw Error(-4, std::string(hipGetErrorString(e)) + " in " + what);
    }
}

DBuf::DBuf(size_t n) : bytes(n)
{
    if (n) {
        hipError_t e = hipMalloc(&p, n);
        if (e != hipSuccess) {
            p = nullptr;
            (void)hipGetLastError();
            throw Error(-5, "hipMalloc of " + std::to_string(n) + " bytes failed");
        }
    }
}

DBuf::DBuf(std::shared_ptr<DBuf> whole, size_t at, size_t n)
    : p(static_cast<uint8_t*>(whole->p) + at), bytes(n), part(std::move(whole))
{
}

DBuf::~DBuf()
{
    if (p && !part) (void)hipFree(p);
}

DBuf& DBuf::operator=(DBuf&& o) noexcept
{
    if (this != &o) {
        if (p && !part) (void)hipFree(p);
        p = o.p;
        bytes = o.bytes;
        part = std::move(o.part);
        o.p = nullptr;
        o.bytes = 0;
    }
    return *this;
}

void DBuf::upload(const void* h, size_t n, hipStream_t s)
{
    CAD_HIP(hipMemcpyAsync(p, h, n, hipMemcpyHostToDevice, s));
    CAD_HIP(hipStreamSynchronize(s));
}

namespace {
constexpr size_t kPieceAlign = 256;
size_t piece(size_t n) { return (n + kPieceAlign - 1) / kPieceAlign * kPieceAlign; }
}  // namespace

void Uploads::put_bytes(DBuf& dst, const void* src, size_t bytes, size_t least)
{
    const size_t at = piece(host.size());
    host.resize(at + std::max(bytes, least), 0);
    if (bytes) std::memcpy(host.data() + at, src, bytes);
    items.push_back(Item{&dst, at, std::max(bytes, least), true});
}

void Uploads::reserve(DBuf& dst, size_t bytes)
{
    items.push_back(Item{&dst, reserved, bytes, false});
    reserved += piece(bytes);
}

void Uploads::flush(hipStream_t s)
{
    if (items.empty()) return;
    const size_t copied = piece(host.size());
    auto whole = std::make_shared<DBuf>(std::max<size_t>(1, copied + reserved));
    if (!host.empty()) whole->upload(host.data(), host.size(), s);
    for (const Item& i : items) *i.dst = DBuf(whole, i.copied ? i.at : copied + i.at, i.bytes);
    items.clear();
    host.clear();
    reserved = 0;
}

Context::~Context()
{
    if (own) (void)hipStreamDestroy(own);
}

GridSys GridPlan::row_sys() const
{
    return GridSys{d_row_first.as<int32_t>(), d_row_count.as<int32_t>(), d_row_counters.as<unsigned>(),
                   d_partials.as<double>()};
}

GridSys GridPlan::col_sys() const
{
    return GridSys{d_col_first.as<int32_t>(), d_col_count.as<int32_t>(), d_col_counters.as<unsigned>(),
                   d_partials.as<double>()};
}

namespace {

constexpr uint32_t kReduceCols = kRowBlock;  // columns of one scatter-reduce work item

// Row chunks of one window of a system: the share of the target tile count,
// capped so that the partial slices stay near partial_cap of the window's
// index traffic -- and, where that cap would leave CUs idle, raised towards
// one tile per CU while its slices stay under the floor bytes a window
// (their write and read then cost less than the parallelism gains):
// small_floor (8 MB by default) for a small system (at most kRowKernelRows
// rows, whose tiles are latency-bound: a 100k-row PCG iteration 47 -> 42 µs),
// 2 MB for a large one (8 MB took the 5M-row matrix's XCD-major plan from 240
// to 360 tiles, 165 -> 245 µs).
// `windows` counts the windows of every system planned together: those of
// many systems already fill the CUs side by side.  At least kScatterBlock
// rows a chunk.
constexpr double kPartialFloorBytes = 2.0 * 1024 * 1024;
constexpr double kMultiSystemTiles = 8.0;  // target tiles a CU, over blocks_per_cu, for several systems

int64_t window_chunks(int64_t R, double share_chunks, double cap_chunks, int cus, int windows, uint32_t W,
                      int vbytes, double small_floor)
{
    int64_t C = std::max<int64_t>(1, std::min<int64_t>(std::llround(share_chunks), int64_t(cap_chunks)));
    const int64_t par = std::max<int64_t>(1, cus / std::max(1, windows));
    const double floor_bytes = R <= kRowKernelRows ? small_floor : kPartialFloorBytes;
    const int64_t floor_c = std::max<int64_t>(1, int64_t(floor_bytes / (2.0 * double(W) * vbytes)));
    C = std::max(C, std::min(par, floor_c));
    return std::max<int64_t>(1, std::min<int64_t>(C, (R + kScatterBlock - 1) / kScatterBlock));
}

// Slots of fewer columns than this take longer the fewer they are (win_cost).
constexpr double kNarrowSlot = 1024;

// Group slots whose column ranges overlap (transitively).
void make_groups(const std::vector<uint32_t>& lo, const std::vector<uint32_t>& hi, ScatterPlan& sp)
{
    const int k = int(lo.size());
    std::vector<int> order(k);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return lo[a] < lo[b]; });
    sp.groups.clear();
    sp.slot_list.clear();
    sp.narrow.assign(size_t(k), 0.0);
    int i = 0;
    while (i < k) {
        uint32_t glo = lo[order[i]], ghi = hi[order[i]];
        int j = i + 1;
        while (j < k && lo[order[j]] < ghi) {
            ghi = std::max(ghi, hi[order[j]]);
            j++;
        }
        std::vector<uint16_t> members;
        for (int t = i; t < j; t++) {
            members.push_back(uint16_t(order[t]));
            const uint32_t width = std::max<uint32_t>(1, hi[order[t]] - lo[order[t]]);
            sp.narrow[size_t(order[t])] = std::max(0.0, std::log2(kNarrowSlot / width));
        }
        std::sort(members.begin(), members.end());  // keep slot order inside a group
        SlotGroup g;
        g.col_lo = glo;
        g.col_hi = ghi;
        g.nslots = uint16_t(members.size());
        g.first = uint16_t(sp.slot_list.size());
        sp.slot_list.insert(sp.slot_list.end(), members.begin(), members.end());
        sp.groups.push_back(g);
        i = j;
    }
}

// The scatter groups of a window size (ScatterLists::groups).  Pattern
// groups come in column order and never overlap.
void pack_groups(const ScatterPlan& sp, uint32_t wmax, int max_slots, ScatterLists& L)
{
    L.groups.clear();
    L.slot_list.clear();
    size_t i = 0;
    while (i < sp.groups.size()) {
        SlotGroup g = sp.groups[i];
        std::vector<uint16_t> slots(sp.slot_list.begin() + g.first, sp.slot_list.begin() + g.first + g.nslots);
        size_t j = i + 1;
        if (g.col_hi - g.col_lo <= wmax)
            for (; j < sp.groups.size(); j++) {
                const SlotGroup& h = sp.groups[j];
                if (h.col_lo < g.col_hi || h.col_hi - g.col_lo > wmax || g.nslots + h.nslots > max_slots) break;
                slots.insert(slots.end(), sp.slot_list.begin() + h.first, sp.slot_list.begin() + h.first + h.nslots);
                g.col_hi = h.col_hi;
                g.nslots = uint16_t(g.nslots + h.nslots);
            }
        g.first = uint16_t(L.slot_list.size());
        L.slot_list.insert(L.slot_list.end(), slots.begin(), slots.end());
        L.groups.push_back(g);
        i = j;
    }
}

// Reduce items of one window ([wl, wh) of system s, chunk slices at off with
// stride W) and of the columns outside every window (written as zeros).
void push_reduce(ScatterLists& L, int s, uint32_t sys_col, uint32_t wl, uint32_t wh, int64_t off, int64_t C)
{
    // one column per thread of a reduce block (kReduceCols), so the reduce
    // launches enough blocks to cover the CUs
    for (uint32_t c0 = wl; c0 < wh; c0 += kReduceCols) {
        ReduceWork r;
        r.col_begin = int64_t(sys_col) + c0;
        r.col_end = int64_t(sys_col) + std::min(wh, c0 + kReduceCols);
        r.part_off = C > 0 ? off + (c0 - wl) : 0;
        r.nchunk = int32_t(C);
        r.stride = C > 0 ? wh - wl : 0;
        r.sys = s;
        r.pad = 0;
        L.reduce.push_back(r);
    }
}

// Chunk-major scatter lists: every window of a system uses the same row
// chunks, and the tiles of one chunk (all its windows, the heavier ones split
// into row parts of equal work) are placed on one XCD one after the other
// (workgroup i runs on XCD i mod 8), so the y values and the index entries
// that the windows of a chunk share are read from HBM once and then hit that
// XCD's L2.  The chunk count is a multiple of the XCD count near the target
// tile count.  Slots left over at the end of an XCD's lane hold empty tiles
// (no rows, no columns).
constexpr int kXcds = 8;

void make_scatter_lists_xcd(const ScatterPlan& sp, const std::vector<int64_t>& sys_rows,
                            const std::vector<uint32_t>& sys_col, int64_t cols_per_sys, uint32_t wmax, int vbytes,
                            int ibytes, double target, int cus, const TuneParams& tune, ScatterLists& L,
                            const std::vector<uint8_t>* on)
{
    (void)sp;
    const int nsys = int(sys_col.size());
    auto in = [&](int s) { return !on || (*on)[size_t(s)] != 0; };
    // Windows of the slot groups; a window with more slots than the lightest
    // is split into parts (row sub-ranges of the chunk), so that every tile
    // of a chunk does about the same work and the chunk's tiles, running
    // side by side on one XCD, stream its rows at the same pace.
    struct Win { uint32_t lo, hi; int group; int nslots; int parts; };
    std::vector<Win> wins;
    double work_per_row = 0, width = 0;
    int minslots = 1 << 30;
    for (size_t gi = 0; gi < L.groups.size(); gi++) {
        const SlotGroup& g = L.groups[gi];
        for (uint32_t wl = g.col_lo; wl < g.col_hi; wl += wmax) {
            const uint32_t wh = std::min(g.col_hi, wl + wmax);
            wins.push_back(Win{wl, wh, int(gi), g.nslots, 1});
            L.widest = std::max(L.widest, wh - wl);
            work_per_row += g.nslots;
            width += wh - wl;
            minslots = std::min(minslots, int(g.nslots));
        }
    }
    const int nw = int(wins.size());
    int tiles_per_chunk = 0;
    for (Win& w : wins) {
        w.parts = std::max(1, int(std::lround(double(w.nslots) / std::max(1, minslots))));
        tiles_per_chunk += w.parts;
    }
    int64_t total_rows = 0;
    int nrun = 0;  // systems planned here that have rows: their windows run side by side
    for (int s = 0; s < nsys; s++)
        if (in(s)) {
            total_rows += sys_rows[s + 1] - sys_rows[s];
            nrun += sys_rows[s + 1] > sys_rows[s];
        }
    // chunks: about target tiles in all, a multiple of the XCD count
    int64_t chunks = std::max<int64_t>(1, std::llround(target / std::max(1, tiles_per_chunk)));
    if (chunks > kXcds) chunks = chunks / kXcds * kXcds;
    std::vector<std::vector<ScatterWork>> lanes(kXcds);
    int64_t off = 0;
    int chunk_id = 0;
    for (int s = 0; s < nsys; s++) {
        if (!in(s)) continue;
        const int64_t R = sys_rows[s + 1] - sys_rows[s];
        int64_t C = 0;
        std::vector<int64_t> woff(size_t(std::max(1, nw)));
        if (R > 0 && nw > 0) {
            const double share = total_rows > 0 ? double(R) / double(total_rows) : 1.0;
            const double cap = tune.partial_cap * double(R) * work_per_row * ibytes /
                               (2.0 * width * vbytes * double(tiles_per_chunk) / std::max(1, nw));
            C = window_chunks(R, double(chunks) * share, cap, cus, tiles_per_chunk * std::max(1, nrun),
                              uint32_t(width / std::max(1, nw)), vbytes, tune.small_floor_bytes);
            const int64_t chunk = (R + C - 1) / C;
            C = (R + chunk - 1) / chunk;
            for (int j = 0; j < nw; j++) {
                woff[size_t(j)] = off;
                off += C * wins[size_t(j)].parts * int64_t(wins[size_t(j)].hi - wins[size_t(j)].lo);
            }
            for (int64_t c = 0; c < C; c++, chunk_id++) {
                auto& lane = lanes[size_t(chunk_id % kXcds)];
                const int64_t c0 = c * chunk, c1 = std::min(R, (c + 1) * chunk);
                for (int j = 0; j < nw; j++) {
                    const Win& wj = wins[size_t(j)];
                    const int64_t W = int64_t(wj.hi - wj.lo);
                    for (int q = 0; q < wj.parts; q++) {
                        ScatterWork w;
                        w.row_begin = sys_rows[s] + c0 + (c1 - c0) * q / wj.parts;
                        w.row_end = sys_rows[s] + c0 + (c1 - c0) * (q + 1) / wj.parts;
                        w.part_off = woff[size_t(j)] + (c * wj.parts + q) * W;
                        w.win_lo = sys_col[s] + wj.lo;
                        w.win_hi = sys_col[s] + wj.hi;
                        w.group = wj.group;
                        w.sys = s;
                        lane.push_back(w);
                    }
                }
            }
            for (int j = 0; j < nw; j++)
                push_reduce(L, s, sys_col[s], wins[size_t(j)].lo, wins[size_t(j)].hi, woff[size_t(j)],
                            C * wins[size_t(j)].parts);
        }
        // columns outside every window are written as zeros
        std::vector<std::pair<uint32_t, uint32_t>> covered;
        if (R > 0)
            for (const Win& w : wins) covered.push_back({w.lo, w.hi});
        std::sort(covered.begin(), covered.end());
        covered.push_back({uint32_t(cols_per_sys), uint32_t(cols_per_sys)});
        uint32_t at = 0;
        for (auto& iv : covered) {
            if (at < iv.first) push_reduce(L, s, sys_col[s], at, iv.first, 0, 0);
            at = std::max(at, iv.second);
        }
    }
    size_t depth = 0;
    for (auto& lane : lanes) depth = std::max(depth, lane.size());
    ScatterWork empty{};
    empty.row_begin = empty.row_end = 0;
    empty.part_off = 0;
    empty.win_lo = empty.win_hi = 0;
    empty.group = 0;
    empty.sys = 0;
    L.work.assign(depth * kXcds, empty);
    for (int x = 0; x < kXcds; x++)
        for (size_t p = 0; p < lanes[size_t(x)].size(); p++) L.work[p * kXcds + size_t(x)] = lanes[size_t(x)][p];
    L.part_elems = off;
}

// Scatter tiles of (system rows) x (group window): every window of a system
// gets row chunks by its time (win_cost), so that the tiles -- about target of
// them -- take equally long; a window's chunks are limited by its partial
// slices (written and read once): partial_cap of its index traffic, or, where
// every window could be cut in two and until there are as many tiles as CUs,
// the floor bytes a window -- small_floor (8 MB by default) for a small system
// (at most kRowKernelRows rows, whose tiles are latency-bound: a 100k-row PCG
// iteration 47 -> 42 µs), 2 MB for a large one -- and to kScatterBlock rows.
// Rounding each window's share by itself, and the floor, made 263 tiles for 256
// CUs at 5M rows of FIT8: seven in a second wave, 197 µs where 256 take 127.
// The floor for a batch whose windows fill the CUs by themselves left mostly
// slices to write and sum: 100 iterations of FP64 PCG over 50 systems 28.9 ms
// against 19.5, the mixed fit of the 50 336 against 317.
void make_scatter_lists(const ScatterPlan& sp, const std::vector<int64_t>& sys_rows,
                        const std::vector<uint32_t>& sys_col, int64_t cols_per_sys, uint32_t wmax, int vbytes,
                        int ibytes, int cus, const TuneParams& tune, bool fp32, ScatterLists& L,
                        const std::vector<uint8_t>* on = nullptr)
{
    L.work.clear();
    L.reduce.clear();
    L.widest = 0;
    pack_groups(sp, wmax, tune.pack_slots, L);
    const int nsys = int(sys_col.size());
    auto in = [&](int s) { return !on || (*on)[size_t(s)] != 0; };
    // Time of a window per row, in units of one slot's loads.  Measured (cycles
    // a tile per 64 rows): FP32 windows take 32 for the row and 7.8 + 2 f a
    // slot, f the window's share of the group's columns (66 to 111 for 4 to 8
    // slots), FP64 ones 18 and 6 + 17.5 f (62 to 206: their adds are slower).  A
    // slot of few columns adds to the same ones over and over: 4 slots of 1,134
    // columns take 74 (FP64 116), 8 of 378 and 1,134 165 (272), 8 of 45 and 135
    // columns 205 (318), where 8 wide ones take 145 (245) of the same rows.
    // Other values of scatter_balance weigh the slot loads (1: loads only)
    // against the entries that fall into the window.  Matrix-free: a slot's
    // columns are computed whether or not they fall into the window
    // (ScatterPlan::slot_cost), after the row's digits (row_cost).
    const double lam = std::min(1.0, std::max(0.0, tune.scatter_balance));
    // the slots' own part of each group (summed once: the sort below asks often)
    std::vector<double> own(L.groups.size(), 0.0);
    for (size_t i = 0; i < L.groups.size(); i++)
        for (int j = 0; j < L.groups[i].nslots; j++) {
            const size_t slot = L.slot_list[size_t(L.groups[i].first + j)];
            own[i] += !sp.slot_cost.empty() ? sp.slot_cost[slot] : tune.weigh_narrow ? sp.narrow[slot] : 0.0;
        }
    auto win_cost = [&](size_t group, uint32_t W) {
        const SlotGroup& g = L.groups[group];
        if (!sp.slot_cost.empty() && vbytes == 8) return sp.row_cost + own[group];
        const double frac = double(W) / double(std::max<uint32_t>(1, g.col_hi - g.col_lo));
        if (lam == 1.0 && vbytes == 8)
            return fp32 ? 4.1 + g.nslots * (1.0 + 0.26 * frac) + 0.32 * own[group]
                        : 3.0 + g.nslots * (1.0 + 2.9 * frac) + 0.45 * own[group];
        return g.nslots * (lam + (1.0 - lam) * frac);
    };
    int nrun = 0;  // systems planned here that have rows: their windows run side by side
    for (int s = 0; s < nsys; s++) nrun += in(s) && sys_rows[s + 1] > sys_rows[s];
    int windows = 0;
    for (auto& g : L.groups) windows += int((g.col_hi - g.col_lo + wmax - 1) / wmax);
    // several systems whose windows outnumber the CUs have tiles of very
    // different sizes (their row counts differ), and systems of an active list
    // (on) stop one after the other: more tiles a CU let the launch balance them
    // (50 systems, about 30 running: 120 µs an iteration in 1,382 tiles, 300 in
    // 256)
    const double share = tune.blocks_per_cu * std::max(cus, 1);
    const bool several = nrun > 1 && (on || double(windows) * nrun > 0.75 * share);
    // one system whose windows are more than half as many as the CUs: in one wave
    // some windows would have one chunk and others two (200,000 rows of 20 slots
    // over 3M columns: 668 µs, 368 in two; 2M rows of five patterns of 12 squares
    // in FP64 1,409 and 818); the lists of 4-byte counts have four waves already
    const bool coarse = nrun == 1 && vbytes == 8 && 2 * windows > cus;
    const double target = share * (several ? kMultiSystemTiles : coarse ? 2.0 : 1.0);
    int64_t off = 0;
    if (tune.scatter_order == 1) {
        make_scatter_lists_xcd(sp, sys_rows, sys_col, cols_per_sys, wmax, vbytes, ibytes, target, cus, tune, L, on);
        return;
    }
    // the windows of every system, and their chunks
    struct Win {
        uint32_t lo, hi;
        int s, group;
        int64_t rows, chunks, cap, most;  // most: the limit while CUs are idle
        double time;
    };
    std::vector<Win> wins;
    double total = 0;
    const double wave = std::max(cus, 1);
    const bool idle = 2.0 * windows * nrun <= wave;  // every window could be cut in two
    for (int s = 0; s < nsys; s++) {
        if (!in(s)) continue;
        const int64_t R = sys_rows[s + 1] - sys_rows[s];
        for (size_t gi = 0; gi < L.groups.size(); gi++) {
            const SlotGroup& g = L.groups[gi];
            for (uint32_t wl = g.col_lo; wl < g.col_hi; wl += wmax) {
                const uint32_t wh = std::min(g.col_hi, wl + wmax), W = wh - wl;
                const double slice = 2.0 * double(W) * vbytes;
                const double cap = tune.partial_cap * double(R) * g.nslots * ibytes / slice;
                const double floor_c = (R <= kRowKernelRows ? tune.small_floor_bytes : kPartialFloorBytes) / slice;
                auto limit = [&](double c) {
                    return std::max<int64_t>(1, std::min<int64_t>(int64_t(c), (R + kScatterBlock - 1) / kScatterBlock));
                };
                Win w{wl, wh, s, int(gi), R, 0, limit(cap), 0, double(R) * win_cost(gi, W)};
                w.most = idle ? std::max(w.cap, limit(floor_c)) : w.cap;
                total += w.time;
                wins.push_back(w);
            }
        }
    }
    // whole shares, then one chunk more wherever the tiles are longest: in one
    // wave until those cannot be cut (more of the shorter ones gain nothing), in
    // several until they are a quarter of those (the Jacobi counts of 500,000
    // rows of 46 slots 33 -> 28 µs, of 100,000 16 -> 13)
    // (shares of what the one tile that every window has leaves of the target:
    // shares of all of it, and a tile for the rest, made more tiles than that)
    const double share0 =
        std::max(0.0, (idle ? std::min(target, wave) : target) - double(windows) * nrun);
    int64_t tiles = 0;
    double stuck = 0;  // the longest tile of a window at its limit
    std::vector<std::pair<double, size_t>> longest;  // a heap by tile time
    for (size_t i = 0; i < wins.size(); i++) {
        Win& w = wins[i];
        if (w.rows <= 0) continue;
        w.chunks = std::max<int64_t>(1, std::min<int64_t>(w.most, int64_t(share0 * w.time / total)));
        tiles += w.chunks;
        longest.push_back({w.time / double(w.chunks), i});
    }
    std::make_heap(longest.begin(), longest.end());
    while (tiles < int64_t(target) && !longest.empty()) {
        std::pop_heap(longest.begin(), longest.end());
        const double time = longest.back().first;
        Win& w = wins[longest.back().second];
        longest.pop_back();
        if (time <= (target <= wave ? stuck : 0.25 * stuck)) break;
        if (w.chunks >= (double(tiles) < wave ? w.most : w.cap)) {
            stuck = std::max(stuck, time);
            continue;
        }
        w.chunks++;
        tiles++;
        longest.push_back({w.time / double(w.chunks), size_t(&w - wins.data())});
        std::push_heap(longest.begin(), longest.end());
    }
    size_t at = 0;
    for (int s = 0; s < nsys; s++) {
        if (!in(s)) continue;
        std::vector<std::pair<uint32_t, uint32_t>> covered;
        for (; at < wins.size() && wins[at].s == s; at++) {
            const Win& wn = wins[at];
            const uint32_t W = wn.hi - wn.lo;
            covered.push_back({wn.lo, wn.hi});
            L.widest = std::max(L.widest, W);
            int64_t C = 0;
            if (wn.rows > 0) {
                const int64_t chunk = (wn.rows + wn.chunks - 1) / wn.chunks;
                C = (wn.rows + chunk - 1) / chunk;
                for (int64_t c = 0; c < C; c++) {
                    ScatterWork w;
                    w.row_begin = sys_rows[s] + c * chunk;
                    w.row_end = sys_rows[s] + std::min(wn.rows, (c + 1) * chunk);
                    w.part_off = off + c * int64_t(W);
                    w.win_lo = sys_col[s] + wn.lo;
                    w.win_hi = sys_col[s] + wn.hi;
                    w.group = int32_t(wn.group);
                    w.sys = s;
                    L.work.push_back(w);
                }
            }
            push_reduce(L, s, sys_col[s], wn.lo, wn.hi, off, C);
            off += C * int64_t(W);
        }
        // columns outside every window are written as zeros
        std::sort(covered.begin(), covered.end());
        covered.push_back({uint32_t(cols_per_sys), uint32_t(cols_per_sys)});
        uint32_t next = 0;
        for (auto& iv : covered) {
            if (next < iv.first) push_reduce(L, s, sys_col[s], next, iv.first, 0, 0);
            next = std::max(next, iv.second);
        }
    }
    L.part_elems = off;
    // longest first: a launch of more tiles than CUs then starts its big
    // chunks in the first wave and fills in with the small ones (each tile
    // writes its own slice, so the order changes no sum)
    std::vector<std::pair<double, size_t>> order;
    order.reserve(L.work.size());
    for (size_t i = 0; i < L.work.size(); i++) {
        const ScatterWork& w = L.work[i];
        order.push_back({-double(w.row_end - w.row_begin) * win_cost(size_t(w.group), w.win_hi - w.win_lo), i});
    }
    std::sort(order.begin(), order.end());
    std::vector<ScatterWork> sorted;
    sorted.reserve(order.size());
    for (const auto& o : order) sorted.push_back(L.work[o.second]);
    L.work = std::move(sorted);
}

// The host side of a list after planning: the bound on the terms a window
// column receives in one work item (rows x slots of the group), for the
// fixed-point scale of the FP32 scatter, and the reduce items ordered by
// system with each system's range of them.
void finish_lists(ScatterLists& L, int nsys)
{
    L.cbits = 0;
    for (const ScatterWork& w : L.work) {
        uint64_t n = uint64_t(std::max<int64_t>(0, w.row_end - w.row_begin)) * L.groups[size_t(w.group)].nslots;
        int b = 0;
        while (n) b++, n >>= 1;
        L.cbits = std::max(L.cbits, b);
    }
    const auto by_system = [](const ReduceWork& a, const ReduceWork& b) { return a.sys < b.sys; };
    if (!std::is_sorted(L.reduce.begin(), L.reduce.end(), by_system))
        std::stable_sort(L.reduce.begin(), L.reduce.end(), by_system);
    L.red_first.assign(size_t(nsys), 0);
    L.red_count.assign(size_t(nsys), 0);
    for (size_t i = L.reduce.size(); i-- > 0;) {
        L.red_first[size_t(L.reduce[i].sys)] = int32_t(i);
        L.red_count[size_t(L.reduce[i].sys)]++;
    }
}

}  // namespace

void IndexTiles::add(const SlotProgram* slots, int n, int first)
{
    // row 4 j + role of the tile whose weights start at `at` gains 3^(e mod 5)
    // for digit e of the list, one role per five digits
    auto put = [&](size_t at, int j, const SquareList& l, int e0, int role, int limbs, int step) {
        for (int e = e0; e < int(l.src.size()) && e < e0 + 5 * limbs; e++) {
            const int row = 4 * j + role + step * ((e - e0) / 5);
            const int q = l.src[size_t(e)], d = q % 16, lane = 16 * (q / 16) + row;
            weights[at + size_t(lane) * 16 + size_t(4 * (d % 4) + d / 4)] = int8_t(pow3((e - e0) % 5));
        }
    };
    for (int j0 = 0; j0 < n; j0 += 4) {
        const SlotProgram& s0 = slots[j0];
        IndexTile t{};
        t.slot_first = uint16_t(first + j0);
        t.nslots = uint16_t(std::min(4, n - j0));
        t.hs = s0.hs;
        t.ds = s0.ds;
        t.col_offset = s0.col_offset;
        t.dense_offset = s0.dense_offset;
        size_t longest[3] = {0, 0, 0};
        for (int j = 0; j < t.nslots; j++)
            for (int l = 0; l < 3; l++) longest[l] = std::max(longest[l], slots[j0 + j].list[l].src.size());
        // a pair without a diagonal list is a plain pair (idx * 1 + 0): the
        // kernels' 24-bit multiply by ds then only meets pairs of at most
        // seven squares a half (an index below 2^24)
        t.kind = uint16_t(s0.kind == 2 && longest[2] == 0 ? 1 : s0.kind);
        const bool pair = t.kind == 1 || t.kind == 2;
        if (longest[0] > (pair ? 10u : 20u) || longest[1] > 10 || longest[2] > 10)
            throw Error(CAD_ERR_PATTERN, "a pattern list too long for an index tile");
        t.wide = (pair ? longest[0] > 5 || longest[1] > 5 : longest[0] > 10) ? 1 : 0;
        const size_t at = weights.size();
        weights.resize(at + 2048, 0);
        for (int j = 0; j < t.nslots; j++) {
            const SlotProgram& s = slots[j0 + j];
            if (!pair) {
                put(at, j, s.list[0], 0, 0, 4, 1);
            } else if (t.kind == 1) {
                put(at, j, s.list[0], 0, 0, 2, 2);
                put(at, j, s.list[1], 0, 1, 2, 2);
            } else {
                put(at, j, s.list[0], 0, 0, 1, 1);
                put(at, j, s.list[1], 0, 1, 1, 1);
                put(at, j, s.list[2], 0, 2, 2, 1);
                if (t.wide) {
                    put(at + 1024, j, s.list[0], 5, 0, 1, 1);
                    put(at + 1024, j, s.list[1], 5, 1, 1, 1);
                }
            }
        }
        tiles.push_back(t);
    }
}

// Dynamic LDS a window may use: the device limit minus 1 KB kept for the
// kernels' static LDS (block-reduction scratch).
size_t lds_budget(const Context& ctx)
{
    return std::min<size_t>(ctx.max_lds, 160 * 1024) - 1024;
}

GridSys GatherPlan::sys() const
{
    return GridSys{d_first.as<int32_t>(), d_count.as<int32_t>(), d_counters.as<unsigned>(), d_partials.as<double>()};
}

void build_scatter_plan(ScatterPlan& sp, const std::vector<uint32_t>& lo, const std::vector<uint32_t>& hi,
                        const std::vector<int64_t>& sys_rows, const std::vector<uint32_t>& sys_col,
                        int64_t cols_per_sys, int ibytes, const Context& ctx, const TuneParams& tune, bool fp32,
                        Uploads& up)
{
    make_groups(lo, hi, sp);
    const size_t lds = lds_budget(ctx);
    // the 4-byte windows serve the Jacobi counts only (once per matrix): per-
    // window chunks, several tiles per CU, the u32 partial slices uncapped
    TuneParams t4 = tune;
    t4.scatter_order = 0;
    t4.blocks_per_cu = std::max(4.0, tune.blocks_per_cu);
    t4.partial_cap = 1.0;
    t4.scatter_balance = 1.0;
    t4.pack_slots = kMaxSegSlots;  // (the count kernel holds a group's slots in registers)
    const int nsys = int(sys_rows.size()) - 1;
    auto build = [&](ScatterLists& L, int wbytes, const TuneParams& t, bool f32) {
        make_scatter_lists(sp, sys_rows, sys_col, cols_per_sys, uint32_t(lds / wbytes), wbytes, ibytes, ctx.cus, t,
                           f32, L);
        finish_lists(L, nsys);
        // slot lists padded to whole 32-bit words (the kernels read them as words)
        std::vector<uint16_t> padded = L.slot_list;
        if (padded.size() % 2) padded.push_back(0);
        up.put(L.d_groups, L.groups);
        up.put(L.d_slot_list, padded);
        up.put(L.d_work, L.work);
        up.put(L.d_reduce, L.reduce);
        up.put(L.d_red_first, L.red_first);
        up.put(L.d_red_count, L.red_count);
        up.put(L.d_red_counters, std::vector<unsigned>(size_t(std::max(1, nsys)), 0u));
        up.reserve(L.d_red_partials, 2 * sizeof(double) * std::max<size_t>(1, L.reduce.size()));
        L.part = DBuf();
    };
    build(sp.f4, 4, t4, false);
    build(sp.f8, 8, tune, false);
    if (fp32) build(sp.f8s, 8, tune, true);
}

void plan_scatter_subset(const ScatterPlan& sp, const std::vector<int64_t>& sys_rows,
                         const std::vector<uint32_t>& sys_col, int64_t cols_per_sys, int ibytes, const Context& ctx,
                         const TuneParams& tune, const std::vector<uint8_t>& on, bool fp32, ScatterLists& L)
{
    make_scatter_lists(sp, sys_rows, sys_col, cols_per_sys, uint32_t(lds_budget(ctx) / 8), 8, ibytes, ctx.cus, tune,
                       fp32, L, &on);
    finish_lists(L, int(sys_rows.size()) - 1);
}

GridSys ScatterLists::reduce_sys() const
{
    return GridSys{d_red_first.as<int32_t>(), d_red_count.as<int32_t>(), d_red_counters.as<unsigned>(),
                   d_red_partials.as<double>()};
}

// Row tiles: a thread owns trpt consecutive rows counted from the tile's first
// row rounded down to trpt, so a tile spans at most its runs (or sub-tiles) of
// bs * trpt rows from there; tiles of a system are a multiple of trpt rows long
// (their misalignment is the system's).  A single system is cut into a
// multiple of the CU count so that every CU gets the same number of tiles; the
// systems of a batch into tiles of one length for all, the shortest (of at
// least kSmallTileRows rows: a tile costs its staging whatever its rows) that
// makes no more tiles than a multiple of the CU count.
void cut_tiles(const cad_matrix* m, const GatherPlan& gp, const std::vector<int>* on, std::vector<RowWork>& tiles,
               std::vector<int32_t>& first, std::vector<int32_t>& count)
{
    constexpr int64_t kSmallTileRows = 2048;
    const int64_t slots = int64_t(std::max(1, m->ctx->cus)) * (kTileBlock / gp.bs);  // blocks resident at once
    const int64_t t = gp.trpt;
    const int64_t cap = (int64_t(gp.runs > 0 ? gp.runs : gp.sub) * gp.bs * t - (t - 1)) / t * t;
    auto rows_of = [&](int s) {
        return on && !(*on)[size_t(s)] ? int64_t(0) : m->sys_row_begin[s + 1] - m->sys_row_begin[s];
    };
    auto tiles_of = [&](int64_t per) {
        int64_t n = 0;
        for (int s = 0; s < m->nsys; s++) n += (rows_of(s) + per - 1) / per;
        return n;
    };
    int64_t total = 0;
    for (int s = 0; s < m->nsys; s++) total += rows_of(s);
    // rows a tile: the shortest whose tiles fit `waves` per resident block
    int64_t per = cap;
    const int64_t least = std::min(cap, m->nsys > 1 ? (kSmallTileRows + t - 1) / t * t : t);
    for (int64_t waves = std::max<int64_t>(1, (total + slots * cap - 1) / (slots * cap));; waves++) {
        if (tiles_of(cap) > slots * waves) continue;
        int64_t lo = least / t, hi = cap / t;  // in units of t rows
        while (lo < hi) {
            const int64_t mid = (lo + hi) / 2;
            if (tiles_of(mid * t) <= slots * waves) hi = mid;
            else lo = mid + 1;
        }
        per = hi * t;
        break;
    }
    tiles.clear();
    first.assign(size_t(m->nsys), 0);
    count.assign(size_t(m->nsys), 0);
    for (int s = 0; s < m->nsys; s++) {
        const int64_t r0 = m->sys_row_begin[s], R = rows_of(s);
        first[size_t(s)] = int32_t(tiles.size());
        for (int64_t a = 0; a < R; a += per) tiles.push_back(RowWork{r0 + a, r0 + std::min(R, a + per), s, 0});
        count[size_t(s)] = int32_t(tiles.size()) - first[size_t(s)];
    }
}

// Segments of the tiled gather: the slot groups must be runs of consecutive
// slots that follow each other in slot order (true for pattern matrices, whose
// groups are the patterns); groups wider than the LDS may hold at most
// kMaxSegSlots slots.
void build_gather_plan(cad_matrix* m, GatherPlan& gp, int vbytes, int rpt, int bs, int sub, Uploads& up)
{
    const Context& ctx = *m->ctx;
    const ScatterPlan& sp = m->splan;
    gp.ok = false;
    gp.rpt = rpt;
    gp.bs = bs;
    gp.sub = sub;
    if (rpt <= 0) return;  // the row kernel
    if (bs != kTileBlock && (bs != kTileBlock / 2 || m->mf)) return;
    if (sub < 1 || sub > 3 || (sub > 1 && (bs != kTileBlock || m->mf))) return;
    const int per_cu = kTileBlock / bs;  // blocks resident per CU
    // Long tiles for the full-block kernels over u16 entries with the most rows
    // a thread that they have, where a CU has more rows than one of their
    // tiles: as many runs as its rows need, in as few tiles as the registers
    // allow.
    gp.runs = 0;
    gp.trpt = rpt;
    if (!m->mf && m->ibytes == 2 && bs == kTileBlock && sub == 1 && rpt == (vbytes == 8 ? 2 : 8)) {
        const int64_t per = (m->rows + ctx.cus - 1) / std::max(1, ctx.cus);
        if (per > int64_t(rpt) * kTileBlock) {
            const int64_t run = int64_t(long_rpt(vbytes)) * kTileBlock, most = long_max_runs(vbytes) * run;
            const int64_t n = (per + most - 1) / most;
            gp.trpt = long_rpt(vbytes);
            gp.runs = int(((per + n - 1) / n + gp.trpt + run - 1) / run);
            gp.runs = std::min(gp.runs, long_max_runs(vbytes));
        }
    }
    // A staged run of columns starts at its element offset inside a 16-byte
    // line (up to Q - 1 elements) so that whole lines map to whole LDS lines:
    // windows leave that room, and phase segments start on line boundaries.
    const uint32_t total = uint32_t((lds_budget(ctx) + 1024) / per_cu - 1024) / uint32_t(vbytes);
    const uint32_t Q = uint32_t(16 / vbytes);
    gp.wmax = total - (Q - 1);
    std::vector<const SlotGroup*> order;
    for (auto& g : sp.groups) order.push_back(&g);
    std::sort(order.begin(), order.end(),
              [&](const SlotGroup* a, const SlotGroup* b) { return sp.slot_list[a->first] < sp.slot_list[b->first]; });
    int next = 0;
    gp.segs.clear();
    gp.lds_elems = 0;
    for (const SlotGroup* g : order) {
        const int first = sp.slot_list[g->first];
        if (first != next) return;
        for (int j = 0; j < g->nslots; j++)
            if (sp.slot_list[g->first + j] != first + j) return;
        GatherSeg seg;
        seg.col_lo = g->col_lo;
        seg.width = g->col_hi - g->col_lo;
        seg.slot_first = uint16_t(first);
        seg.nslots = g->nslots;
        seg.nwin = uint16_t((seg.width + gp.wmax - 1) / gp.wmax);
        seg.pad = 0;
        if (seg.nwin > 1 && seg.nslots > kMaxSegSlots) return;
        gp.lds_elems = std::max(gp.lds_elems, std::min(seg.width, gp.wmax) + Q - 1);
        gp.segs.push_back(seg);
        next = first + g->nslots;
    }
    if (next != m->k || gp.segs.empty()) return;
    // Steps of the stored-index kernel: consecutive single-window segments are
    // packed into one staging phase while they fit the LDS together; a wide
    // segment is a step of its own.
    gp.steps.clear();
    gp.phases.clear();
    uint32_t phase_w = 0;
    int open_step = -1;  // the step that stages the current phase
    for (const GatherSeg& sg : gp.segs) {
        const bool wide = sg.nwin > 1;
        if (wide || open_step < 0 || phase_w + sg.width + Q - 1 > total) {
            open_step = -1;
            phase_w = 0;
        }
        // (a wide step of a matrix-free matrix is one index tile)
        const int per_step = gp.runs > 0 ? (wide ? long_wide_slots(vbytes, gp.runs) : kLongStep)
                             : !wide     ? kMaxSegSlots
                             : m->mf     ? 4
                                         : wide_step_slots(rpt * m->ibytes);
        for (int j0 = 0; j0 < sg.nslots; j0 += per_step) {
            GatherStep st{};
            st.slot_first = uint16_t(sg.slot_first + j0);
            st.nslots = uint16_t(std::min<int>(per_step, sg.nslots - j0));
            st.col_lo = sg.col_lo;
            st.width = sg.width;
            st.nwin = sg.nwin;
            st.phase_first = -1;
            st.phase_count = 0;
            if (m->mf) st.tile_first = m->slot_tile[size_t(st.slot_first)];
            for (int j = 0; j < st.nslots; j++) {
                const int slot = st.slot_first + j;
                st.off[j] = (m->ibytes == 2 ? m->slot_lo[size_t(slot)] : 0u) - sg.col_lo;
            }
            if (wide && j0 > 0) {
                // the windows of this step in the other direction, from the
                // one the step before ended on
                st.wflags = uint16_t(kWideStaged | ((j0 / per_step) % 2 ? kWideReverse : 0));
            }
            if (!wide) {
                if (j0 == 0) {
                    if (open_step < 0) {
                        st.phase_first = int16_t(gp.phases.size());
                        open_step = int(gp.steps.size());
                    }
                    gp.phases.push_back(PhaseSeg{sg.col_lo, sg.width, phase_w, 0u});
                }
                st.lds_off = phase_w;
                for (int j = 0; j < st.nslots; j++) st.off[j] += phase_w;
            }
            gp.steps.push_back(st);
        }
        if (!wide) {
            GatherStep& opener = gp.steps[size_t(open_step)];
            opener.phase_count = int16_t(int(gp.phases.size()) - opener.phase_first);
            gp.lds_elems = std::max(gp.lds_elems, phase_w + sg.width + Q - 1);
            phase_w = (phase_w + sg.width + Q - 1 + Q - 1) / Q * Q;
        }
    }
    cut_tiles(m, gp, nullptr, gp.tiles, gp.first, gp.count);
    up.put(gp.d_steps, gp.steps);
    up.put(gp.d_phases, gp.phases);
    up.put(gp.d_tiles, gp.tiles);
    up.put(gp.d_first, gp.first);
    up.put(gp.d_count, gp.count);
    up.put(gp.d_counters, std::vector<unsigned>(size_t(std::max(1, m->nsys)), 0u));
    up.reserve(gp.d_partials, 2 * sizeof(double) * std::max<size_t>(1, gp.tiles.size()));
    gp.ok = true;
}

void build_plans(cad_matrix* m)
{
    const Context& ctx = *m->ctx;
    // per-system column bases (block-diagonal batches); one system by default
    if (m->sys_row_begin.empty()) {
        m->nsys = 1;
        m->sys_row_begin = {0, m->rows};
        m->sys_col = {0};
        m->cols_per_sys = m->cols;
    }
    Uploads up;
    up.put(m->d_sys_col, m->sys_col);
    // (a matrix-free matrix sizes its scatter partials as a u16 matrix would)
    build_scatter_plan(m->splan, m->slot_lo, m->slot_hi, m->sys_row_begin, m->sys_col, m->cols_per_sys,
                       m->mf ? 2 : m->ibytes, ctx, m->tune, true, up);
    build_gather_plan(m, m->gplan4, 4, m->tune.rpt4, m->tune.bs4, m->tune.sub4, up);
    build_gather_plan(m, m->gplan8, 8, m->tune.rpt8, m->tune.bs8, m->tune.sub8, up);

    GridPlan& g = m->grid;
    g.rows.clear();
    g.cols.clear();
    g.row_first.assign(m->nsys, 0);
    g.row_count.assign(m->nsys, 0);
    g.col_first.assign(m->nsys, 0);
    g.col_count.assign(m->nsys, 0);
    // row blocks of the row kernels: one row a thread for a small matrix (its
    // gathers use the row kernel, whose rows' loads are then all in flight)
    const int64_t rchunk = int64_t(kRowBlock) * (m->rows <= kRowKernelRows ? 1 : kRowsPerThread);
    const int64_t cchunk = int64_t(kRowBlock) * 2;  // enough column blocks to cover the CUs
    for (int s = 0; s < m->nsys; s++) {
        g.row_first[s] = int32_t(g.rows.size());
        for (int64_t r = m->sys_row_begin[s]; r < m->sys_row_begin[s + 1]; r += rchunk)
            g.rows.push_back(RowWork{r, std::min(m->sys_row_begin[s + 1], r + rchunk), s, 0});
        g.row_count[s] = int32_t(g.rows.size()) - g.row_first[s];
        g.col_first[s] = int32_t(g.cols.size());
        const int64_t c0 = m->sys_col[s], c1 = c0 + m->cols_per_sys;
        for (int64_t c = c0; c < c1; c += cchunk) g.cols.push_back(ColWork{c, std::min(c1, c + cchunk), s, c == c0});
        g.col_count[s] = int32_t(g.cols.size()) - g.col_first[s];
    }
    up.put(g.d_rows, g.rows);
    up.put(g.d_cols, g.cols);
    up.put(g.d_row_first, g.row_first);
    up.put(g.d_row_count, g.row_count);
    up.put(g.d_col_first, g.col_first);
    up.put(g.d_col_count, g.col_count);
    std::vector<unsigned> zeros(std::max(1, m->nsys), 0u);
    up.put(g.d_row_counters, zeros);
    up.put(g.d_col_counters, zeros);
    up.reserve(g.d_partials, 2 * sizeof(double) * std::max<size_t>(1, std::max(g.rows.size(), g.cols.size())));
    // max |y| per row block, for the fixed-point FP32 scatter
    up.reserve(m->splan.d_ymax_part, sizeof(unsigned) * std::max<size_t>(1, g.rows.size()));
    up.flush(ctx.stream);
}

}  // namespace cad
