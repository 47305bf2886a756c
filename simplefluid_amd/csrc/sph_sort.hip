// Sorting particles by cell key on gfx950, and the cell-start table.
//
// Both sort modes produce the same stable permutation (ties keep the input
// order) and the same lower-bound table cstart[c] = #particles with key < c.
//
// Cell-count sort (default): one kernel.  The integrate pass already linked
// each particle into its cell's chain of runs and counted particles per tile
// of cells, so a block of cell_sort_kernel owns a tile: it takes its
// prefix from the tile sums, counts its cells by following their chains,
// scans the counts (cstart), lists the members cell by cell, each cell's by
// ascending input index (from the chain's links in registers; a longer
// chain's runs are ranked among each other first), and gathers their state
// into its sorted place (pos, vel, id, perm).  No block waits for another.
// Radix sort: one histogram kernel for all 8-bit digits, then one kernel per
// digit that ranks a tile of keys in LDS (wave64 ballot-matching of the
// digit bits, so equal digits rank in lane order without LDS atomics) and
// finds its global offsets by decoupled look-back; a gather kernel then
// reorders the state.  It is kept for key spaces too large to count.
//
// Look-back waits are bounded: a wait that exceeds its bound raises the
// device error flag instead of hanging, and every data-dependent store is
// range-checked.
#include <algorithm>

#include "sph_internal.hpp"

namespace sph {

namespace {

constexpr int kBins = 256;
constexpr int kSortBlock = 256;
constexpr int kSortWaves = kSortBlock / 64;
constexpr uint32_t kFlagAgg = 1u << 30;
constexpr uint32_t kFlagInc = 2u << 30;
constexpr uint32_t kValMask = (1u << 30) - 1u;
constexpr uint32_t kSpinLimit = 1u << 22;
constexpr int kHistItems = 16;

__device__ __forceinline__ uint32_t ld_agent(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Exclusive scan of one value per thread over a 256-thread block; *total
// receives the block sum.
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* s_w, uint32_t* total = nullptr) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
        const uint32_t sw = s_w[w];
        if (w < wave) pre += sw;
        tot += sw;
    }
    __syncthreads();
    if (total) *total = tot;
    return pre + x - v;
}

// Inclusive prefix of the tiles before `tile` in a look-back status array
// (one word per tile and digit: 2-bit flag, 30-bit value).
__device__ __forceinline__ uint32_t look_back(const uint32_t* status, uint32_t stride, uint32_t tile, uint32_t* err) {
    uint32_t prefix = 0;
    int t = (int)tile - 1;
    uint32_t spins = 0;
    while (t >= 0) {
        const uint32_t s = ld_agent(status + (size_t)t * stride);
        const uint32_t f = s & ~kValMask;
        if (f == 0u) {
            if (++spins > kSpinLimit) {
                atomicOr(err, 1u);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
            continue;
        }
        prefix += s & kValMask;
        if (f == kFlagInc) break;
        --t;
    }
    return prefix;
}

// ---------------------------------------------------------------- cell count

// Exclusive scan of one value per thread over a block of BLOCK threads;
// total receives the block sum.
template <int BLOCK>
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* s_w, uint32_t& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; ++w) {
        const uint32_t sw = s_w[w];
        if (w < wave) pre += sw;
        tot += sw;
    }
    total = tot;
    return pre + x - v;
}

// Exclusive scan of the T per-tile sums (head[C .. C+T)) into
// head[C+T+1 .. C+2T+1); with tile_pre, a list of the tiles that need work (not
// empty, or their cells hold another prefix) behind it, its length in
// head[C+T].  Block i scans sums [1024 i, 1024 (i + 1)) and adds up
// all the ones before itself: the reads are coalesced, independent and in
// cache, where one block over all of them waited on itself round by round
// (22k tiles: 14 us).
constexpr int kTileScanBlock = 1024;
// Up to this many tiles each sort block sums the tiles before its own itself
// (24 words per thread at most; tile_scan_kernel's launch costs 5 us); above
// it tile_scan_kernel runs first.
constexpr uint32_t kInlineTiles = 6144;

__global__ __launch_bounds__(kTileScanBlock) void tile_scan_kernel(uint32_t* __restrict__ head, uint32_t C,
                                                                   uint32_t T, const uint32_t* __restrict__ frame,
                                                                   const uint32_t* __restrict__ tile_pre) {
    if (frame && (frame[0] | frame[1])) return;
    __shared__ uint32_t s_w[kTileScanBlock / 64];
    __shared__ uint32_t s_pre[kTileScanBlock / 64];
    __shared__ uint32_t s_at;
    const uint32_t* tsum = head + C;
    const uint32_t i0 = blockIdx.x * (uint32_t)kTileScanBlock, i = i0 + threadIdx.x;
    uint32_t before = 0;
#pragma unroll 8
    for (uint32_t e = threadIdx.x; e < i0; e += (uint32_t)kTileScanBlock) before += tsum[e];
    const uint32_t own = i < T ? tsum[i] : 0u;
    const uint32_t held = tile_pre && i < T ? tile_pre[i] : 0u;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
    if ((threadIdx.x & 63u) == 0u) s_pre[threadIdx.x >> 6] = before;
    uint32_t total;
    uint32_t run = block_scan<kTileScanBlock>(own, s_w, total);
#pragma unroll
    for (int w = 0; w < kTileScanBlock / 64; ++w) run += s_pre[w];
    if (i < T) head[C + T + 1u + i] = run;
    if (!tile_pre) return;
    const bool need = i < T && (own != 0u || held != run);
    uint32_t listed;
    __syncthreads();  // s_w is read by the scan before
    const uint32_t at = block_scan<kTileScanBlock>(need ? 1u : 0u, s_w, listed);
    if (threadIdx.x == 0 && listed) s_at = atomicAdd(head + C + T, listed);
    __syncthreads();
    if (need) head[C + 2u * T + 1u + s_at + at] = i;
}

// Members a cell may hold for the stable in-cell rank.  Rest-density fluid
// holds a few per cell.
constexpr uint32_t kMaxRankCell = 1024;
// Members of a tile listed in LDS, at most eight per cell; a fuller tile lists
// them in global memory.
constexpr uint32_t kTileMembers = 4096;
// Links of one cell followed in its chain; a longer chain (a pile of
// particles in one cell, or an upload in random order of a very full one)
// makes the block find the tile's members by scanning all keys instead.  A
// link costs a read's latency twice, the scan the keys' bytes at one CU's
// rate, kScanQuads 16-byte loads in flight per lane: about the same at one
// link per 2,048 keys.
constexpr uint32_t kMinLinks = 32, kMaxLinks = 1024;
constexpr uint32_t kScanQuads = 6;

struct CellSortArgs {
    uint32_t n, C;
    uint32_t shift;      // cells per tile, as a shift
    uint32_t max_links;
    uint32_t* head;
    const uint32_t* next;
    const uint32_t* key0;
    uint32_t* cstart;
    uint32_t* tile_pre;
    uint32_t* tmp;       // a tile's runs or members on their way to their order, from its sorted place on
    const float4* pos_in;
    const float4* vel_in;
    const uint32_t* id_in;
    float4* pos_out;
    float4* vel_out;
    uint32_t* id_out;
    uint32_t* perm;
    float* soa;
    uint32_t* queue;
    uint32_t* err;
    uint32_t* frame;     // device frame loop's state, or null
    int gather;          // 0: the cell-start table only (radix mode)
};

// Block b sorts the particles of tile b, of up to BLOCK V cells.  Thread t
// owns V consecutive cells; their chains are followed together, so a wave waits
// once per link for the longest chain among its cells, and the first
// kHeldLinks links stay in registers for the listing.  The kernel is bound
// by the latency of its dependent steps at small sizes (tile sums and heads,
// the links, the members' state) and by memory at large ones; one particle's
// state is moved once.
constexpr int kHeldLinks = 5;

// One thread per cell for tiles of up to 512 cells (grids of up to 2^20),
// where the chip waits on each block's dependent steps; four cells per thread
// for tiles of 1024, where 1024-lane blocks only hold up each other's phases.
// Measured at 1024 cells, one against four: DoubleDambreak at resolution 24
// (54 tiles) 7.0 against 11.5 us, 65k dam break (489 tiles) 7.8 against 11.3
// us, 1M (2013 tiles) 29.2 against 23.1 us.
template <int BLOCK, int V>
struct TileSort {
    static constexpr uint32_t kCells = (uint32_t)(BLOCK * V);
    static constexpr uint32_t kMembers = kCells * 8u < kTileMembers ? kCells * 8u : kTileMembers;
    // A tile whose runs are ranked keeps each cell's first run in that room.
    static constexpr uint32_t kRanked = kMembers - (kCells + 1u);
    static_assert(kCells <= 1u << kTileShiftMax, "a tile");
    static_assert(V == 1 || V == 4, "one head, or four in one 16-byte load, per thread");
    uint32_t w[BLOCK / 64];
    uint32_t pre[BLOCK / 64];
    uint32_t big, unsorted;
    uint32_t off[kCells + 1];
    uint32_t mem[kMembers];
};

// The cells of tile b that a thread owns: V == 4 has four of a whole tile, one
// or none where V == 1; past the grid none.  [i0, end), whole: V of them.
template <int V>
struct OwnCells {
    uint32_t i0, end;
    bool whole;
    __device__ __forceinline__ OwnCells(const CellSortArgs& a, uint32_t b) {
        const uint32_t base = b << a.shift, cells = 1u << a.shift;
        i0 = base + (uint32_t)V * threadIdx.x;
        end = V == 1 && base + cells < a.C ? base + cells : a.C;
        whole = i0 + (uint32_t)V <= end;
    }
    __device__ __forceinline__ void heads(const CellSortArgs& a, uint32_t (&r)[V]) const {
        if (V == 4 && whole) {
            const uint4 hv = *reinterpret_cast<const uint4*>(a.head + i0);
            r[0] = hv.x;
            r[V > 1 ? 1 : 0] = V > 1 ? hv.y : hv.x;
            r[V > 2 ? 2 : 0] = V > 2 ? hv.z : hv.x;
            r[V > 3 ? 3 : 0] = V > 3 ? hv.w : hv.x;
        } else {
#pragma unroll
            for (int v = 0; v < V; ++v) r[v] = i0 + (uint32_t)v < end ? a.head[i0 + v] : 0u;
        }
    }
};

// Sorts tile b of T: pre particles before it, `members` in it, heads its own
// cells' chains, held what tile_pre says of it (read by every thread before any
// thread of the block rewrites it).  sh.big and sh.unsorted are 0.
template <int BLOCK, int V>
__device__ __forceinline__ void sort_tile(const CellSortArgs& a, TileSort<BLOCK, V>& sh, uint32_t T, uint32_t b,
                                          uint32_t pre, uint32_t members, uint32_t held, const OwnCells<V>& own_cells,
                                          const uint32_t (&heads)[V]) {
    constexpr uint32_t kCells = TileSort<BLOCK, V>::kCells, kMembers = TileSort<BLOCK, V>::kMembers,
                       kRanked = TileSort<BLOCK, V>::kRanked;
    uint32_t(&s_w)[BLOCK / 64] = sh.w;
    uint32_t &s_big = sh.big, &s_unsorted = sh.unsorted;
    uint32_t(&s_off)[kCells + 1] = sh.off;
    uint32_t(&s_mem)[kMembers] = sh.mem;
    const uint32_t C = a.C;
    const int tid = threadIdx.x;
    const uint32_t cells = 1u << a.shift;
    const uint32_t base = b << a.shift;
    const uint32_t i0 = own_cells.i0, Ce = own_cells.end;
    const bool whole = own_cells.whole;
    uint32_t r[kHeldLinks + 1][V];
#pragma unroll
    for (int v = 0; v < V; ++v) r[0][v] = heads[v];
    if (members == 0u) {
        // An empty tile's cells all hold its prefix; skip the rewrite when
        // this table already holds that prefix there (most empty tiles of
        // a sparse grid keep theirs from step to step).
        if (held == pre) return;
        if (tid == 0) a.tile_pre[b] = pre;
        if (V == 4 && whole) {
            *reinterpret_cast<uint4*>(a.cstart + i0) = make_uint4(pre, pre, pre, pre);
        } else {
            for (uint32_t e = i0; e < Ce && e < i0 + (uint32_t)V; ++e) a.cstart[e] = pre;
        }
        if (b == T - 1u && tid == 0) a.cstart[C] = pre;
        return;
    }
    if (tid == 0) a.tile_pre[b] = 0xffffffffu;
    const __amdgpu_buffer_rsrc_t rnext = buffer_of(a.next, a.n);
    // The run before r in its cell; for the empty run, past the array's end, 0.
    auto link = [&](uint32_t run) -> uint32_t {
        return __builtin_amdgcn_raw_buffer_load_b32(rnext, (int)(run ? run_first(run) << 2 : 0xfffffffcu), 0, 0);
    };
    auto any = [&](const uint32_t* q) __attribute__((always_inline)) -> bool {
        uint32_t o = 0;
#pragma unroll
        for (int v = 0; v < V; ++v) o |= q[v];
        return o != 0u;
    };
    uint32_t cnt[V], more[V];  // per cell: members, links past the held ones
#pragma unroll
    for (int v = 0; v < V; ++v) {
        cnt[v] = run_len(r[0][v]);
        more[v] = 0u;
    }
#pragma unroll
    for (int l = 0; l < kHeldLinks; ++l) {
#pragma unroll
        for (int v = 0; v < V; ++v) r[l + 1][v] = 0u;
        if (__ballot(any(r[l]))) {
#pragma unroll
            for (int v = 0; v < V; ++v) r[l + 1][v] = link(r[l][v]);
#pragma unroll
            for (int v = 0; v < V; ++v) cnt[v] += run_len(r[l + 1][v]);
        }
    }
    // The heads are empty again for the integrate pass.
    if (any(r[0])) {
        if (V == 4 && whole) {
            *reinterpret_cast<uint4*>(a.head + i0) = make_uint4(0u, 0u, 0u, 0u);
        } else {
            for (uint32_t e = i0; e < Ce && e < i0 + (uint32_t)V; ++e) a.head[e] = 0u;
        }
    }
    {
        uint32_t q[V];
#pragma unroll
        for (int v = 0; v < V; ++v) q[v] = r[kHeldLinks][v];
        uint32_t links = (uint32_t)kHeldLinks;
        if (any(q)) s_unsorted = 1u;  // longer than the registers hold (a last run may follow none: no matter)
        while (any(q)) {
            if (++links > a.max_links) {
                s_big = 1u;
                break;
            }
#pragma unroll
            for (int v = 0; v < V; ++v) {
                more[v] += q[v] ? 1u : 0u;
                q[v] = link(q[v]);
                cnt[v] += run_len(q[v]);
            }
        }
    }
    __syncthreads();
    const bool big = s_big != 0u;
    if (big) {
        // Find the tile's members by scanning all keys: their counts per cell
        // (s_off) and, in any order, themselves (tmp; s_off's last word counts
        // them).
        for (uint32_t i = (uint32_t)tid; i <= kCells; i += BLOCK) s_off[i] = 0u;
        __syncthreads();
        const __amdgpu_buffer_rsrc_t rkey = buffer_of(a.key0, a.n);
        const uint32_t room = a.gather && pre < a.n ? min(members, a.n - pre) : 0u;
        for (uint32_t q0 = (uint32_t)tid; 4u * q0 < a.n; q0 += kScanQuads * (uint32_t)BLOCK) {
            u32x4 key[kScanQuads];
#pragma unroll
            for (uint32_t u = 0; u < kScanQuads; ++u)
                key[u] = __builtin_amdgcn_raw_buffer_load_b128(rkey, (int)(q0 << 4), (int)(u * (uint32_t)BLOCK * 16u), 0);
#pragma unroll
            for (uint32_t u = 0; u < kScanQuads; ++u) {
                const uint32_t c[4] = {key[u].x - base, key[u].y - base, key[u].z - base, key[u].w - base};
                if (min(min(c[0], c[1]), min(c[2], c[3])) >= cells) continue;
#pragma unroll
                for (uint32_t e = 0; e < 4u; ++e) {
                    const uint32_t k = 4u * (q0 + u * (uint32_t)BLOCK) + e;
                    if (c[e] < cells && k < a.n) {
                        atomicAdd(&s_off[c[e]], 1u);
                        const uint32_t at = atomicAdd(&s_off[kCells], 1u);
                        if (at < room) a.tmp[pre + at] = k;
                    }
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < V; ++v) cnt[v] = s_off[V * tid + v];
        __syncthreads();
    }
    uint32_t own = 0, total;
#pragma unroll
    for (int v = 0; v < V; ++v) own += cnt[v];
    uint32_t off[V];
    off[0] = block_scan<BLOCK>(own, s_w, total);
#pragma unroll
    for (int v = 1; v < V; ++v) off[v] = off[v - 1] + cnt[v - 1];
    if (V == 4 && whole) {
        *reinterpret_cast<uint4*>(a.cstart + i0) = make_uint4(pre + off[0], pre + off[V > 1 ? 1 : 0],
                                                              pre + off[V > 2 ? 2 : 0], pre + off[V > 3 ? 3 : 0]);
    } else {
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (i0 + (uint32_t)v < Ce) a.cstart[i0 + v] = pre + off[v];
    }
    if (b == T - 1u && tid == 0) a.cstart[C] = pre + total;
    if (!a.gather) return;
    if (pre > a.n || total > a.n - pre || total > members) {  // inconsistent sums: never write out of bounds
        if (tid == 0) atomicOr(a.err, 2u);
        return;
    }
#pragma unroll
    for (int v = 0; v < V; ++v) s_off[V * tid + v] = off[v];
    if (tid == 0) s_off[kCells] = total;
    // The members, cell by cell, each cell's by ascending index.
    const bool unsorted = big || s_unsorted != 0u;
    const bool in_lds = !big && total <= (unsorted ? kRanked : kMembers);
    uint32_t* const s_list = unsorted ? s_mem + (kCells + 1u) : s_mem;
    uint32_t* const list = a.perm + pre;  // too many for LDS: where they end up
    uint32_t* const tmp = a.tmp + pre;
    if (!unsorted) {
        // Every cell's runs are in registers: their first particles order them.
        auto put_all = [&](auto&& put) __attribute__((always_inline)) {
#pragma unroll
            for (int l = 0; l < kHeldLinks; ++l) {
                if (__ballot(any(r[l])) != 0u) {
#pragma unroll
                    for (int v = 0; v < V; ++v) {
                        const uint32_t k = run_first(r[l][v]);
                        uint32_t at = off[v];
#pragma unroll
                        for (int o = 0; o < kHeldLinks; ++o)
                            if (o != l) at += run_first(r[o][v]) < k ? run_len(r[o][v]) : 0u;
                        const uint32_t end = k + run_len(r[l][v]);
                        for (uint32_t t = k; t < end; ++t, ++at) put(at, t);
                    }
                }
            }
        };
        if (in_lds)
            put_all([&](uint32_t i, uint32_t k) { s_mem[i] = k; });
        else
            put_all([&](uint32_t i, uint32_t k) { list[i] = k; });
    } else if (!big) {
        // Longer chains: all runs of the tile go to tmp, cell by cell, and each
        // finds its place among its cell's (a rank by members costs that many
        // times more: cells of 54, 216,000 particles, 230 us).
        uint32_t* const s_first = s_mem;  // each cell's first run in tmp
        uint32_t runs[V], mine = 0u;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            runs[v] = more[v];
#pragma unroll
            for (int l = 0; l < kHeldLinks; ++l) runs[v] += r[l][v] ? 1u : 0u;
            mine += runs[v];
        }
        uint32_t nruns, at[V];
        __syncthreads();  // s_w is read by the scan before
        at[0] = block_scan<BLOCK>(mine, s_w, nruns);
#pragma unroll
        for (int v = 1; v < V; ++v) at[v] = at[v - 1] + runs[v - 1];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            s_first[V * tid + v] = at[v];
#pragma unroll
            for (int l = 0; l < kHeldLinks; ++l)
                if (r[l][v]) tmp[at[v]++] = r[l][v];
        }
        uint32_t q[V];
#pragma unroll
        for (int v = 0; v < V; ++v) q[v] = r[kHeldLinks][v];
        while (any(q)) {
#pragma unroll
            for (int v = 0; v < V; ++v) {
                if (q[v]) tmp[at[v]++] = q[v];
                q[v] = link(q[v]);
            }
        }
        if (tid == 0) s_first[kCells] = nruns;
        __threadfence_block();
        __syncthreads();
        for (uint32_t i = (uint32_t)tid; i < nruns; i += BLOCK) {
            const uint32_t k = run_first(tmp[i]), len = run_len(tmp[i]);
            const uint32_t c = k < a.n ? a.key0[k] - base : cells;
            if (c >= cells) {
                atomicOr(a.err, 4u);
                continue;
            }
            uint32_t d = s_off[c];
#pragma unroll 4
            for (uint32_t t = s_first[c]; t < s_first[c + 1u]; ++t) {
                const uint32_t q = tmp[t];
                d += run_first(q) < k ? run_len(q) : 0u;
            }
            if (s_off[c + 1u] - s_off[c] > kMaxRankCell) atomicOr(a.err, 8u);
            for (uint32_t t = 0; t < len && d + t < total; ++t) {
                if (in_lds)
                    s_list[d + t] = k + t;
                else
                    list[d + t] = k + t;
            }
        }
    } else {
        // From tmp to their cells, then each to its rank, in tmp again.
        // f(j, k, c): member j of src, k, lies in cell c; eight loads of each
        // kind in flight.
        auto each = [&](const uint32_t* src, auto&& f) __attribute__((always_inline)) {
            constexpr int kEach = 8;
            for (uint32_t j0 = (uint32_t)tid; j0 < total; j0 += (uint32_t)(kEach * BLOCK)) {
                uint32_t k[kEach], c[kEach];
#pragma unroll
                for (int u = 0; u < kEach; ++u) k[u] = src[min(j0 + (uint32_t)(u * BLOCK), total - 1u)];
#pragma unroll
                for (int u = 0; u < kEach; ++u) c[u] = a.key0[min(k[u], a.n - 1u)] - base;
#pragma unroll
                for (int u = 0; u < kEach; ++u) {
                    const uint32_t j = j0 + (uint32_t)(u * BLOCK);
                    if (j >= total) break;
                    if (k[u] < a.n && c[u] < cells)
                        f(j, k[u], c[u]);
                    else
                        atomicOr(a.err, 4u);
                }
            }
        };
        __threadfence_block();
        __syncthreads();
        each(tmp, [&](uint32_t, uint32_t k, uint32_t c) {
            const uint32_t at = atomicAdd(&s_off[c], 1u);
            if (at < total) list[at] = k;
        });
        __syncthreads();
        // The counters ended at the next cell's start.
#pragma unroll
        for (int v = 0; v < V; ++v) s_off[V * tid + v] = off[v];
        __threadfence_block();
        __syncthreads();
        bool over = false;
        each(list, [&](uint32_t j, uint32_t k, uint32_t c) {
            const uint32_t lo = s_off[c], hi = s_off[c + 1u];
            uint32_t d = j;
            if (hi - lo <= kMaxRankCell) {
                d = lo;
#pragma unroll 8
                for (uint32_t t = lo; t < hi; ++t) d += list[t] < k ? 1u : 0u;
            } else {
                // A cell this full only arises from collapsed or non-finite
                // positions (clamped into one cell).  Ranking it costs its
                // size per member, so it keeps the order its members were
                // listed in (a valid permutation, not the stable one) and
                // raises the error flag instead.  The block moves it alone:
                // 20,000 such particles among 1.9M make the sort 540 us, 200,000
                // among 1M 1,120 (one key at a time per lane: 4,700 and 4,600).
                over = true;
            }
            tmp[d] = k;
        });
        if (over) atomicOr(a.err, 8u);
    }
    __threadfence_block();
    __syncthreads();
    // V members per thread at a time, so that their state's loads overlap
    // (one at a time, a full tile's 256-thread block waited for eight to
    // sixteen loads in a row).
    const __amdgpu_buffer_rsrc_t rpos = buffer_of(a.pos_in, a.n);
    const __amdgpu_buffer_rsrc_t rvel = buffer_of(a.vel_in, a.n);
    const __amdgpu_buffer_rsrc_t rid = buffer_of(a.id_in, a.n);
    for (uint32_t j0 = (uint32_t)tid; j0 < total; j0 += V * BLOCK) {
        uint32_t k[V];
        float4 pk[V], vk[V];
        uint32_t ik[V];
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const uint32_t j = j0 + (uint32_t)(v * BLOCK);
            k[v] = 0xffffffffu;
            if (j < total) k[v] = in_lds ? s_list[j] : big ? tmp[j] : list[j];
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            // No member: past the buffers' ends.
            pk[v] = load4(rpos, min(k[v], a.n) << 4);
            vk[v] = load4(rvel, min(k[v], a.n) << 4);
            ik[v] = __builtin_amdgcn_raw_buffer_load_b32(rid, (int)(min(k[v], a.n) << 2), 0, 0);
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const uint32_t j = j0 + (uint32_t)(v * BLOCK);
            if (j >= total) break;
            if (k[v] >= a.n) {
                atomicOr(a.err, 4u);
                continue;
            }
            const uint32_t dst = pre + j;
            if (in_lds || big) a.perm[dst] = k[v];
            a.pos_out[dst] = pk[v];
            if (a.soa) {  // the planes, for the gathered density pass
                a.soa[dst] = pk[v].x;
                a.soa[a.n + dst] = pk[v].y;
                a.soa[2 * (size_t)a.n + dst] = pk[v].z;
            }
            a.vel_out[dst] = vk[v];
            a.id_out[dst] = ik[v];
        }
    }
}

template <int BLOCK, int V>
__global__ __launch_bounds__(BLOCK) void cell_sort_kernel(CellSortArgs a) {
    // A frame that is complete (pending, or halted already) skips the step;
    // the first kernel of the step turns pending into halt for the others.
    if (a.frame && (a.frame[0] | a.frame[1])) {
        if (blockIdx.x == 0 && threadIdx.x == 0) a.frame[0] = 1u;
        return;
    }
    constexpr int kWaves = BLOCK / 64;
    __shared__ TileSort<BLOCK, V> sh;
    const uint32_t b = blockIdx.x, C = a.C;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Tile counters of this step's persistent density and force launches.
    if (b == 0 && tid < kQueueWords && a.queue) a.queue[tid] = 0u;
    const uint32_t T = gridDim.x;
    const OwnCells<V> own(a, b);
    uint32_t heads[V];
    own.heads(a, heads);
    const uint32_t held = a.tile_pre[b];
    const uint32_t members = a.head[C + b];
    uint32_t pre;
    if (T <= kInlineTiles) {
        uint32_t x = 0;
#pragma unroll 8
        for (uint32_t i = (uint32_t)tid; i < b; i += BLOCK) x += a.head[C + i];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
        if (lane == 0) sh.pre[wave] = x;
        if (tid == 0) sh.big = sh.unsorted = 0u;
        __syncthreads();
        pre = 0u;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) pre += sh.pre[w];
    } else {
        pre = a.head[C + T + 1u + b];
        if (tid == 0) sh.big = sh.unsorted = 0u;
        __syncthreads();
    }
    sort_tile<BLOCK, V>(a, sh, T, b, pre, members, held, own, heads);
}

// A sparse grid's tiles are mostly empty, and a block of its own for each of
// them, whose reads of the prefix and of the table wait on each other, takes
// most of the sort.  Where tile_scan_kernel runs anyway it lists the tiles
// that need work, and as many blocks as are resident at once take those in
// turn.  Sort pass, block per tile against list: 1,100 scenes of 125 particles
// (134,000 tiles) 115 -> 33 us, 260 of 512 (32,000) 35 -> 20, 60 of 180 (7,300)
// 16.1 -> 15.0.  With fewer tiles the scan's launch costs what the list saves
// (30 scenes of 4,600, 3,700 tiles: 15.6 against 18.1); with more particles a
// tile few are empty.
constexpr uint32_t kSparseMembers = 64;    // particles per tile below which
constexpr uint32_t kSparseBlocks = 1536;   // six a CU, as registers allow

template <int BLOCK, int V>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(6, 6))) void cell_sort_sparse_kernel(
    CellSortArgs a, uint32_t T) {
    if (a.frame && (a.frame[0] | a.frame[1])) {
        if (blockIdx.x == 0 && threadIdx.x == 0) a.frame[0] = 1u;
        return;
    }
    __shared__ TileSort<BLOCK, V> sh;
    const uint32_t C = a.C;
    if (blockIdx.x == 0 && threadIdx.x < (uint32_t)kQueueWords && a.queue) a.queue[threadIdx.x] = 0u;
    const uint32_t listed = a.head[C + T];
    for (uint32_t i = blockIdx.x; i < listed; i += gridDim.x) {
        const uint32_t t = a.head[C + 2u * T + 1u + i];
        const OwnCells<V> own(a, t);
        uint32_t heads[V];
        own.heads(a, heads);
        const uint32_t pre = a.head[C + T + 1u + t], members = a.head[C + t], held = a.tile_pre[t];
        __syncthreads();  // the tile before is done with the room they share
        if (threadIdx.x == 0) sh.big = sh.unsorted = 0u;
        __syncthreads();
        sort_tile<BLOCK, V>(a, sh, T, t, pre, members, held, own, heads);
    }
}

// --------------------------------------------------------------------- radix

// Digit histograms of all passes; zeroes the look-back status words and the
// tile tickets of this sort.
__global__ __launch_bounds__(kSortBlock) void radix_histogram_kernel(
    const uint32_t* __restrict__ keys, uint32_t n, int passes, uint32_t* __restrict__ hist,
    uint32_t* __restrict__ status, uint32_t status_words, uint32_t* __restrict__ tickets) {
    __shared__ uint32_t s_hist[kMaxPasses * kBins];
    for (int i = threadIdx.x; i < kMaxPasses * kBins; i += kSortBlock) s_hist[i] = 0;
    __syncthreads();
    // Each thread counts a contiguous run of keys and only flushes a digit to
    // LDS when it changes: sorted-ish input keeps the high digits constant.
    const uint32_t first = (blockIdx.x * kSortBlock + threadIdx.x) * kHistItems;
    uint32_t cur[kMaxPasses], cnt[kMaxPasses];
#pragma unroll
    for (int p = 0; p < kMaxPasses; ++p) { cur[p] = 0xffffffffu; cnt[p] = 0; }
    for (int q = 0; q < kHistItems; ++q) {
        const uint32_t i = first + q;
        if (i >= n) break;
        const uint32_t k = keys[i];
#pragma unroll
        for (int p = 0; p < kMaxPasses; ++p) {
            if (p >= passes) break;
            const uint32_t d = (k >> (8 * p)) & 255u;
            if (d != cur[p]) {
                if (cnt[p]) atomicAdd(&s_hist[p * kBins + cur[p]], cnt[p]);
                cur[p] = d;
                cnt[p] = 0;
            }
            cnt[p]++;
        }
    }
#pragma unroll
    for (int p = 0; p < kMaxPasses; ++p)
        if (p < passes && cnt[p]) atomicAdd(&s_hist[p * kBins + cur[p]], cnt[p]);
    const uint32_t stride = gridDim.x * kSortBlock;
    const uint32_t tid = blockIdx.x * kSortBlock + threadIdx.x;
    for (uint32_t i = tid; i < status_words; i += stride) status[i] = 0u;
    if (tid < (uint32_t)kMaxPasses) tickets[tid] = 0u;
    __syncthreads();
    for (int i = threadIdx.x; i < passes * kBins; i += kSortBlock) {
        const uint32_t v = s_hist[i];
        if (v) atomicAdd(&hist[i], v);
    }
}

template <int ITEMS>
__global__ __launch_bounds__(kSortBlock) void radix_pass_kernel(
    const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
    uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out,
    const uint32_t* __restrict__ hist, uint32_t* status, uint32_t* ticket, uint32_t n, int shift,
    uint32_t* err) {
    constexpr int TILE = kSortBlock * ITEMS;
    __shared__ uint32_t s_keys[TILE];
    __shared__ uint32_t s_vals[TILE];
    __shared__ uint32_t s_wcnt[kSortWaves][kBins];
    __shared__ uint32_t s_gbase[kBins];
    __shared__ uint32_t s_lstart[kBins];
    __shared__ uint32_t s_w[kSortWaves];
    __shared__ uint32_t s_tile;

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    if (tid == 0) s_tile = atomicAdd(ticket, 1u);
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) s_wcnt[w][tid] = 0u;
    __syncthreads();
    const uint32_t tile = s_tile;
    const uint32_t tbase = tile * (uint32_t)TILE;

    uint32_t key[ITEMS], val[ITEMS], rank[ITEMS];
    const uint32_t wbase = tbase + (uint32_t)(wave * 64 * ITEMS) + (uint32_t)lane;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const uint32_t idx = wbase + (uint32_t)(i * 64);
        const bool valid = idx < n;
        key[i] = valid ? keys_in[idx] : 0xffffffffu;
        val[i] = valid ? (vals_in ? vals_in[idx] : idx) : 0u;
    }
    const uint64_t lt_mask = (1ull << lane) - 1ull;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const bool valid = wbase + (uint32_t)(i * 64) < n;
        const uint32_t d = (key[i] >> shift) & 255u;
        uint64_t m = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            m &= bit ? bb : ~bb;
        }
        const uint32_t pre = (uint32_t)__popcll(m & lt_mask);
        const uint32_t cnt = (uint32_t)__popcll(m);
        uint32_t base = 0;
        if (valid) base = s_wcnt[wave][d];
        __builtin_amdgcn_wave_barrier();
        rank[i] = base + pre;
        if (valid && pre == 0) s_wcnt[wave][d] = base + cnt;
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();

    // Thread tid owns digit tid from here on.
    uint32_t tot = 0;
#pragma unroll
    for (int w = 0; w < kSortWaves; ++w) {
        const uint32_t c = s_wcnt[w][tid];
        s_wcnt[w][tid] = tot;
        tot += c;
    }
    uint32_t* my = status + (size_t)tile * kBins + tid;
    st_agent(my, (tile == 0 ? kFlagInc : kFlagAgg) | tot);
    const uint32_t lstart = block_exclusive_scan(tot, s_w);
    const uint32_t hbase = block_exclusive_scan(hist[tid], s_w);
    s_lstart[tid] = lstart;
    uint32_t prefix = 0;
    if (tile > 0) {
        prefix = look_back(status + tid, kBins, tile, err);
        st_agent(my, kFlagInc | (prefix + tot));
    }
    s_gbase[tid] = hbase + prefix;
    __syncthreads();

#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        if (wbase + (uint32_t)(i * 64) < n) {
            const uint32_t d = (key[i] >> shift) & 255u;
            const uint32_t pos = s_lstart[d] + s_wcnt[wave][d] + rank[i];
            s_keys[pos] = key[i];
            s_vals[pos] = val[i];
        }
    }
    __syncthreads();
    const uint32_t count = n - tbase < (uint32_t)TILE ? n - tbase : (uint32_t)TILE;
#pragma unroll
    for (int q = 0; q < ITEMS; ++q) {
        const uint32_t idx = (uint32_t)(q * kSortBlock + tid);
        if (idx < count) {
            const uint32_t k = s_keys[idx];
            const uint32_t d = (k >> shift) & 255u;
            const uint32_t out = s_gbase[d] + idx - s_lstart[d];
            if (out < n) {
                keys_out[out] = k;
                vals_out[out] = s_vals[idx];
            } else {
                atomicOr(err, 2u);  // inconsistent histogram: never write out of bounds
            }
        }
    }
}

__global__ void radix_reorder_kernel(uint32_t n, const uint32_t* __restrict__ perm,
                                     const float4* __restrict__ pos_in, const float4* __restrict__ vel_in,
                                     const uint32_t* __restrict__ id_in, float4* __restrict__ pos_out,
                                     float4* __restrict__ vel_out, uint32_t* __restrict__ id_out,
                                     uint32_t* __restrict__ hist_zero, uint32_t* __restrict__ err,
                                     float* __restrict__ soa) {
    if (blockIdx.x == 0)
        for (uint32_t i = threadIdx.x; i < (uint32_t)(kMaxPasses * kBins); i += blockDim.x) hist_zero[i] = 0u;
    const uint32_t k = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint32_t s = perm[k];
    if (s >= n) {
        atomicOr(err, 4u);
        return;
    }
    const float4 ps = pos_in[s];
    pos_out[k] = ps;
    if (soa) {
        soa[k] = ps.x;
        soa[n + k] = ps.y;
        soa[2 * (size_t)n + k] = ps.z;
    }
    vel_out[k] = vel_in[s];
    id_out[k] = id_in[s];
}

inline uint32_t blocks_for(size_t n, int b) { return (uint32_t)((n + b - 1) / b); }

}  // namespace

uint32_t sort_tiles(uint32_t n, int items) {
    const uint32_t tile = (uint32_t)(kSortBlock * items);
    return (n + tile - 1) / tile;
}

int sort_key_passes(uint32_t ncells) {
    int bits = 1;
    while (bits < 32 && (1ull << bits) < (uint64_t)ncells) ++bits;
    return (bits + 7) / 8;
}

#define SPH_CELL_SORT(block, v) HIP_KERNEL_NAME(cell_sort_kernel<block, v>)

static void launch_cell_sort(hipStream_t st, const SortPlan& sp, int gather) {
    const uint32_t tiles = scan_tiles(sp.ncells, sp.tile_shift);
    const bool sparse = tiles > kInlineTiles && sp.n / tiles < kSparseMembers && sp.tile_shift == kTileShiftMax;
    if (tiles > kInlineTiles)
        hipLaunchKernelGGL(tile_scan_kernel, dim3((tiles + kTileScanBlock - 1) / kTileScanBlock), dim3(kTileScanBlock),
                           0, st, sp.head, sp.ncells, tiles, sp.frame, sparse ? sp.tile_pre : nullptr);
    CellSortArgs a;
    a.n = sp.n;
    a.C = sp.ncells;
    a.shift = sp.tile_shift;
    a.max_links = std::min(std::max(sp.n >> 11, kMinLinks), kMaxLinks);
    a.head = sp.head;
    a.next = sp.next;
    a.key0 = sp.key0;
    a.cstart = sp.cstart;
    a.tile_pre = sp.tile_pre;
    a.tmp = sp.tmp;
    a.pos_in = sp.pos_in;
    a.vel_in = sp.vel_in;
    a.id_in = sp.id_in;
    a.pos_out = sp.pos_out;
    a.vel_out = sp.vel_out;
    a.id_out = sp.id_out;
    a.perm = sp.perm;
    a.soa = sp.soa_out;
    a.queue = sp.queue;
    a.err = sp.err;
    a.frame = sp.frame;
    a.gather = gather;
    if (sp.tile_shift <= 8u)
        hipLaunchKernelGGL(SPH_CELL_SORT(256, 1), dim3(tiles), dim3(256), 0, st, a);
    else if (sp.tile_shift == 9u)
        hipLaunchKernelGGL(SPH_CELL_SORT(512, 1), dim3(tiles), dim3(512), 0, st, a);
    else if (sparse)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(cell_sort_sparse_kernel<256, 4>), dim3(kSparseBlocks), dim3(256), 0, st, a,
                           tiles);
    else
        hipLaunchKernelGGL(SPH_CELL_SORT(256, 4), dim3(tiles), dim3(256), 0, st, a);
}

hipError_t launch_sort_keys(hipStream_t st, const SortPlan& sp) {
    if (sp.n == 0) return hipSuccess;
    if (sp.mode == kSortCellCount) {
        launch_cell_sort(st, sp, 1);
        return hipGetLastError();
    }
    launch_cell_sort(st, sp, 0);
    if (sp.frame) return hipErrorInvalidValue;  // the frame loop runs the cell-count sort only
    const uint32_t tiles = sort_tiles(sp.n, sp.items);
    const uint32_t hist_blocks = (sp.n + kSortBlock * kHistItems - 1) / (kSortBlock * kHistItems);
    const uint32_t status_words = (uint32_t)sp.passes * tiles * kBins;
    hipLaunchKernelGGL(radix_histogram_kernel, dim3(hist_blocks), dim3(kSortBlock), 0, st, sp.key0, sp.n,
                       sp.passes, sp.hist, sp.status, status_words, sp.tickets);
    for (int p = 0; p < sp.passes; ++p) {
        const bool last = p == sp.passes - 1;
        const uint32_t* kin = p == 0 ? sp.key0 : sp.kbuf[(p - 1) & 1];
        const uint32_t* vin = p == 0 ? nullptr : sp.vbuf[(p - 1) & 1];
        uint32_t* kout = last ? sp.skey : sp.kbuf[p & 1];
        uint32_t* vout = last ? sp.perm : sp.vbuf[p & 1];
        uint32_t* status = sp.status + (size_t)p * tiles * kBins;
        const uint32_t* hist = sp.hist + p * kBins;
        switch (sp.items) {
            case 4:
                hipLaunchKernelGGL(radix_pass_kernel<4>, dim3(tiles), dim3(kSortBlock), 0, st, kin, vin,
                                   kout, vout, hist, status, sp.tickets + p, sp.n, 8 * p, sp.err);
                break;
            case 12:
                hipLaunchKernelGGL(radix_pass_kernel<12>, dim3(tiles), dim3(kSortBlock), 0, st, kin, vin,
                                   kout, vout, hist, status, sp.tickets + p, sp.n, 8 * p, sp.err);
                break;
            case 16:
                hipLaunchKernelGGL(radix_pass_kernel<16>, dim3(tiles), dim3(kSortBlock), 0, st, kin, vin,
                                   kout, vout, hist, status, sp.tickets + p, sp.n, 8 * p, sp.err);
                break;
            default:
                hipLaunchKernelGGL(radix_pass_kernel<8>, dim3(tiles), dim3(kSortBlock), 0, st, kin, vin,
                                   kout, vout, hist, status, sp.tickets + p, sp.n, 8 * p, sp.err);
                break;
        }
    }
    return hipGetLastError();
}

hipError_t launch_sort_gather(hipStream_t st, const SortPlan& sp) {
    if (sp.n == 0) return hipSuccess;
    if (sp.mode == kSortRadix)
        hipLaunchKernelGGL(radix_reorder_kernel, dim3(blocks_for(sp.n, sp.reorder_block)), dim3(sp.reorder_block),
                           0, st, sp.n, sp.perm, sp.pos_in, sp.vel_in, sp.id_in, sp.pos_out, sp.vel_out,
                           sp.id_out, sp.hist, sp.err, sp.soa_out);
    return hipGetLastError();
}

}  // namespace sph
