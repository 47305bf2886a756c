// Shared device-side definitions of the gfx950 SPH engine.
//
// Data layout in HBM (N particles, C cells over all scenes):
//   pos[2], vel[2]  float4 x N   state order / sorted order (16 B aligned loads); in
//                                sorted order pos.w = p/rho^2 and vel.w = 1/rho
//                                (written by the density pass for the force pass)
//   id[2]           uint32 x N   original particle id, state / sorted order
//   key0            uint32 x N   cell key of the state positions (written by integrate)
//   head            uint32 x C+3T+1 per cell, the newest run of particles that entered it
//                                (0: none; built by the integrate pass, cleared by the
//                                sort), then particles per tile of cells, then (with many
//                                tiles) the list of those that need work: its length, the
//                                exclusive scan of the tile sums, the list
//   next            uint32 x N   per run (at its first particle), the cell's run before it
//   radix ping-pong 2 x (uint32 key + uint32 value) x N (radix mode)
//   cstart          uint32 x C+1 lower-bound cell-start table: cstart[c] = #particles with key < c
//   rho             float  x N   density (sorted order)
//   mask            uint32 x 9N  neighbour bits, row-major [row][particle] (layout at
//                                mask_span below)
// All kernels are written for wave64 and 256 CUs in 8 XCDs.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sph {

// Per-scene constants, one table entry per scene (a single-scene handle has
// a table of one).  Kernels read a tile's entry through scene_at.
struct SceneConst {
    float bmin[3];
    float inv_cs;      // 1 / (h (1 + 2^-10)), the cell size's reciprocal
    float lo[3];       // clamp bounds: box_min + r
    float h;
    float hi[3];       // box_max - r
    float h2;
    int   G[3];        // grid cells per axis
    uint32_t cell_offset;  // first cell key of this scene
    float cD;          // m * 315/(64 pi h^9)
    float cP;          // m * 45/(pi h^6)
    float cV;          // mu * m * 45/(pi h^6)
    float inv_rho0;
    float B;
    float attr;        // attractive-pressure ratio (0 when off)
    float e;           // restitution
    float dt;
    float g[3];
    int   attractive;
    uint32_t p_begin;  // particle range of this scene (state and sorted order)
    uint32_t p_end;
    float mu;
    float inv_csx;     // x cells are cs/xsub wide: xsub * inv_cs
    float xsubf;       // x cells per cs (1, 2 or 4)
    float hc2;         // (h * inv_cs)^2: the support radius squared in y/z cell units
    float wmargin;     // x-window safety margin in x cells
    float cfl;         // CFL number (0: fixed dt)
    float c0;          // sqrt(7 B / rho0), the EOS sound speed
    float dt_max;      // the parameter dt: the step, or its cap under CFL
    float rho0;        // rest density (the walls' half-space fluid)
    float inv_h;       // 1 / h
    float cW;          // 2 * 45 rho0 / h: the walls' pressure term
    float wmax[3];     // box_max (box_min is bmin)
    float scale_a;     // powers of two that the reverse pass keeps the acceleration's and the density's
    float unscale_a;   // adjoint by, and their inverses: the pairs' terms leave the constant factors of their
    float scale_r;     // sums out (up to 10^16), and so lie as far inside the float range as with them
    float unscale_r;
};
static_assert(sizeof(SceneConst) == 192, "SceneConst layout");

constexpr int kRows = 9;          // 3x3 (dz, dy) rows of three x-adjacent cells
constexpr int kMaskBits = 32;     // candidates per row tracked in the mask

__device__ __forceinline__ int cell_coord(float x, float bmin, float inv_cs, int G) {
    float f = (x - bmin) * inv_cs;
    f = fminf(fmaxf(f, 0.0f), (float)(G - 1));
    return (int)f;
}

__device__ __forceinline__ float dist2(float dx, float dy, float dz) {
    return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
}

// Workgroups go round-robin over the 8 XCDs; give each XCD one contiguous run
// of logical blocks so the neighbour data its blocks share stays in its L2.
__device__ __forceinline__ uint32_t xcd_block(uint32_t bid, uint32_t nblocks) {
    const uint32_t X = 8;
    const uint32_t q = nblocks / X, r = nblocks % X;
    const uint32_t x = bid % X, i = bid / X;
    return x * q + (x < r ? x : r) + i;
}

// A tile's (scene, first particle) and its scene's constants.  Tile and
// scene are the same for the whole block, and neither table is written
// while a pass runs, so both are read as constant memory: with a uniform
// index the loads are scalar and the constants sit in SGPRs, instead of
// per-lane loads that fences between LDS phases make the compiler repeat.
typedef __attribute__((address_space(4))) const uint32_t ConstWord;
__device__ __forceinline__ uint2 tile_at(const uint2* tiles, uint32_t t) {
    ConstWord* p = (ConstWord*)(tiles + t);
    return make_uint2(p[0], p[1]);
}
__device__ __forceinline__ SceneConst scene_at(const SceneConst* scenes, uint32_t s) {
    ConstWord* p = (ConstWord*)(scenes + s);
    SceneConst c;
    uint32_t* d = reinterpret_cast<uint32_t*>(&c);
#pragma unroll
    for (uint32_t i = 0; i < sizeof(SceneConst) / 4; ++i) d[i] = p[i];
    return c;
}

// Work over tiles.  A plain launch has one block per tile, in XCD-aware
// order.  A persistent launch (queue != null, gridDim >= 8) gives each XCD an
// equal contiguous share of the tiles; the XCD's blocks (blockIdx % 8) take
// tiles from that share through an atomic counter, so costly tiles do not
// hold up a fixed split.  The eight counters are zeroed before the launch.
template <class Body>
__device__ __forceinline__ void for_each_tile(uint32_t ntiles, uint32_t* __restrict__ queue, Body&& body) {
    if (!queue) {
        const uint32_t t = xcd_block(blockIdx.x, gridDim.x);
        if (t < ntiles) body(t);
        return;
    }
    __shared__ uint32_t s_next;
    const uint32_t x = blockIdx.x & 7u;
    const uint32_t t_beg = (uint32_t)(((uint64_t)ntiles * x) >> 3);
    const uint32_t t_end = (uint32_t)(((uint64_t)ntiles * (x + 1u)) >> 3);
    for (;;) {
        if (threadIdx.x == 0) s_next = t_beg + atomicAdd(queue + x, 1u);
        __syncthreads();
        const uint32_t t = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_next);  // the same in every lane
        __syncthreads();
        if (t >= t_end) break;
        body(t);
    }
}

// Neighbour rows.  Cells are cs = h(1 + 2^-10) in y and z and cs/xsub in x.
// The candidates of a particle lie in the 3x3 rows (dy, dz) of y/z cells
// around its own; within a row, only x cells inside the chord of the support
// sphere at that row's nearest y/z distance can hold neighbours.  A row's x
// cells are contiguous in sorted order, and cstart holds a lower bound for
// every cell (empty ones included), so a row is the single range
// [cstart[first x cell], cstart[last x cell + 1]).  The window is a superset
// of the neighbours (distances are under-estimated by 2^-10 cells and the
// chord is widened by wmargin); the predicate d^2 < h^2 decides membership.
struct RowGeom {
    float fx;            // x coordinate in x cells
    uint32_t row0;       // key of cell (x = 0, cy, cz)
    float qy[3], qz[3];  // squared y / z distance to rows -1, 0, +1 (cell units);
                         // 4 for a row outside the grid, which empties its window
};

__device__ __forceinline__ RowGeom row_geom(const SceneConst& sc, float x, float y, float z) {
    RowGeom g;
    g.fx = (x - sc.bmin[0]) * sc.inv_csx;
    const float fy = (y - sc.bmin[1]) * sc.inv_cs;
    const float fz = (z - sc.bmin[2]) * sc.inv_cs;
    const int cy = (int)fminf(fmaxf(fy, 0.0f), (float)(sc.G[1] - 1));
    const int cz = (int)fminf(fmaxf(fz, 0.0f), (float)(sc.G[2] - 1));
    const float m = 0.0009765625f;
    const float ry = fminf(fmaxf(fy - (float)cy, 0.0f), 1.0f);
    const float rz = fminf(fmaxf(fz - (float)cz, 0.0f), 1.0f);
    const float ly = fmaxf(ry - m, 0.0f), uy = fmaxf(1.0f - ry - m, 0.0f);
    const float lz = fmaxf(rz - m, 0.0f), uz = fmaxf(1.0f - rz - m, 0.0f);
    g.qy[0] = cy > 0 ? ly * ly : 4.0f;
    g.qy[1] = 0.0f;
    g.qy[2] = cy < sc.G[1] - 1 ? uy * uy : 4.0f;
    g.qz[0] = cz > 0 ? lz * lz : 4.0f;
    g.qz[1] = 0.0f;
    g.qz[2] = cz < sc.G[2] - 1 ? uz * uz : 4.0f;
    // A particle with a non-finite coordinate has no neighbours (every d^2
    // with it is NaN, which fails d^2 < h^2): all its windows are empty, so
    // a pile of such particles in one clamped cell costs nothing here.
    if (!(__builtin_isfinite(x) && __builtin_isfinite(y) && __builtin_isfinite(z))) {
#pragma unroll
        for (int i = 0; i < 3; ++i) g.qy[i] = g.qz[i] = 4.0f;
    }
    g.row0 = sc.cell_offset + ((uint32_t)cz * (uint32_t)sc.G[1] + (uint32_t)cy) * (uint32_t)sc.G[0];
    return g;
}

// Raw buffer resource over n elements of T: loads past the end return 0.
template <class T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const T* p, uint32_t n) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, (int)(n * (uint32_t)sizeof(T)), 0x00020000);
}

// Window [lo, hi) of the row whose cell (x = 0) is c, for a particle whose
// chord there has the squared half length w2; rcs is a buffer over cstart.
__device__ __forceinline__ void chord_window(__amdgpu_buffer_rsrc_t rcs, const SceneConst& sc, float fx, float w2,
                                             uint32_t c, uint32_t& lo, uint32_t& hi) {
    lo = 0u;
    hi = 0u;
    if (!(w2 > 0.0f)) return;
    const float wx = __builtin_amdgcn_sqrtf(w2) * sc.xsubf + sc.wmargin;
    const float gmax = (float)(sc.G[0] - 1);
    const uint32_t x0 = (uint32_t)(int)fminf(fmaxf(fx - wx, 0.0f), gmax);
    const uint32_t x1 = (uint32_t)(int)fminf(fmaxf(fx + wx, 0.0f), gmax);
    lo = __builtin_amdgcn_raw_buffer_load_b32(rcs, (int)((c + x0) << 2), 0, 0);
    hi = __builtin_amdgcn_raw_buffer_load_b32(rcs, (int)((c + x1 + 1u) << 2), 0, 0);
}

// Window of row (dy, dz).
__device__ __forceinline__ void row_window(__amdgpu_buffer_rsrc_t rcs, const SceneConst& sc, const RowGeom& g,
                                           int dy, int dz, uint32_t& lo, uint32_t& hi) {
    const float w2 = sc.hc2 - (g.qy[dy + 1] + g.qz[dz + 1]);
    chord_window(rcs, sc, g.fx, w2, g.row0 + (uint32_t)(dz * sc.G[1] + dy) * (uint32_t)sc.G[0], lo, hi);
}

// The window of one row (dy, dz) of a particle: row_geom and row_window for
// that row alone.
__device__ __forceinline__ void split_window(__amdgpu_buffer_rsrc_t rcs, const SceneConst& sc, const float4& p, int dy,
                                             int dz, uint32_t& lo, uint32_t& hi) {
    const float fx = (p.x - sc.bmin[0]) * sc.inv_csx;
    const float f[2] = {(p.y - sc.bmin[1]) * sc.inv_cs, (p.z - sc.bmin[2]) * sc.inv_cs};
    const int d[2] = {dy, dz};
    int c[2];
    float q[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        c[i] = (int)fminf(fmaxf(f[i], 0.0f), (float)(sc.G[i + 1] - 1));
        const float m = 0.0009765625f;
        const float r = fminf(fmaxf(f[i] - (float)c[i], 0.0f), 1.0f);
        const float near = fmaxf((d[i] < 0 ? r : 1.0f - r) - m, 0.0f);
        const bool in = d[i] < 0 ? c[i] > 0 : c[i] < sc.G[i + 1] - 1;
        q[i] = d[i] == 0 ? 0.0f : in ? near * near : 4.0f;
    }
    lo = hi = 0u;
    if (!(__builtin_isfinite(p.x) && __builtin_isfinite(p.y) && __builtin_isfinite(p.z))) return;
    const uint32_t row = ((uint32_t)(c[1] + dz) * (uint32_t)sc.G[1] + (uint32_t)(c[0] + dy)) * (uint32_t)sc.G[0];
    chord_window(rcs, sc, fx, sc.hc2 - (q[0] + q[1]), sc.cell_offset + row, lo, hi);
}

// Row masks.  The density pass tests a row's candidates [lo, hi) four at a
// time and shifts one bit per slot into the row's mask (slots past hi shift
// in zeros), so candidate c of a row with T groups sits at bit 4T-1-c and
// only the last 32 slots survive; the 32 slots before those go to a second
// word of the same form (mask_hi, written and read for rows of more than 32
// slots only, by handles with room for it).  Candidates before the words'
// are re-tested with the predicate.  row_neighbors visits a row's
// neighbours in ascending order: first the re-tested head, then the bits
// from the highest (the lowest candidate) down.
__device__ __forceinline__ uint32_t mask_span(uint32_t lo, uint32_t hi) { return (hi - lo + 3u) & ~3u; }

// Bit of candidate j of a row (>= 32 when j precedes the mask's slots).
__device__ __forceinline__ uint32_t mask_bit(uint32_t lo, uint32_t hi, uint32_t j) {
    return mask_span(lo, hi) - 1u - (j - lo);
}

template <class Retest, class F>
__device__ __forceinline__ void row_neighbors(uint32_t lo, uint32_t hi, uint32_t m, Retest&& retest, F&& f) {
    const uint32_t span = mask_span(lo, hi);
    const uint32_t jb = lo + span - 32u;  // candidate of bit 31 (wraps when span < 32)
    if (span > 32u)
        for (uint32_t j = lo; j < jb; ++j)
            if (retest(j)) f(j);
    // Bit 31 - i of m is candidate jb + i; reversed, the lowest set bit is
    // the next candidate in ascending order, and r & (r - 1) clears it.
    for (uint32_t r = __builtin_bitreverse32(m); r; r &= r - 1u) f(jb + (uint32_t)__builtin_ctz(r));
}

// The first candidate the mask covers: lo, or for a row of more than 32
// candidates the first of its last 32.
__device__ __forceinline__ uint32_t row_first(uint32_t lo, uint32_t hi) {
    const uint32_t span = mask_span(lo, hi);
    return span > 32u ? lo + span - 32u : lo;
}

// The same for `words` words together (the one before the mask holds the 32
// slots before the mask's).
__device__ __forceinline__ uint32_t row_first(uint32_t lo, uint32_t hi, uint32_t words) {
    const uint32_t span = mask_span(lo, hi), w = words * 32u;
    return span > w ? lo + span - w : lo;
}

// A word's slots as bits in ascending order of candidates: of the word whose
// last slot is `after` slots before the row's end, bit i is candidate
// row_first(lo, hi, 1 + after / 32) + i.
__device__ __forceinline__ uint32_t mask_ascending(uint32_t word, uint32_t span, uint32_t after) {
    uint32_t r = __builtin_bitreverse32(word);
    const uint32_t slots = span - after;
    if (slots - 1u < 31u) r >>= 32u - slots;
    return r;
}

// The centre row's mask word (its last slot `after` slots before the row's
// end) without particle k's own bit.
__device__ __forceinline__ uint32_t without_self(uint32_t word, uint32_t lo, uint32_t hi, uint32_t k, uint32_t after) {
    const uint32_t b = mask_bit(lo, hi, k) - after;
    return b < (uint32_t)kMaskBits ? word & ~(1u << b) : word;
}

// row_neighbors with the mask's visits given as offsets: g(i) for candidate
// row_first(lo, hi) + i (f(j) for the re-tested head, as before).  A caller
// reading the row from a staged copy then adds the row's offset once per
// row instead of once per neighbour.  Same neighbours, same order.
template <class Retest, class F, class G>
__device__ __forceinline__ void row_neighbors_from(uint32_t lo, uint32_t hi, uint32_t m, Retest&& retest, F&& f,
                                                   G&& g) {
    const uint32_t span = mask_span(lo, hi);
    const uint32_t j0 = row_first(lo, hi);
    for (uint32_t j = lo; j < j0; ++j)
        if (retest(j)) f(j);
    // Reversed, bit i is candidate lo + span - 32 + i; a row of fewer than
    // 32 slots drops the 32 - span empty low bits, so bit i is lo + i.
    uint32_t r = __builtin_bitreverse32(m);
    if (span - 1u < 31u) r >>= 32u - span;
    for (; r; r &= r - 1u) g((uint32_t)__builtin_ctz(r));
}

// Wave-wide minimum / maximum of one value per lane (all 64 lanes active):
// DPP within each row of 16 lanes, then row broadcasts fold row 0 into 1 and
// row 2 into 3 (lane 15 and 47 to the odd rows), then rows 0-1 into 2-3
// (lane 31 to rows 2 and 3), so lane 63 holds the result.  The operation's
// identity is the "old" operand: rows the row mask leaves out take it and
// keep their own value, and the compiler folds each move into the min / max
// as its DPP source.
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_min(uint32_t v) {
    return min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, CTRL, ROWS, 0xF, false));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_max(uint32_t v) {
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false));
}
__device__ __forceinline__ uint32_t wave_umin(uint32_t v) {
    v = dpp_min<0xB1, 0xF>(v);   // quad_perm 1,0,3,2
    v = dpp_min<0x4E, 0xF>(v);   // quad_perm 2,3,0,1
    v = dpp_min<0x141, 0xF>(v);  // row_half_mirror
    v = dpp_min<0x140, 0xF>(v);  // row_mirror
    v = dpp_min<0x142, 0xA>(v);  // row_bcast:15
    v = dpp_min<0x143, 0xC>(v);  // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
    v = dpp_max<0xB1, 0xF>(v);
    v = dpp_max<0x4E, 0xF>(v);
    v = dpp_max<0x141, 0xF>(v);
    v = dpp_max<0x140, 0xF>(v);
    v = dpp_max<0x142, 0xA>(v);
    v = dpp_max<0x143, 0xC>(v);
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Direct copy of 16 bytes at byte offset off of a buffer into LDS: lane i
// writes dst[i] (the wave's active lanes; dst is the same for all lanes).
// No registers hold the data; lds_copy_wait() waits for the wave's copies.
typedef __attribute__((address_space(3))) void lds_void;
__device__ __forceinline__ void lds_copy16(__amdgpu_buffer_rsrc_t r, float4* dst, uint32_t off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)dst, 16, (int)off, 0, 0, 0);
}
__device__ __forceinline__ void lds_copy_wait() {
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0); expcnt and lgkmcnt unconstrained
    __builtin_amdgcn_wave_barrier();
}

// LDS order between a wave's own stores and its later loads of other
// lanes' entries (and back).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Components go through named vector members: reading elements of the
// builtin's result by subscript inside __builtin_bit_cast loses all but one
// dword of the load with this compiler.
__device__ __forceinline__ float4 load4(__amdgpu_buffer_rsrc_t r, uint32_t byte_off) {
    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)byte_off, 0, 0);
    float4 f;
    f.x = __uint_as_float(v.x);
    f.y = __uint_as_float(v.y);
    f.z = __uint_as_float(v.z);
    f.w = __uint_as_float(v.w);
    return f;
}

__device__ __forceinline__ uint32_t cell_key(const SceneConst& sc, float x, float y, float z) {
    const int cx = cell_coord(x, sc.bmin[0], sc.inv_csx, sc.G[0]);
    const int cy = cell_coord(y, sc.bmin[1], sc.inv_cs, sc.G[1]);
    const int cz = cell_coord(z, sc.bmin[2], sc.inv_cs, sc.G[2]);
    return sc.cell_offset + ((uint32_t)cz * (uint32_t)sc.G[1] + (uint32_t)cy) * (uint32_t)sc.G[0] + (uint32_t)cx;
}

// Cells per tile of the sort, as a shift: the integrate pass also sums
// particles per tile, so every sort block finds its prefix without waiting.
// A tile's block moves its particles alone, so small grids take small tiles:
// a fluid settled over the floor of a 500k-cell grid fills 50 tiles of 1024
// cells, up to 1,700 particles each (49k particles: sort 10.9 us, 9.8 with
// tiles of 512, 9.2 with 256; DoubleDambreak at resolution 24, 55k cells:
// frame 8.06 ms, 7.76 with 256).  Above 2^20 cells more tiles cost
// more in the sums each block adds up than their balance gives.
// Cells that hold more than the usual few particles each (a support radius of
// more than four particle radii; `members`: of a cell of fluid at rest) come
// in tiles of fewer, down to four, so that a full tile holds about 2,048
// particles, as long as there are no more tiles than a 64th of the particles:
// with 54 and 250 particles a cell (216,000 particles, support 12 and 20
// radii) tiles of 256 cells left 16 to 76 blocks to move them, sort 230 and
// 2,935 us; with fewer cells, and runs ranked instead of members, 17.6 and 28.
constexpr uint32_t kTileShiftMax = 10;
constexpr uint32_t kTileShiftMin = 2;
constexpr uint32_t tile_shift_for(uint32_t ncells) {
    return ncells <= (1u << 19) ? 8u : ncells <= (1u << 20) ? 9u : kTileShiftMax;
}
constexpr uint32_t tile_shift_for(uint32_t ncells, uint32_t n, float members) {
    uint32_t shift = tile_shift_for(ncells);
    if (members > 8.0f)
        while (shift > kTileShiftMin && members * (float)(1u << shift) > 2048.0f && ncells >> (shift - 1u) <= n / 64u)
            --shift;
    return shift;
}
__host__ __device__ constexpr uint32_t scan_tiles(uint32_t ncells, uint32_t shift) {
    return (ncells + (1u << shift) - 1u) >> shift;
}

// Runs.  A cell's members are kept as a chain of runs: consecutive particles
// of one wave with the same key, at most 15 of them so that a run packs into
// one word (first particle in 28 bits, length in 4; 0 is the chain's end).
// Lanes follow the last sorted order, so a cell mostly has one or two runs.
constexpr uint32_t kRunMax = 15;
constexpr uint32_t kRunMask = (1u << 28) - 1u;
__device__ __forceinline__ uint32_t run_first(uint32_t r) { return r & kRunMask; }
__device__ __forceinline__ uint32_t run_len(uint32_t r) { return r >> 28; }

// Lane masks of the wave's runs of equal v (active lanes only).  first: this
// lane starts one; end: the lane after the last of this lane's run.
struct LaneRun {
    bool first;
    int leader, end;
};
__device__ __forceinline__ LaneRun lane_run(uint32_t v, bool active) {
    const int lane = (int)(threadIdx.x & 63u);
    const uint32_t kk = active ? v : 0xffffffffu;
    // The lane below's value (DPP wave_shr:1).
    const uint32_t prev = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)kk, 0x138, 0xF, 0xF, false);
    LaneRun r;
    r.first = active && (lane == 0 || prev != kk);
    const uint64_t starts = __ballot(r.first);
    const uint64_t act = __ballot(active);
    const uint64_t upto = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
    const uint64_t le = starts & upto;
    r.leader = le ? 63 - __clzll(le) : lane;
    const uint64_t above = (starts | ~act) & ~upto;
    r.end = above ? __ffsll((long long)above) - 1 : 64;
    return r;
}

// Links particle k (lanes hold consecutive particles) into its cell's chain,
// one exchange per run.  All lanes of the wave must call it; `active` marks
// the lanes that hold a particle.
__device__ __forceinline__ void push_run(uint32_t* __restrict__ head, uint32_t* __restrict__ next, uint32_t key,
                                         uint32_t k, bool active) {
    const int lane = (int)(threadIdx.x & 63u);
    const LaneRun r = lane_run(key, active);
    // A run's lanes 0, 15, 30, 45 and 60 each start a link.
    const uint64_t links = 0x1000200040008001ull;
    if (active && ((links >> (lane - r.leader)) & 1ull)) {
        const int len = min(r.end - lane, (int)kRunMax);
        next[k] = atomicExch(head + key, k | ((uint32_t)len << 28));
    }
}

// Adds the wave's particles to their tiles' sums: one atomic per run of
// lanes in one tile, or one in all where the wave has a single tile.
__device__ __forceinline__ void add_tile_sums(uint32_t* __restrict__ tsum, uint32_t shift, uint32_t key,
                                              bool active) {
    const uint32_t lane = threadIdx.x & 63u, tile = key >> shift;
    const uint64_t act = __ballot(active);
    if (act == 0u) return;
    const uint32_t first = (uint32_t)__builtin_ctzll(act);
    const uint32_t one = (uint32_t)__builtin_amdgcn_readlane((int)tile, (int)first);
    if (__ballot(active && tile != one) == 0u) {
        if (lane == first) atomicAdd(tsum + one, (uint32_t)__popcll(act));
        return;
    }
    const LaneRun r = lane_run(tile, active);
    if (r.first) atomicAdd(tsum + tile, (uint32_t)(r.end - (int)lane));
}

// |v|^2 for the CFL step; NaN counts as 0.
__device__ __forceinline__ float speed2(float vx, float vy, float vz) {
    return fmaxf(fmaf(vz, vz, fmaf(vy, vy, vx * vx)), 0.0f);
}

// Adds the wave's largest |v|^2 to one of kSpeedSlots words (float bits;
// integer maxima of the bit patterns order non-negative floats), picked by
// block: on one word the waves' atomics queue (414 of them: force pass 10.1
// against 8.4 us).  All lanes of the wave must call it, lanes without a
// particle with 0.
constexpr uint32_t kSpeedSlots = 64;
__device__ __forceinline__ void wave_max_v2(uint32_t* __restrict__ slots, float v2) {
    const uint32_t m = wave_umax(__float_as_uint(v2));
    if ((threadIdx.x & 63u) == 0u) atomicMax(slots + blockIdx.x % kSpeedSlots, m);
}

// Walls.  Each box face bounds a half-space of fluid at rest density; a
// particle at distance u h (u < 1) from a face gets that fluid's poly6
// density rho0 wall_rho(u) and its spiky pressure term, taken at the
// particle's own p/rho^2, cW (p/rho^2) wall_j(u) along the face's inward
// normal:
//   wall_rho(u) = (1-u)^5 (128 + 325u + 345u^2 + 175u^3 + 35u^4) / 256
//               = (315/256) int_u^1 (1 - t^2)^4 dt          (rho0/2 at u = 0)
//   wall_j(u)   = (1-u)^4 (1 + 4u) / 30 = int_u^1 (1-s)^2 (s^2 - u^2) ds
// with the derivatives the reverse pass needs.
__device__ __forceinline__ float wall_rho(float u) {
    if (!(u < 1.0f)) return 0.0f;
    u = fmaxf(u, 0.0f);
    const float w = 1.0f - u;
    const float w2 = w * w;
    const float w5 = (w2 * w2) * w;
    const float poly = 128.0f + u * (325.0f + u * (345.0f + u * (175.0f + u * 35.0f)));
    return (w5 * poly) * 0.00390625f;
}
__device__ __forceinline__ float wall_j(float u) {
    if (!(u < 1.0f)) return 0.0f;
    u = fmaxf(u, 0.0f);
    const float w = 1.0f - u;
    const float w2 = w * w;
    return ((w2 * w2) * (1.0f + 4.0f * u)) * (float)(1.0 / 30.0);
}
__device__ __forceinline__ float wall_rho_du(float u) {
    if (!(u < 1.0f)) return 0.0f;
    u = fmaxf(u, 0.0f);
    const float s = 1.0f - u * u;
    const float s2 = s * s;
    return -1.23046875f * (s2 * s2);
}
__device__ __forceinline__ float wall_j_du(float u) {
    if (!(u < 1.0f)) return 0.0f;
    u = fmaxf(u, 0.0f);
    const float w = 1.0f - u;
    return -(float)(2.0 / 3.0) * u * ((w * w) * w);
}

// Tait EOS, exponent 7 by the chain x^2, x^4, (x^4 x^2) x; p < 0 is clamped
// to 0 or scaled by the attractive ratio.
__device__ __forceinline__ float eos(const SceneConst& sc, float rho) {
    const float x = rho * sc.inv_rho0;
    const float x2 = x * x;
    const float x4 = x2 * x2;
    const float x7 = (x4 * x2) * x;
    float p = sc.B * (x7 - 1.0f);
    if (p < 0.0f) p = sc.attractive ? p * sc.attr : 0.0f;
    return p;
}

}  // namespace sph
