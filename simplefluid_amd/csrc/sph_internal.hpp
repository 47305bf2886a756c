// Host-side declarations shared by the engine's translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sph_device.hpp"

namespace sph {

constexpr int kMaxPasses = 4;   // 8-bit digits, keys up to 32 bits

constexpr int kSortCellCount = 0;   // one-digit (counting) radix sort, default
constexpr int kSortRadix = 1;       // multi-pass 8-bit LSD radix sort

struct SortPlan {
    uint32_t n = 0;
    uint32_t ncells = 0;
    uint32_t tile_shift = 0;          // cells per tile, as a shift
    int mode = kSortCellCount;
    int passes = 1;                   // radix: 8-bit digits
    int items = 8;                    // radix: keys per thread of a digit-pass tile
    int reorder_block = 256;
    const uint32_t* key0 = nullptr;   // unsorted keys (state order)
    uint32_t* head = nullptr;         // C chain heads (cleared by the sort), T tile sums and the sort's room
    const uint32_t* next = nullptr;   // per run, the cell's run before it
    uint32_t* cstart = nullptr;       // C + 1, written by the sort
    uint32_t* tile_pre = nullptr;     // per tile: the prefix this cstart holds in all its cells
                                      // when the tile was empty at its last write, else 0xffffffff
    uint32_t* tmp = nullptr;          // cell-count: runs or members of a tile on their way to their order (n)
    uint32_t* kbuf[2] = {nullptr, nullptr};  // radix ping-pong
    uint32_t* vbuf[2] = {nullptr, nullptr};
    uint32_t* skey = nullptr;         // radix: sorted keys
    uint32_t* perm = nullptr;         // sorted index -> state index
    uint32_t* hist = nullptr;         // radix: kMaxPasses x 256, zero on entry
    uint32_t* status = nullptr;       // radix: passes x tiles x 256
    uint32_t* tickets = nullptr;      // radix: kMaxPasses
    uint32_t* err = nullptr;
    uint32_t* queue = nullptr;        // kQueueWords tile counters, zeroed by the sort
    uint32_t* frame = nullptr;        // device frame loop's state (cell-count mode), else null
    const float4* pos_in = nullptr;
    const float4* vel_in = nullptr;
    const uint32_t* id_in = nullptr;
    float4* pos_out = nullptr;
    float* soa_out = nullptr;         // sorted x, y, z planes (3 N floats) for the gathered density
                                      // pass; null when the density pass is staged (it reads pos_out)
    float4* vel_out = nullptr;
    uint32_t* id_out = nullptr;
};

uint32_t sort_tiles(uint32_t n, int items);
// head holds C chain heads, then T = scan_tiles(C, tile_shift) per-tile sums, the
// length of the list of tiles that need work, the sums' exclusive scan and
// that list (T words each; both only where there are more tiles than a block
// sums itself).
inline size_t sort_head_words(uint32_t ncells, uint32_t shift) {
    return (size_t)ncells + 3 * (size_t)scan_tiles(ncells, shift) + 1;
}
int sort_key_passes(uint32_t ncells);
// Cell-start table and the sort; cell-count mode gathers the state too ...
hipError_t launch_sort_keys(hipStream_t st, const SortPlan& sp);
// ... radix mode: the gather of the state into sorted order.
hipError_t launch_sort_gather(hipStream_t st, const SortPlan& sp);

// Arguments of the per-particle passes.  Work is split in tiles of blockDim
// particles that never straddle two scenes (tiles[t] = (scene, first)).
struct StepArgs {
    float4* pos_s;           // sorted positions; w <- p/rho^2 (density pass)
    const float* soa;        // the same positions as x, y, z planes (3 N floats)
    float4* vel_s;           // sorted velocities; w <- 1/rho (density pass)
    float4* pos_o;           // state out (integrate), or null with xyz_out
    float4* vel_o;
    const uint32_t* id_s;
    uint32_t* id_o;
    uint32_t* key0;          // next step's unsorted keys
    uint32_t* head;          // next step's chain heads, then per-tile sums (atomic); null: no next step
    uint32_t* next;          // next step's runs
    const uint32_t* cstart;  // cell-start table of this step
    float* rho;
    uint32_t* mask;
    uint32_t* mask_hi;       // the 32 slots before mask's, rows of more than 32 slots; or null
    uint16_t* nlist;         // split form: neighbour lists, else null
    uint32_t* ncount;        // split form: their lengths
    float* xyz_out;          // state out in original order too (3 n floats each), or null
    float* vel_out;
    float4* acc;             // optional: acceleration (sorted order)
    const SceneConst* scenes;
    const uint2* tiles;
    uint32_t ntiles;
    // One word for both: with a register more to hold, the staged force pass
    // fetched its buffer descriptors back from vector lanes in its walk over
    // global memory (216,000 particles, rows of 200 candidates: 257 -> 278 us).
    uint32_t n : 28;         // below 2^28
    uint32_t tile_shift : 4; // cells per tile of the sort, as a shift
    uint32_t ncells;
    uint32_t* queue;         // persistent launch: 8 tile counters (zeroed by the sort), else null
    uint32_t* vmax2;         // CFL: kSpeedSlots words of max |v|^2 (float bits) of the state the step starts
                             // from (density), of the new state (force), else null
    SceneConst* cfl_scene;   // CFL: receives the scene (one) with the dt that the density pass finds from vmax2,
                             // for the force pass to read, else null
    float* dt_out;           // CFL: receives that dt
    uint32_t* frame;         // device frame loop's state, else null
};

// Tile counters of the persistent density and force launches (8 each),
// zeroed by the sort of every step.
constexpr int kQueueWords = 16;

hipError_t launch_hash(hipStream_t st, int block, uint32_t grid, const float4* pos, const float4* vel,
                       uint32_t* key0, uint32_t* next, uint32_t* head, uint32_t ncells, uint32_t tile_shift,
                       uint32_t* vmax2, const SceneConst* scenes, const uint2* tiles, uint32_t ntiles);
// Upload and hash of one scene in one pass (vel_in null: zero velocity).
hipError_t launch_upload_hash(hipStream_t st, const float* xyz, const float* vel_in, float4* pos, float4* vel,
                              uint32_t* id, uint32_t* key0, uint32_t* next, uint32_t* head, uint32_t n,
                              uint32_t ncells, uint32_t tile_shift, const SceneConst& sc);
// Device frame loop state, 4 words: halt (steps are skipped), pending (the
// frame reached 1/30 s in the current step), steps taken, frame time (float
// bits).  reset zeroes them; the density pass adds its step and sets pending,
// so the step that completes the frame runs to its end, and the next step's
// sort turns pending into halt.
constexpr int kFrameWords = 4;
hipError_t launch_frame_reset(hipStream_t st, uint32_t* frame);
// staged: the density pass reads each row's candidates from LDS (same results).
hipError_t launch_density(hipStream_t st, int block, uint32_t grid, const StepArgs& a, int staged = 0);
// staged: the force pass reads each row's candidates from LDS (same results).
hipError_t launch_force(hipStream_t st, int block, uint32_t grid, const StepArgs& a, int staged = 0);
// The split form of both passes, for at most kSplitMax particles: tiles of 64
// particles, a block of nine waves (density) or four (force) each; the
// density pass leaves every particle's neighbours as a list of kListMax
// indices for the force pass (a particle with more is walked by its masks).
// Same results as the other forms, bit for bit.
constexpr uint32_t kSplitMax = 65536;   // the lists hold 16-bit indices
constexpr uint32_t kListMax = 128;
constexpr int kSplitTile = 64;
constexpr uint32_t kListOver = 0xffffu;  // the length of a list that is too long
constexpr uint32_t kRowOver = 255u;      // the count of a row longer than two mask words
static_assert(kRowOver > kListMax + 1u, "such a row's particle is over its list's length too");
// Tiles up to which handles take it.  Two force blocks fit a CU, so 512 tiles
// run at once; from there on the chip is full and its extra work shows.
// Measured per step, the split form against the best of the others: 512
// particles 17.9 against 30.2 us, 4,096 18.0 against 27.8, 23,520 21.7 against
// 31.9, 32,768 (512 tiles) 22.6 against 30.6, 40,960 (640) 31.0 against 31.8,
// 49,152 (768) 32.5 against 32.5, 57,800 39.0 against 34.3.
constexpr uint32_t kSplitTiles = 640;
static_assert(kSplitTiles * kSplitTile <= kSplitMax, "every handle of so many tiles has 16-bit indices");
hipError_t launch_density_split(hipStream_t st, const StepArgs& a);
hipError_t launch_force_split(hipStream_t st, const StepArgs& a);
// Resident blocks per CU of the force kernel at this block size and form
// (the runtime's occupancy figure; 0 if it cannot say).
int force_blocks_per_cu(int block, int staged);
hipError_t launch_fill_u32(hipStream_t st, uint32_t* p, uint32_t value, size_t count);
// Debug: neighbour CSR as the force pass sees it.
hipError_t launch_neighbors(hipStream_t st, int block, uint32_t grid, const StepArgs& a,
                            const uint32_t* offsets, uint32_t* counts_or_list, int fill);
// Debug: keys of the sorted positions.
hipError_t launch_sorted_keys(hipStream_t st, int block, uint32_t ntiles, const float4* pos_s, uint32_t* skey,
                              const SceneConst* scenes, const uint2* tiles);
// Original-order gather for get_*: out[3*id[k]+c] = src[k].c
hipError_t launch_unpermute3(hipStream_t st, uint32_t n, const float4* src, const uint32_t* id,
                             float* out);
// Copies words of device memory and, behind them, *flag to dst (page-locked
// host memory).
hipError_t launch_copy_out(hipStream_t st, const uint32_t* src, size_t words, const uint32_t* flag, uint32_t* dst);
// x, y, z of src4, or src1 where that is null, in original order, then *flag, to
// dst (page-locked host memory), for at most kReadSmall particles: one block,
// which puts them in order in LDS (40 KB, and from there on one CU's writes
// over the bus take longer than the launch they save).
constexpr uint32_t kReadSmall = 3400;
hipError_t launch_read_small(hipStream_t st, uint32_t n, const float4* src4, const float* src1, const uint32_t* id,
                             const uint32_t* flag, float* dst);
hipError_t launch_unpermute1(hipStream_t st, uint32_t n, const float* src, const uint32_t* id,
                             float* out);
// Copies a state: n positions, velocities and ids.
hipError_t launch_copy_state(hipStream_t st, uint32_t n, float4* dp, float4* dv, uint32_t* di, const float4* sp,
                             const float4* sv, const uint32_t* si);
// dst[k] = (src[3k], src[3k+1], src[3k+2], 0), or zero when src is null.
hipError_t launch_pack3(hipStream_t st, uint32_t n, const float* src, float4* dst);

// Reverse pass of one step over a taped step (sorted order of that step).
struct AdjArgs {
    const float4* pos_s;
    const float4* vel_s;
    const float4* acc;
    const float* rho;
    const uint32_t* mask;
    const uint32_t* cstart;
    const uint32_t* perm;
    const float4* pos_p;     // the same of the step before, whose integration the density pass reverses too,
    const float4* vel_p;     // or null
    const float4* acc_p;
    float4* xbar;            // adjoint: of the step's output (integrate), then of its sorted state (force,
    float4* vbar;            // density)
    float4* xbar_o;          // integrate: of the step's sorted state; density: of its input, or of the sorted
    float4* vbar_o;          // state of the step before
    float4* abar;
    float* rhobar;
    double2* tile_acc;       // per tile: running (dL/dB, dL/dmu) sums over the reverse steps
    // Split form: the particles' (dL/dB, dL/dmu) terms of the step, which the
    // density pass adds up in tiles of 256, each scene's first one, and the
    // neighbour lists (force to density) and their lengths.
    double2* part;
    const uint32_t* tile_first;
    uint16_t* nlist;
    uint32_t* ncount;
    const SceneConst* scenes;
    const uint2* tiles;
    uint32_t ntiles;
    uint32_t n;
    uint32_t ncells;
};

hipError_t launch_adj_integrate(hipStream_t st, int block, uint32_t grid, const AdjArgs& a);
// staged: each row's candidates read from LDS (same results; whole waves only).
hipError_t launch_adj_force(hipStream_t st, int block, uint32_t grid, const AdjArgs& a, int staged = 0);
hipError_t launch_adj_density(hipStream_t st, int block, uint32_t grid, const AdjArgs& a, int staged = 0);
// The split form of both, over tiles of kSplitTile particles: same results.
hipError_t launch_adj_force_split(hipStream_t st, const AdjArgs& a);
hipError_t launch_adj_density_split(hipStream_t st, const AdjArgs& a);
// Per-scene totals of the tile accumulators in a fixed order: scene s sums
// tiles [tile_first[s], tile_first[s + 1]) into acc_a[s], acc_b[s].
hipError_t launch_scene_tile_sums(hipStream_t st, uint32_t nscenes, const uint32_t* tile_first,
                                  const double2* tile_acc, double* acc_a, double* acc_b);
// out[k] = (g[3 id[k]], g[3 id[k]+1], g[3 id[k]+2], 0)
hipError_t launch_gather3(hipStream_t st, uint32_t n, const float* g, const uint32_t* id, float4* out);

}  // namespace sph
