// One SPH step on caller-owned device arrays that allocates nothing: the
// intermediates of the step (sorted state, cell tables, neighbour masks,
// tile table, scene constants) live in one file-scope device array,
// `scratch`, of fixed size.  No counterpart in the reference: it is for
// callers that cannot allocate device memory, such as code under HIP graph
// capture or a serving loop that runs one fluid step per request.
//
// The step is the one sph_advance_steps runs as the first step after
// sph_set_particles (hash, cell-count sort, density, force), with the same
// kernels, form and grid rule, so its results equal that entry point's bit for
// bit.
//
// Limits: at most kMaxParticles particles and kMaxCells grid cells (the
// largest x subdivision of 4, 2, 1 whose grid fits is used, as a handle of
// that size would pick).  Every call on one GPU shares that GPU's scratch:
// calls that overlap on one GPU race, and each call rewrites the scratch
// from the start (chain heads, tile prefixes and the error word are cleared by
// a kernel, not by memset, so the call may be graph-captured).
#include <cstring>
#include <mutex>

#include "sph_engine.hpp"

namespace sph {

namespace {

constexpr uint32_t kMaxParticles = 65536;
constexpr uint32_t kMaxCells = 1u << 20;
constexpr uint32_t kMaxTiles = kMaxParticles / kSplitTile;
constexpr uint32_t kScanTilesMax = 2048;
static_assert(scan_tiles(kMaxCells, tile_shift_for(kMaxCells)) <= kScanTilesMax &&
                  scan_tiles(1u << 19, tile_shift_for(1u << 19)) <= kScanTilesMax && kMaxParticles / 64 < kScanTilesMax,
              "the most tiles of each tile size");

// Byte offsets of the arrays inside the scratch, each 256-byte aligned.
constexpr size_t align256(size_t x) { return (x + 255u) & ~(size_t)255u; }
struct Layout {
    static constexpr size_t N = kMaxParticles;
    static constexpr size_t pos = 0;
    static constexpr size_t vel = align256(pos + 16 * N);
    static constexpr size_t pos_s = align256(vel + 16 * N);
    static constexpr size_t vel_s = align256(pos_s + 16 * N);
    static constexpr size_t id = align256(vel_s + 16 * N);
    static constexpr size_t id_s = align256(id + 4 * N);
    static constexpr size_t key0 = align256(id_s + 4 * N);
    static constexpr size_t next = align256(key0 + 4 * N);
    static constexpr size_t tmp = align256(next + 4 * N);
    static constexpr size_t perm = align256(tmp + 4 * N);
    static constexpr size_t nlist = align256(perm + 4 * N);
    // The gathered form's planes and second mask words, in the lists' room.
    static constexpr size_t soa = nlist;
    static constexpr size_t mask_hi = align256(soa + 12 * N);
    static_assert(mask_hi + 4 * (size_t)kRows * N <= nlist + 2 * (size_t)kListMax * N, "they fit there");
    static constexpr size_t ncount = align256(nlist + 2 * (size_t)kListMax * N);
    static constexpr size_t rho = align256(ncount + 4 * N);
    static constexpr size_t mask = align256(rho + 4 * N);
    static constexpr size_t head = align256(mask + 4 * (size_t)kRows * N);
    static constexpr size_t cstart = align256(head + 4 * ((size_t)kMaxCells + 2 * kScanTilesMax) + 16);
    static constexpr size_t tile_pre = align256(cstart + 4 * ((size_t)kMaxCells + 1));
    static constexpr size_t tiles = align256(tile_pre + 4 * (size_t)kScanTilesMax);
    static constexpr size_t scene = align256(tiles + 8 * (size_t)kMaxTiles);
    static constexpr size_t err = align256(scene + sizeof(SceneConst));
    static constexpr size_t total = align256(err + 4);
};

// The step's scratch on each GPU the library runs on (about 32 MB), held
// until the process ends.  Host code reaches it only through the address
// hipGetSymbolAddress returns on that device.
static __device__ __align__(256) uint8_t scratch[Layout::total];

constexpr int kMaxDevices = 64;
std::mutex g_mu;
void* g_scratch[kMaxDevices] = {};

// Scene constants, the tile table (scene 0, first particle t * kSplitTile, in
// every form: a wave's tiles spread over more CUs than larger ones), empty
// chains, tile sums and tile prefixes, and the error word cleared.
__global__ void noalloc_setup_kernel(SceneConst sc, uint32_t ncells, uint32_t tile_shift, uint8_t* __restrict__ base) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
    if (i == 0) {
        *reinterpret_cast<SceneConst*>(base + Layout::scene) = sc;
        *reinterpret_cast<uint32_t*>(base + Layout::err) = 0u;
    }
    const uint32_t T = scan_tiles(ncells, tile_shift);
    uint32_t* head = reinterpret_cast<uint32_t*>(base + Layout::head);
    // Whole 16-byte words; the scratch behind the last tile sum is unused.
    for (uint32_t w = i; w < (ncells + 2u * T + 3u) / 4u; w += stride)
        reinterpret_cast<uint4*>(head)[w] = make_uint4(0u, 0u, 0u, 0u);
    uint32_t* tile_pre = reinterpret_cast<uint32_t*>(base + Layout::tile_pre);
    for (uint32_t t = i; t < T; t += stride) tile_pre[t] = 0xffffffffu;
    uint2* tiles = reinterpret_cast<uint2*>(base + Layout::tiles);
    for (uint32_t t = i; t * kSplitTile < sc.p_end; t += stride) tiles[t] = make_uint2(0u, t * kSplitTile);
}

// The scratch address on the current device, looked up once per device.
hipError_t scratch_ptr(uint8_t** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_mu);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch[dev] = p;
    }
    *out = static_cast<uint8_t*>(g_scratch[dev]);
    return hipSuccess;
}

int fail_noalloc(int code, const char* msg) {
    set_thread_error(msg);
    return code;
}

}  // namespace

}  // namespace sph

using namespace sph;

extern "C" int sph_step_noalloc(const sph_params* p, const float* xyz_in, const float* vel_in, float* xyz_out,
                                float* vel_out, uint32_t n, void* stream) {
    if (!p || !xyz_in || !xyz_out || !vel_out) return fail_noalloc(SPH_E_INVALID, "sph_step_noalloc: null argument");
    if (n == 0 || n > kMaxParticles)
        return fail_noalloc(SPH_E_INVALID, "sph_step_noalloc: n must be 1 .. 65536 (the scratch's particle limit)");
    if (p->cfl_number != 0.0f) return fail_noalloc(SPH_E_INVALID, "sph_step_noalloc: fixed dt only (cfl_number = 0)");
    // The grid a handle of n <= 65536 particles picks: the largest x
    // subdivision whose cell count stays within 2^20.
    SceneConst sc;
    int rc = SPH_E_INVALID, sub = 1;
    for (int xsub : {4, 2, 1}) {
        rc = derive_scene_noalloc(*p, sc, xsub);
        if (rc != SPH_OK) return fail_noalloc(rc, "sph_step_noalloc: invalid parameters (as sph_create checks them)");
        if ((uint64_t)sc.G[0] * sc.G[1] * sc.G[2] <= kMaxCells) {
            sub = xsub;
            break;
        }
        rc = SPH_E_CAPACITY;
    }
    if (rc != SPH_OK)
        return fail_noalloc(SPH_E_INVALID, "sph_step_noalloc: the grid exceeds 2^20 cells (the scratch's cell limit)");
    const uint32_t C = (uint32_t)((uint64_t)sc.G[0] * sc.G[1] * sc.G[2]);
    const uint32_t shift = tile_shift_for(C, n, cell_members(*p, sub));
    sc.cell_offset = 0;
    sc.p_begin = 0;
    sc.p_end = n;
    uint8_t* base = nullptr;
    hipError_t e = scratch_ptr(&base);
    if (e != hipSuccess) return fail_noalloc(SPH_E_HIP, "sph_step_noalloc: no scratch address on this device");
    hipStream_t st = static_cast<hipStream_t>(stream);
    auto at = [&](size_t off) { return base + off; };
    float4* pos = reinterpret_cast<float4*>(at(Layout::pos));
    float4* vel = reinterpret_cast<float4*>(at(Layout::vel));
    uint32_t* id = reinterpret_cast<uint32_t*>(at(Layout::id));
    uint32_t* head = reinterpret_cast<uint32_t*>(at(Layout::head));
    uint32_t* key0 = reinterpret_cast<uint32_t*>(at(Layout::key0));
    uint32_t* next = reinterpret_cast<uint32_t*>(at(Layout::next));
    const SceneConst* scd = reinterpret_cast<const SceneConst*>(at(Layout::scene));

    // The form a handle of so many particles and such rows takes.
    const bool split = (n + kSplitTile - 1) / kSplitTile <= kSplitTiles && !(cell_members(*p, 1) > kWideRows);
    // Five launches: setup, upload and hash, sort, density, force (which
    // writes the caller's arrays itself).
    hipLaunchKernelGGL(noalloc_setup_kernel, dim3(256), dim3(256), 0, st, sc, C, shift, base);
    e = hipGetLastError();
    if (e == hipSuccess) e = launch_upload_hash(st, xyz_in, vel_in, pos, vel, id, key0, next, head, n, C, shift, sc);
    SortPlan sp;
    sp.n = n;
    sp.ncells = C;
    sp.tile_shift = shift;
    sp.mode = kSortCellCount;
    sp.key0 = key0;
    sp.head = head;
    sp.next = next;
    sp.cstart = reinterpret_cast<uint32_t*>(at(Layout::cstart));
    sp.tile_pre = reinterpret_cast<uint32_t*>(at(Layout::tile_pre));
    sp.tmp = reinterpret_cast<uint32_t*>(at(Layout::tmp));
    sp.perm = reinterpret_cast<uint32_t*>(at(Layout::perm));
    sp.err = reinterpret_cast<uint32_t*>(at(Layout::err));
    sp.pos_in = pos;
    sp.vel_in = vel;
    sp.id_in = id;
    sp.pos_out = reinterpret_cast<float4*>(at(Layout::pos_s));
    sp.vel_out = reinterpret_cast<float4*>(at(Layout::vel_s));
    sp.id_out = reinterpret_cast<uint32_t*>(at(Layout::id_s));
    if (!split) sp.soa_out = reinterpret_cast<float*>(at(Layout::soa));
    if (e == hipSuccess) e = launch_sort_keys(st, sp);
    StepArgs a;
    std::memset(&a, 0, sizeof(a));
    a.pos_s = sp.pos_out;
    a.vel_s = sp.vel_out;
    a.id_s = sp.id_out;
    a.xyz_out = xyz_out;
    a.vel_out = vel_out;
    a.cstart = sp.cstart;
    a.rho = reinterpret_cast<float*>(at(Layout::rho));
    a.mask = reinterpret_cast<uint32_t*>(at(Layout::mask));
    if (split) {
        a.nlist = reinterpret_cast<uint16_t*>(at(Layout::nlist));
        a.ncount = reinterpret_cast<uint32_t*>(at(Layout::ncount));
    } else {
        a.soa = sp.soa_out;
        a.mask_hi = reinterpret_cast<uint32_t*>(at(Layout::mask_hi));
    }
    a.scenes = scd;
    a.tiles = reinterpret_cast<const uint2*>(at(Layout::tiles));
    a.ntiles = (n + kSplitTile - 1) / kSplitTile;
    a.n = n;
    a.ncells = C;
    if (e == hipSuccess) e = split ? launch_density_split(st, a) : launch_density(st, kSplitTile, a.ntiles, a);
    if (e == hipSuccess) e = split ? launch_force_split(st, a) : launch_force(st, kSplitTile, a.ntiles, a);
    if (e != hipSuccess) return fail_noalloc(SPH_E_HIP, "sph_step_noalloc: kernel launch failed");
    return SPH_OK;
}
