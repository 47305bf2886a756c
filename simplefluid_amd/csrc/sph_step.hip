// Per-particle passes of one SPH step on gfx950:
//   hash     cell key and chain links of every state position (first step
//            only; afterwards the integrate pass produces the next keys)
//   density  rho, EOS, neighbour bit masks (candidate tests happen here once)
//   force    pressure + viscosity from the masks, integrate, clamp, next key
// (sorting and the gather into sorted order live in sph_sort.hip).
// Neighbour order is canonical: rows (dz, dy) = (-1..1, -1..1), dz outer; a
// row is the contiguous sorted range of the x cells inside the support
// sphere's chord at that row; ascending index.  Density sums and force sums
// run in that order.  Density and force each come in three forms with the same
// results: candidates read from global memory ("gathered"), each row's
// candidates first copied by the wave into LDS ("staged"), both one particle
// per lane, or several waves to 64 particles ("split").
#include <atomic>
#include <cstddef>

#include "sph_internal.hpp"

namespace sph {

namespace {

// Tiles handled by this block (hash and the debug neighbour dump): a
// contiguous run per block when gridDim < ntiles, XCD-aware order.
__device__ __forceinline__ void tile_span(uint32_t ntiles, uint32_t& t0, uint32_t& t1) {
    const uint32_t lb = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t per = (ntiles + gridDim.x - 1) / gridDim.x;
    t0 = lb * per;
    t1 = t0 + per < ntiles ? t0 + per : ntiles;
}

// m = (m << 1) | (sign bit of c): one funnel shift (v_alignbit_b32).
__device__ __forceinline__ uint32_t push_sign(uint32_t m, float c) {
    return __builtin_amdgcn_alignbit(m, __float_as_uint(c), 31u);
}

// A trip pushes four bits into m; those it pushes out go on into mh, which so
// holds the 32 slots before m's at the row's end (one funnel shift a trip).
__device__ __forceinline__ uint32_t push_out(uint32_t mh, uint32_t m) {
    return __builtin_amdgcn_alignbit(mh, m, 28u);
}

// Candidates come from the x, y, z planes: one 16-byte load per plane gives
// four consecutive candidates (three loads per trip instead of four, which
// relieves the texture address units this pass otherwise saturates).
// Trips of four full candidates run without slot checks; the row's last,
// partial trip masks the slots past its end.
template <bool FULL>
__device__ __forceinline__ void density_trip(const float4& pi, float h2, const float4& X, const float4& Y,
                                             const float4& Z, int rem, float& sum, uint32_t& m, uint32_t& mh) {
    mh = push_out(mh, m);
    const float xs[4] = {X.x, X.y, X.z, X.w}, ys[4] = {Y.x, Y.y, Y.z, Y.w}, zs[4] = {Z.x, Z.y, Z.z, Z.w};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        // q = d2 - h2 is negative exactly when d2 < h2 (an exact tie rounds
        // to +0), and -q = h2 - d2 (rounding is symmetric) is the kernel's t;
        // slots past the row end get q = 1.  c = min(q, 0) is q where q < 0
        // and +0 elsewhere, a NaN q included (the minimum of a quiet NaN and
        // a number is the number): a NaN distance (a candidate with a
        // non-finite coordinate) may carry a set sign bit, and it is no
        // neighbour, as d2 < h2 says.  So c's sign bit is d2 < h2, and -c is
        // t = max(h2 - d2, 0): c * c * -c adds t^3, and -0 where t is 0.
        float q = dist2(pi.x - xs[u], pi.y - ys[u], pi.z - zs[u]) - h2;
        if (!FULL && u != 0 && u >= rem) q = 1.0f;
        const float c = fminf(q, 0.0f);
        sum = fmaf(c * c, -c, sum);
        m = push_sign(m, c);
    }
}

// Density, EOS and their stores from the neighbours' sum and the walls'.
__device__ __forceinline__ void density_finish(const StepArgs& a, const SceneConst& sc, uint32_t k, float sum,
                                               float wr) {
    const float rho = sc.cD * sum + sc.rho0 * wr;
    const float p = eos(sc, rho);
    const float ir = 1.0f / rho;
    a.rho[k] = rho;
    // p/rho^2 and 1/rho ride in the unused w of the sorted position and
    // velocity, so the force pass gets them with the same loads.  Neighbour
    // reads of pos_s in this pass take x, y, z only.
    reinterpret_cast<float*>(a.pos_s + k)[3] = (p * ir) * ir;
    reinterpret_cast<float*>(a.vel_s + k)[3] = ir;
}

__device__ __forceinline__ void density_one(const StepArgs& a, const SceneConst& sc, uint32_t k,
                                            __amdgpu_buffer_rsrc_t rpos, __amdgpu_buffer_rsrc_t rx,
                                            __amdgpu_buffer_rsrc_t ry, __amdgpu_buffer_rsrc_t rz,
                                            __amdgpu_buffer_rsrc_t rcs) {
    const float4 pi = load4(rpos, k << 4);
    const RowGeom g = row_geom(sc, pi.x, pi.y, pi.z);
    uint32_t lo[kRows], hi[kRows];
#pragma unroll
    for (int row = 0; row < kRows; ++row) row_window(rcs, sc, g, row % 3 - 1, row / 3 - 1, lo[row], hi[row]);
    const float h2 = sc.h2;
    float sum = 0.0f;
#pragma unroll
    for (int row = 0; row < kRows; ++row) {
        uint32_t m = 0u, mh = 0u;
        const uint32_t cnt = hi[row] - lo[row];
        uint32_t off = lo[row] << 2;
        const uint32_t full_end = (lo[row] + (cnt & ~3u)) << 2;
        // Slots past the row end shift in zero bits (past the array end the
        // buffer returns 0).  Each trip's planes are loaded while the trip
        // before is tested, so a lane has two trips' loads in flight.
        if (off != full_end) {
            float4 X = load4(rx, off), Y = load4(ry, off), Z = load4(rz, off);
            for (off += 16u; off != full_end; off += 16u) {
                const float4 Xn = load4(rx, off), Yn = load4(ry, off), Zn = load4(rz, off);
                density_trip<true>(pi, h2, X, Y, Z, 4, sum, m, mh);
                X = Xn;
                Y = Yn;
                Z = Zn;
            }
            density_trip<true>(pi, h2, X, Y, Z, 4, sum, m, mh);
        }
        const int rem = (int)(cnt & 3u);
        if (rem > 0) density_trip<false>(pi, h2, load4(rx, off), load4(ry, off), load4(rz, off), rem, sum, m, mh);
        if (cnt > 32u && a.mask_hi) a.mask_hi[(size_t)row * a.n + k] = mh;
        a.mask[(size_t)row * a.n + k] = m;
    }
    // The walls' half-space fluid, faces in the order x-, x+, y-, y+, z-, z+.
    float wr = 0.0f;
    const float pk[3] = {pi.x, pi.y, pi.z};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        wr += wall_rho((pk[d] - sc.bmin[d]) * sc.inv_h);
        wr += wall_rho((sc.wmax[d] - pk[d]) * sc.inv_h);
    }
    density_finish(a, sc, k, sum, wr);
}

// Candidates a wave stages per row in the density pass, plus the slots a
// row's last, partial trip reads past its end (masked out).  With 124
// floats per plane, a trip's reads of all three planes fit the 8-bit dword
// offsets of ds_read2_b32 from one address (z at 248..251).
constexpr uint32_t kStageD = 120;
static_assert(kSpeedSlots == 64, "a wave reads the speed slots");
static_assert(kStageD <= 128, "the copy into a slot takes two records per lane");
constexpr uint32_t kPlaneD = kStageD + 4;
struct DensitySlot {
    float v[3 * kPlaneD];  // the x plane, then y, then z
};

// Four consecutive slot entries of plane d (0 x, 1 y, 2 z) from the x
// plane's address of the first.
__device__ __forceinline__ float4 slot_quad(const float* p, int d) {
    const float* q = p + d * kPlaneD;
    return make_float4(q[0], q[1], q[2], q[3]);
}

// Four consecutive sorted positions as x, y, z quadruples (the gathered
// trip's planes, read from the position records instead).
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
__device__ __forceinline__ void load_quad(__amdgpu_buffer_rsrc_t rpos, uint32_t j, float4& X, float4& Y, float4& Z) {
    // x, y, z of each record (12-byte loads: the w lane is not needed).
    const u32x3 p0 = __builtin_amdgcn_raw_buffer_load_b96(rpos, (int)(j << 4), 0, 0);
    const u32x3 p1 = __builtin_amdgcn_raw_buffer_load_b96(rpos, (int)((j + 1u) << 4), 0, 0);
    const u32x3 p2 = __builtin_amdgcn_raw_buffer_load_b96(rpos, (int)((j + 2u) << 4), 0, 0);
    const u32x3 p3 = __builtin_amdgcn_raw_buffer_load_b96(rpos, (int)((j + 3u) << 4), 0, 0);
    X = make_float4(__uint_as_float(p0.x), __uint_as_float(p1.x), __uint_as_float(p2.x), __uint_as_float(p3.x));
    Y = make_float4(__uint_as_float(p0.y), __uint_as_float(p1.y), __uint_as_float(p2.y), __uint_as_float(p3.y));
    Z = make_float4(__uint_as_float(p0.z), __uint_as_float(p1.z), __uint_as_float(p2.z), __uint_as_float(p3.z));
}

// The sorted range the staged density pass copies for one row: the union of
// the wave's windows of that row.  A wave whose active lanes (a prefix of the
// wave) share one y/z column holds their x cells in ascending order, so every
// lane's window of a row lies in the row's x cells [cx0 - wmax, cx1 + 1 +
// wmax]: cx0 and cx1 the first and last lanes' cells, wmax above every
// lane's half chord in x cells.  Such a wave bounds each row's union by two
// scalar reads of the cell-start table (a superset of the exact union, copied
// whole) instead of a wave-wide minimum and maximum, which the other waves,
// and rows whose superset does not fit the slot, still take.
struct WaveColumn {
    bool one_col;
    uint32_t row0, x0c, x1c;
};

__device__ __forceinline__ WaveColumn wave_column(const SceneConst& sc, const RowGeom& g, bool active) {
    WaveColumn wc;
    const uint64_t act = __ballot(active);
    wc.row0 = __builtin_amdgcn_readfirstlane(g.row0);
    wc.one_col = act != 0u && __ballot(active && g.row0 != wc.row0) == 0u;
    wc.x0c = wc.x1c = 0u;
    if (wc.one_col) {
        const float gmax = (float)(sc.G[0] - 1);
        const int cx = (int)fminf(fmaxf(g.fx, 0.0f), gmax);
        const int cx0 = __builtin_amdgcn_readfirstlane(cx);
        const int cx1 = __builtin_amdgcn_readlane(cx, 63 - __builtin_clzll(act));
        // sqrt(hc2) bounds every lane's sqrt(w2) up to rounding, which the
        // added 1/16 cell covers.
        const float wmax = __builtin_amdgcn_sqrtf(sc.hc2) * sc.xsubf + sc.wmargin + 0.0625f;
        wc.x0c = (uint32_t)(int)fminf(fmaxf((float)cx0 - wmax, 0.0f), gmax);
        wc.x1c = (uint32_t)(int)fminf(fmaxf((float)cx1 + 1.0f + wmax, 0.0f), gmax);
    }
    return wc;
}

// [nlo, nhi) of row `row` for a slot of CAP entries (empty when no lane has
// a window in the row); false when it is empty or does not fit (the row is
// then read from global memory).  Every lane of the wave calls it.
template <uint32_t CAP>
__device__ __forceinline__ bool row_union(const StepArgs& a, const SceneConst& sc, const WaveColumn& wc, int row,
                                          uint32_t lo, uint32_t hi, uint32_t& nlo, uint32_t& nhi) {
    const bool has = hi > lo;
    nlo = nhi = 0u;
    if (__ballot(has) == 0u) return false;
    if (wc.one_col) {
        // Some lane's window of this row is not empty, so the row's column
        // lies inside the grid and both reads inside the table.
        const uint32_t c = wc.row0 + (uint32_t)((row / 3 - 1) * sc.G[1] + (row % 3 - 1)) * (uint32_t)sc.G[0];
        nlo = *(ConstWord*)(a.cstart + (c + wc.x0c));
        nhi = *(ConstWord*)(a.cstart + (c + wc.x1c + 1u));
        if (nlo < nhi && nhi - nlo <= CAP) return true;
    }
    nlo = wave_umin(has ? lo : 0xffffffffu);
    nhi = wave_umax(has ? hi : 0u);
    return nlo < nhi && nhi - nlo <= CAP;
}

// density_one with each row's candidates read from LDS: per row the wave
// copies the positions of the union of its lanes' windows into its slot as
// x, y, z planes (coalesced record loads), then every lane runs its own
// four-candidate trips over the slot.  It reads the sorted position records
// only, so the reorder pass need not write the planes for it.  Same
// candidates, same order, same arithmetic: density_one's results bit for
// bit.  Every lane of the wave calls it; inactive lanes have empty windows
// and store nothing.
__device__ __forceinline__ void density_one_staged(const StepArgs& a, const SceneConst& sc, uint32_t k, bool active,
                                                   __amdgpu_buffer_rsrc_t rpos, __amdgpu_buffer_rsrc_t rcs,
                                                   DensitySlot& slot) {
    const float4 pi = load4(rpos, k << 4);  // zeros past the buffer end
    const RowGeom g = row_geom(sc, pi.x, pi.y, pi.z);
    uint32_t lo[kRows], hi[kRows];
#pragma unroll
    for (int row = 0; row < kRows; ++row) {
        row_window(rcs, sc, g, row % 3 - 1, row / 3 - 1, lo[row], hi[row]);
        if (!active) lo[row] = hi[row] = 0u;
    }
    const uint32_t lane = threadIdx.x & 63u;
    const float h2 = sc.h2;
    float sum = 0.0f;
    const WaveColumn wc = wave_column(sc, g, active);
    // Row r + 1's records are loaded into registers while row r's trips run
    // from the slot, and stored into the slot once those trips are done, so
    // each copy's latency hides behind the previous row's work.  A copy holds
    // at most 2 x 64 records: lanes take entries lane and lane + 64.
    uint32_t nlo = 0u, nhi = 0u;
    bool nfit;
    float4 n0 = make_float4(0.f, 0.f, 0.f, 0.f), n1 = n0;
    auto fetch = [&](int row) {
        nfit = row_union<kStageD>(a, sc, wc, row, lo[row], hi[row], nlo, nhi);
        if (nfit) {
            if (lane < nhi - nlo) n0 = load4(rpos, (nlo + lane) << 4);
            if (lane + 64u < nhi - nlo) n1 = load4(rpos, (nlo + lane + 64u) << 4);
        }
    };
    fetch(0);
#pragma unroll
    for (int row = 0; row < kRows; ++row) {
        uint32_t m = 0u, mh = 0u;
        const uint32_t cnt = hi[row] - lo[row];
        const bool has = cnt > 0u;
        const uint32_t ulo = nlo, uhi = nhi;
        const bool fit = nfit;
        if (fit) {
            const uint32_t span = uhi - ulo;
            if (lane < span) {
                slot.v[lane] = n0.x;
                slot.v[kPlaneD + lane] = n0.y;
                slot.v[2 * kPlaneD + lane] = n0.z;
            }
            if (lane + 64u < span) {
                slot.v[lane + 64u] = n1.x;
                slot.v[kPlaneD + lane + 64u] = n1.y;
                slot.v[2 * kPlaneD + lane + 64u] = n1.z;
            }
            wave_lds_sync();
        }
        if (row + 1 < kRows) fetch(row + 1);
        if (fit) {
            // One induction variable, the trip's slot address, is also the
            // loop's exit test.
            const float* p = slot.v + (lo[row] - ulo);
            const float* const full_end = p + (cnt & ~3u);
            for (; p != full_end; p += 4)
                density_trip<true>(pi, h2, slot_quad(p, 0), slot_quad(p, 1), slot_quad(p, 2), 4, sum, m, mh);
            const int rem = (int)(cnt & 3u);
            if (rem > 0)
                density_trip<false>(pi, h2, slot_quad(p, 0), slot_quad(p, 1), slot_quad(p, 2), rem, sum, m, mh);
            wave_lds_sync();
        } else if (has) {
            // Past the buffer end the records read as zeros, as the planes do.
            uint32_t j = lo[row];
            const uint32_t full_end = j + (cnt & ~3u);
            float4 X, Y, Z;
            for (; j != full_end; j += 4u) {
                load_quad(rpos, j, X, Y, Z);
                density_trip<true>(pi, h2, X, Y, Z, 4, sum, m, mh);
            }
            const int rem = (int)(cnt & 3u);
            if (rem > 0) {
                load_quad(rpos, j, X, Y, Z);
                density_trip<false>(pi, h2, X, Y, Z, rem, sum, m, mh);
            }
        }
        if (cnt > 32u && a.mask_hi) a.mask_hi[(size_t)row * a.n + k] = mh;
        if (active) a.mask[(size_t)row * a.n + k] = m;
    }
    if (!active) return;
    float wr = 0.0f;
    const float pk[3] = {pi.x, pi.y, pi.z};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        wr += wall_rho((pk[d] - sc.bmin[d]) * sc.inv_h);
        wr += wall_rho((sc.wmax[d] - pk[d]) * sc.inv_h);
    }
    density_finish(a, sc, k, sum, wr);
}

struct ForceAcc {
    float px, py, pz, vx, vy, vz;
};

// A particle's next key and its new |v|^2.
struct Moved {
    uint32_t key;
    float v2;
};

// pos.w = p/rho^2 and vel.w = 1/rho of each particle.
__device__ __forceinline__ void force_pair(const SceneConst& sc, const float4& pi, const float4& vi,
                                           const float4& pj, const float4& vj, ForceAcc& f) {
    const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
    const float d2 = dist2(dx, dy, dz);
    // Hardware reciprocal square root.  d2 of two distinct particles is never
    // denormal; coincident particles (d2 = 0) get a finite 1/r times a zero
    // offset, so their pressure term vanishes as it does with 1/r := 0.
    const float inv_r = __builtin_amdgcn_rsqf(fmaxf(d2, 1e-30f));
    const float r = d2 * inv_r;
    const float hr = sc.h - r;
    const float w = hr * hr;
    const float s = ((pi.w + pj.w) * w) * inv_r;
    f.px = fmaf(s, dx, f.px);
    f.py = fmaf(s, dy, f.py);
    f.pz = fmaf(s, dz, f.pz);
    const float vv = hr * vj.w;
    f.vx = fmaf(vv, vj.x - vi.x, f.vx);
    f.vy = fmaf(vv, vj.y - vi.y, f.vy);
    f.vz = fmaf(vv, vj.z - vi.z, f.vz);
}

__device__ __forceinline__ Moved force_finish(const StepArgs& a, const SceneConst& sc, uint32_t k,
                                                 const float4& pi, const float4& vi, const ForceAcc& f);

// One row's pairs in ascending order of candidates: the re-tested ones before
// the masks', the second word's, the mask m's.  pos(j), vel(j): candidate j's
// records; walk(r, j0): the pairs of the bits of r (bit i: candidate j0 + i).
template <class P, class V, class W>
__device__ __forceinline__ void force_row(const StepArgs& a, const SceneConst& sc, uint32_t k, int row, uint32_t lo,
                                          uint32_t hi, uint32_t m, const float4& pi, const float4& vi, ForceAcc& f,
                                          P&& pos, V&& vel, W&& walk) {
    const uint32_t span = mask_span(lo, hi);
    if (span > 32u) {
        uint32_t mh = a.mask_hi ? a.mask_hi[(size_t)row * a.n + k] : 0u;
        if (row == 4) mh = without_self(mh, lo, hi, k, 32u);
        const uint32_t j1 = row_first(lo, hi, a.mask_hi ? 2u : 1u);
        for (uint32_t j = lo; j < j1; ++j) {
            const float4 pj = pos(j);
            if (j != k && dist2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z) < sc.h2)
                force_pair(sc, pi, vi, pj, vel(j), f);
        }
        walk(mask_ascending(mh, span, 32u), row_first(lo, hi, 2u));
    }
    walk(mask_ascending(m, span, 0u), row_first(lo, hi));
}

// The walk over records in global memory: each one's are loaded while the one
// before is summed, so a lane has two neighbours' loads in flight; unrolled
// twice, the two register sets swap roles instead of being copied.
__device__ __forceinline__ void walk_gathered(const SceneConst& sc, __amdgpu_buffer_rsrc_t rpos,
                                              __amdgpu_buffer_rsrc_t rvel, const float4& pi, const float4& vi,
                                              uint32_t r, uint32_t j0, ForceAcc& f) {
    if (!r) return;
    uint32_t j = j0 + (uint32_t)__builtin_ctz(r);
    float4 pj = load4(rpos, j << 4), vj = load4(rvel, j << 4);
#pragma unroll 2
    for (r &= r - 1u; r; r &= r - 1u) {
        j = j0 + (uint32_t)__builtin_ctz(r);
        const float4 pn = load4(rpos, j << 4), vn = load4(rvel, j << 4);
        force_pair(sc, pi, vi, pj, vj, f);
        pj = pn;
        vj = vn;
    }
    force_pair(sc, pi, vi, pj, vj, f);
}

__device__ __forceinline__ Moved force_one(const StepArgs& a, const SceneConst& sc, uint32_t k,
                                              __amdgpu_buffer_rsrc_t rpos, __amdgpu_buffer_rsrc_t rvel,
                                              __amdgpu_buffer_rsrc_t rcs) {
    const float4 pi = load4(rpos, k << 4);
    const float4 vi = load4(rvel, k << 4);
    const RowGeom g = row_geom(sc, pi.x, pi.y, pi.z);
    uint32_t lo[kRows], hi[kRows], mk[kRows];
#pragma unroll
    for (int row = 0; row < kRows; ++row) {
        row_window(rcs, sc, g, row % 3 - 1, row / 3 - 1, lo[row], hi[row]);
        mk[row] = a.mask[(size_t)row * a.n + k];
    }
    mk[4] = without_self(mk[4], lo[4], hi[4], k, 0u);
    ForceAcc f = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int row = 0; row < kRows; ++row) {
        force_row(
            a, sc, k, row, lo[row], hi[row], mk[row], pi, vi, f, [&](uint32_t j) { return load4(rpos, j << 4); },
            [&](uint32_t j) { return load4(rvel, j << 4); },
            [&](uint32_t r, uint32_t j0) { walk_gathered(sc, rpos, rvel, pi, vi, r, j0, f); });
    }
    return force_finish(a, sc, k, pi, vi, f);
}

// Integrate, clamp and stores of particle k, given its neighbours' sums, the
// walls' differences wj and its id; returns its next key.
__device__ __forceinline__ Moved force_finish(const StepArgs& a, const SceneConst& sc, uint32_t k,
                                                 const float4& pi, const float4& vi, const ForceAcc& f,
                                                 const float wj[3], uint32_t id) {
    const float cvi = sc.cV * vi.w;
    // The walls' pressure term at this particle's own p/rho^2.
    const float cwi = sc.cW * pi.w;
    float aw[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) aw[d] = cwi * wj[d];
    const float a0 = ((sc.cP * f.px + cvi * f.vx) + sc.g[0]) + aw[0];
    const float a1 = ((sc.cP * f.py + cvi * f.vy) + sc.g[1]) + aw[1];
    const float a2 = ((sc.cP * f.pz + cvi * f.vz) + sc.g[2]) + aw[2];
    if (a.acc) a.acc[k] = make_float4(a0, a1, a2, 0.0f);
    float v[3] = {vi.x + sc.dt * a0, vi.y + sc.dt * a1, vi.z + sc.dt * a2};
    float p[3] = {pi.x + sc.dt * v[0], pi.y + sc.dt * v[1], pi.z + sc.dt * v[2]};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if (p[d] < sc.lo[d]) {
            p[d] = sc.lo[d];
            if (v[d] < 0.0f) v[d] = -sc.e * v[d];
        } else if (p[d] > sc.hi[d]) {
            p[d] = sc.hi[d];
            if (v[d] > 0.0f) v[d] = -sc.e * v[d];
        }
    }
    if (a.pos_o) {
        a.pos_o[k] = make_float4(p[0], p[1], p[2], 0.0f);
        a.vel_o[k] = make_float4(v[0], v[1], v[2], 0.0f);
        a.id_o[k] = id;
    }
    if (a.xyz_out) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            a.xyz_out[3 * (size_t)id + d] = p[d];
            a.vel_out[3 * (size_t)id + d] = v[d];
        }
    }
    return {cell_key(sc, p[0], p[1], p[2]), speed2(v[0], v[1], v[2])};
}

__device__ __forceinline__ Moved force_finish(const StepArgs& a, const SceneConst& sc, uint32_t k,
                                                 const float4& pi, const float4& vi, const ForceAcc& f) {
    const float pk[3] = {pi.x, pi.y, pi.z};
    float wj[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
        wj[d] = wall_j((pk[d] - sc.bmin[d]) * sc.inv_h) - wall_j((sc.wmax[d] - pk[d]) * sc.inv_h);
    return force_finish(a, sc, k, pi, vi, f, wj, a.id_s[k]);
}

// Candidates a wave stages per row: its lanes' windows of one row lie in
// one sorted range of about 64 + 2 chords of particles when the wave sits in
// one y/z column (73 on average on the 1M dam break, 99 at the 99th
// percentile of the 4.4M sphere drop); a wider range (a wave across two
// columns, or a dense state) is walked from global memory.  A wave has two
// slots, one filled while the other is walked.  104 is the most that leaves
// room for 24 waves a CU, six per SIMD (159.7 of 160 KB); against 96 the
// force pass takes 117 for 130 us on the collapsed 1M dam break (alike, 72 to
// 77, on the fresh one), 185 for 191 on 96 scenes of 20k, 336 for 347 on the
// 4.4M drop.  Wider rows copied piece by piece
// through the slot: 102 to 169 spilled registers, 76 and 410 us.
constexpr uint32_t kStage = 104;
static_assert(kStage <= 128, "the copy into a slot takes two records per lane");
struct StageSlot {
    float4 pos[kStage];
    float4 vel[kStage];
};

// force_one with each row's candidates read from LDS: per row, the wave
// copies the union of its lanes' windows (contiguous, so the copy is
// coalesced) into a slot, then every lane walks its own mask over the
// slot.  Same pairs, same order, same arithmetic: the results are
// force_one's bit for bit.  Every lane of the wave calls it (the copy and
// the wave-wide bounds need them all); inactive lanes have empty windows.
__device__ __forceinline__ Moved force_one_staged(const StepArgs& a, const SceneConst& sc, uint32_t k,
                                                     bool active, __amdgpu_buffer_rsrc_t rpos,
                                                     __amdgpu_buffer_rsrc_t rvel, __amdgpu_buffer_rsrc_t rcs,
                                                     StageSlot& slot_a, StageSlot& slot_b) {
    // Loads past the buffer end return zeros.
    const float4 pi = load4(rpos, k << 4);
    const float4 vi = load4(rvel, k << 4);
    const RowGeom g = row_geom(sc, pi.x, pi.y, pi.z);
    uint32_t lo[kRows], hi[kRows], mk[kRows];
#pragma unroll
    for (int row = 0; row < kRows; ++row) {
        row_window(rcs, sc, g, row % 3 - 1, row / 3 - 1, lo[row], hi[row]);
        mk[row] = active ? a.mask[(size_t)row * a.n + k] : 0u;
        if (!active) lo[row] = hi[row] = 0u;
    }
    if (active) mk[4] = without_self(mk[4], lo[4], hi[4], k, 0u);
    const uint32_t lane = threadIdx.x & 63u;
    ForceAcc f = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // Each row's union of windows is copied into one of two slots by direct
    // loads into LDS (no registers), row r + 1's copy issued before row r is
    // walked, so the copy runs behind the walk.  Lane i of a copy writes
    // entry i (and i + 64) of the slot.
    uint32_t nlo, nhi;
    bool nfit;
    auto fetch = [&](int row) {
        const bool has = hi[row] > lo[row];
        nlo = wave_umin(has ? lo[row] : 0xffffffffu);
        nhi = wave_umax(has ? hi[row] : 0u);
        nfit = nlo < nhi && nhi - nlo <= kStage;
        if (!nfit) return;
        StageSlot& sl = (row & 1) ? slot_b : slot_a;
        const uint32_t span = nhi - nlo;
        if (lane < span) {
            lds_copy16(rpos, sl.pos, (nlo + lane) << 4);
            lds_copy16(rvel, sl.vel, (nlo + lane) << 4);
        }
        if (span > 64u && lane + 64u < span) {
            lds_copy16(rpos, sl.pos + 64, (nlo + lane + 64u) << 4);
            lds_copy16(rvel, sl.vel + 64, (nlo + lane + 64u) << 4);
        }
    };
    fetch(0);
#pragma unroll
    for (int row = 0; row < kRows; ++row) {
        const uint32_t ulo = nlo, uhi = nhi;
        const bool fit = nfit;
        StageSlot& slot = (row & 1) ? slot_b : slot_a;
        if (fit) lds_copy_wait();
        if (row + 1 < kRows) fetch(row + 1);
        if (ulo >= uhi) continue;
        if (fit) {
            // Entry j of the row sits at slot.pos[j - ulo], its velocity
            // kStage records further on.
            const float4* base = slot.pos - ulo;
            force_row(
                a, sc, k, row, lo[row], hi[row], mk[row], pi, vi, f, [&](uint32_t j) { return base[j]; },
                [&](uint32_t j) { return base[j + kStage]; },
                [&](uint32_t r, uint32_t j0) {
                    const float4* bm = base + j0;
                    for (; r; r &= r - 1u) {
                        const uint32_t i = (uint32_t)__builtin_ctz(r);
                        force_pair(sc, pi, vi, bm[i], bm[i + kStage], f);
                    }
                });
        } else {
            force_row(
                a, sc, k, row, lo[row], hi[row], mk[row], pi, vi, f, [&](uint32_t j) { return load4(rpos, j << 4); },
                [&](uint32_t j) { return load4(rvel, j << 4); },
                [&](uint32_t r, uint32_t j0) {
                    for (; r; r &= r - 1u) {
                        const uint32_t j = j0 + (uint32_t)__builtin_ctz(r);
                        force_pair(sc, pi, vi, load4(rpos, j << 4), load4(rvel, j << 4), f);
                    }
                });
        }
    }
    return active ? force_finish(a, sc, k, pi, vi, f) : Moved{0u, 0.0f};
}

// The step's bookkeeping, done by the density pass between the sort and the
// force pass: the sort has read the tile sums, which are cleared for the
// integrate pass, and the CFL step is set (launches of their own cost 4-6 us
// of a 40 us step each: 26k particles).  dt = min(dt_max, (cfl h) / (c0 +
// |v|max)), in this op order; it goes into the copy of the scene that the force
// pass reads, since this pass's own blocks read the table.  With a frame state, the
// step is added to the frame time (float, as the host frame loop adds it) and
// a frame of at least 1/30 s marks pending.
__device__ __forceinline__ void step_bookkeeping(const StepArgs& a) {
    if (a.cfl_scene && blockIdx.x == 0 && threadIdx.x < kSpeedSlots) {  // the first wave
        constexpr uint32_t kWords = sizeof(SceneConst) / 4u, kDt = offsetof(SceneConst, dt) / 4u;
        static_assert(kWords <= kSpeedSlots, "a lane a word");
        const uint32_t word = reinterpret_cast<const uint32_t*>(a.scenes)[min(threadIdx.x, kWords - 1u)];
        const uint32_t v2 = wave_umax(a.vmax2[threadIdx.x]);
        a.vmax2[threadIdx.x] = 0u;
        const SceneConst sc = scene_at(a.scenes, 0u);
        const float dt = fminf(sc.dt_max, (sc.cfl * sc.h) / (sc.c0 + sqrtf(__uint_as_float(v2))));
        if (threadIdx.x < kWords)
            reinterpret_cast<uint32_t*>(a.cfl_scene)[threadIdx.x] = threadIdx.x == kDt ? __float_as_uint(dt) : word;
        if (threadIdx.x == 0) {
            *a.dt_out = dt;
            if (a.frame) {
                const float ft = __uint_as_float(a.frame[3]) + dt;
                a.frame[3] = __float_as_uint(ft);
                a.frame[2] += 1u;
                if (!((double)ft < 0.0333333333)) a.frame[1] = 1u;
            }
        }
    }
    if (!a.head) return;
    const uint32_t words = scan_tiles(a.ncells, a.tile_shift) + 1u;  // and the sparse sort's count
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < words; i += gridDim.x * blockDim.x)
        a.head[a.ncells + i] = 0u;
}

// Next step's key, its run in the cell's chain, the tile sums and the largest
// speed (whole wave).
__device__ __forceinline__ void finish_particle(const StepArgs& a, uint32_t k, const Moved& to, bool active) {
    const uint32_t key = to.key;
    if (!a.head) return;  // a single step: there is no next one
    add_tile_sums(a.head + a.ncells, a.tile_shift, key, active);
    if (a.vmax2) wave_max_v2(a.vmax2, to.v2);
    if (active) a.key0[k] = key;
    push_run(a.head, a.next, key, k, active);  // last: it waits for its exchange's answer
}

template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void density_kernel(StepArgs a) {
    if (a.frame && a.frame[0]) return;
    step_bookkeeping(a);
    const __amdgpu_buffer_rsrc_t rpos = buffer_of(a.pos_s, a.n);
    const __amdgpu_buffer_rsrc_t rx = buffer_of(a.soa, a.n);
    const __amdgpu_buffer_rsrc_t ry = buffer_of(a.soa + a.n, a.n);
    const __amdgpu_buffer_rsrc_t rz = buffer_of(a.soa + 2 * (size_t)a.n, a.n);
    const __amdgpu_buffer_rsrc_t rcs = buffer_of(a.cstart, a.ncells + 1u);
    for_each_tile(a.ntiles, a.queue, [&](uint32_t t) {
        const uint2 ti = tile_at(a.tiles, t);
        const SceneConst sc = scene_at(a.scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        if (k < sc.p_end) density_one(a, sc, k, rpos, rx, ry, rz, rcs);
    });
}

// density_kernel with the rows staged in LDS (1.5 KB per wave).  Eight
// waves per SIMD: the bound fits it in 56 VGPRs (33 SGPRs in lanes of others).
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(8, 8))) void density_staged_kernel(StepArgs a) {
    if (a.frame && a.frame[0]) return;
    step_bookkeeping(a);
    __shared__ DensitySlot s_slot[BLOCK / 64];
    const __amdgpu_buffer_rsrc_t rpos = buffer_of(a.pos_s, a.n);
    const __amdgpu_buffer_rsrc_t rcs = buffer_of(a.cstart, a.ncells + 1u);
    DensitySlot& slot = s_slot[threadIdx.x >> 6];
    for_each_tile(a.ntiles, a.queue, [&](uint32_t t) {
        const uint2 ti = tile_at(a.tiles, t);
        const SceneConst sc = scene_at(a.scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        density_one_staged(a, sc, k, k < sc.p_end, rpos, rcs, slot);
    });
}

// Bound by its gathers: two records per neighbour, in a chain.  Six waves per
// SIMD (80 VGPRs, no VGPR spills).  With the second mask word read instead of
// the candidates before the mask's re-tested: 197k 37.5 -> 34.9 us, 65k
// collapsed 31.9 -> 25.0.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(6, 6))) void force_kernel(StepArgs a) {
    if (a.frame && a.frame[0]) return;
    const __amdgpu_buffer_rsrc_t rpos = buffer_of(a.pos_s, a.n);
    const __amdgpu_buffer_rsrc_t rvel = buffer_of(a.vel_s, a.n);
    const __amdgpu_buffer_rsrc_t rcs = buffer_of(a.cstart, a.ncells + 1u);
    uint32_t* queue = a.queue ? a.queue + 8 : nullptr;
    for_each_tile(a.ntiles, queue, [&](uint32_t t) {
        const uint2 ti = tile_at(a.tiles, t);
        const SceneConst sc = scene_at(a.scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        const bool active = k < sc.p_end;
        Moved to = {0u, 0.0f};
        if (active) to = force_one(a, sc, k, rpos, rvel, rcs);
        finish_particle(a, k, to, active);
    });
}

// force_kernel with the rows staged in LDS (two 3.25 KB slots per wave).  Bound
// by latency, of LDS reads in a chain per neighbour and of a row's copy.  Six
// waves per SIMD: the bound fits it in 80 VGPRs (nine spilled).  With the
// second mask word: the 1M dam break 74.4 -> 71.7 us fresh, 149 -> 117
// collapsed (a quarter of its rows over 32 candidates), 96 scenes of 20k
// 198 -> 185, the 4.4M drop 347 -> 336.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(6, 6))) void force_staged_kernel(StepArgs a) {
    if (a.frame && a.frame[0]) return;
    __shared__ StageSlot s_slot_a[BLOCK / 64];
    __shared__ StageSlot s_slot_b[BLOCK / 64];
    const __amdgpu_buffer_rsrc_t rpos = buffer_of(a.pos_s, a.n);
    const __amdgpu_buffer_rsrc_t rvel = buffer_of(a.vel_s, a.n);
    const __amdgpu_buffer_rsrc_t rcs = buffer_of(a.cstart, a.ncells + 1u);
    uint32_t* queue = a.queue ? a.queue + 8 : nullptr;
    StageSlot& slot_a = s_slot_a[threadIdx.x >> 6];
    StageSlot& slot_b = s_slot_b[threadIdx.x >> 6];
    for_each_tile(a.ntiles, queue, [&](uint32_t t) {
        const uint2 ti = tile_at(a.tiles, t);
        const SceneConst sc = scene_at(a.scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        const bool active = k < sc.p_end;
        const Moved to = force_one_staged(a, sc, k, active, rpos, rvel, rcs, slot_a, slot_b);
        finish_particle(a, k, to, active);
    });
}

// ------------------------------------------------------------- split form
//
// With few particles the chip is idle and a pass lasts as long as one wave's
// serial chain: nine rows one after the other, each waiting for its copy or
// its gathers (500 particles, 8 waves: density 12.5 us, force 11.3 us; 24k:
// 13.4 and 13.9 us).  The split form shortens that chain.  Density: nine
// waves per 64 particles, one per row, so all copies are in flight together
// and every row's trips run at the same time; the rows' neighbours then go
// into one list per particle, with their terms, and the first wave adds the
// terms in list order, so the sum is the other forms' bit for bit.  The force
// pass walks that list, without windows, masks or rows.

constexpr uint32_t kKept = 5;        // a gathered row's terms kept in its copy's place
constexpr uint32_t kChunk = 64;      // entries of a list in LDS at a time
template <bool V>
struct Bool {
    static constexpr bool value = V;
};

static_assert(kKept * kSplitTile * 4 <= sizeof(DensitySlot), "the kept terms fit a row's copy");

struct SplitShared {
    DensitySlot rec[kRows];                        // the rows' copies, as planes: lanes read them in step,
                                                   // which records of 16 bytes would serve four at a time
    float term[kChunk + 4][kSplitTile];            // the neighbours' terms, itself included
    uint16_t id[kChunk + 1][kSplitTile];           // the neighbours; the particle itself goes to the last place
    uint32_t count[3][kSplitTile];                 // neighbours per row, one byte a row (itself included)
    float wall[kSplitTile];
};

// One candidate's term c = min(d^2 - h^2, 0), formed as density_trip forms it.
__device__ __forceinline__ float split_term(const float4& pi, float h2, float x, float y, float z) {
    return dist2(pi.x - x, pi.y - y, pi.z - z) - h2;
}

// Runs a row's trips: candidate j's term goes to f(c), m and mh receive the
// mask words.  quad(j, X, Y, Z): the coordinates of candidates j .. j + 3; it
// may be asked for up to seven past the row, whose values are not used.
struct Quad {
    float4 X, Y, Z;
};
template <class G, class F>
__device__ __forceinline__ void split_trips(G&& quad, const float4& pi, float h2, uint32_t lo, uint32_t hi,
                                            uint32_t& m, uint32_t& mh, F&& f) {
    m = 0u;
    mh = 0u;
    if (lo >= hi) return;
    Quad cur, nxt;
    auto test = [&](const Quad& q, uint32_t left) {
        mh = push_out(mh, m);
        const float xs[4] = {q.X.x, q.X.y, q.X.z, q.X.w}, ys[4] = {q.Y.x, q.Y.y, q.Y.z, q.Y.w},
                    zs[4] = {q.Z.x, q.Z.y, q.Z.z, q.Z.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float t = split_term(pi, h2, xs[u], ys[u], zs[u]);
            if (u != 0) t = (uint32_t)u < left ? t : 1.0f;
            const float c = fminf(t, 0.0f);
            m = push_sign(m, c);
            f(c);
        }
    };
    uint32_t j = lo;
    const uint32_t full_end = lo + ((hi - lo) & ~3u);
    quad(j, cur);
    // The next trip's records load while this one's are tested, the two
    // register sets in turn.
    for (;;) {
        if (j == full_end) {
            if (j != hi) test(cur, hi - j);
            break;
        }
        quad(j + 4u, nxt);
        test(cur, 4u);
        j += 4u;
        if (j == full_end) {
            if (j != hi) test(nxt, hi - j);
            break;
        }
        quad(j + 4u, cur);
        test(nxt, 4u);
        j += 4u;
    }
}

// Visits the candidates of a word's ascending bits (bit i: j0 + i), the next
// one's record loading while this one's is used.
template <class G, class F>
__device__ __forceinline__ void split_bits(uint32_t r, uint32_t j0, G&& get, F&& f) {
    if (!r) return;
    uint32_t j = j0 + (uint32_t)__builtin_ctz(r);
    float4 p = get(j);
#pragma unroll 2
    for (;;) {
        r &= r - 1u;
        const uint32_t jn = r ? j0 + (uint32_t)__builtin_ctz(r) : j;
        const float4 pn = get(jn);
        f(j, p);
        if (!r) break;
        j = jn;
        p = pn;
    }
}

__global__ __launch_bounds__(64 * kRows) void density_split_kernel(StepArgs a) {
    if (a.frame && a.frame[0]) return;
    step_bookkeeping(a);
    __shared__ SplitShared sh;
    const __amdgpu_buffer_rsrc_t rpos = buffer_of(a.pos_s, a.n);
    const __amdgpu_buffer_rsrc_t rcs = buffer_of(a.cstart, a.ncells + 1u);
    const uint2 ti = tile_at(a.tiles, xcd_block(blockIdx.x, gridDim.x));
    const SceneConst sc = scene_at(a.scenes, ti.x);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t k = ti.y + lane;
    const bool active = k < sc.p_end;
    const float4 pi = load4(rpos, k << 4);  // zeros past the buffer end
    uint32_t lo, hi;
    split_window(rcs, sc, pi, w % 3 - 1, w / 3 - 1, lo, hi);
    if (!active) lo = hi = 0u;
    // The row's union of windows.
    const bool has = hi > lo;
    const uint32_t ulo = wave_umin(has ? lo : 0xffffffffu);
    const uint32_t uhi = wave_umax(has ? hi : 0u);
    const bool fit = ulo < uhi && uhi - ulo <= kStageD;
    if (fit) {
        float* v = sh.rec[w].v;
        const bool c0 = lane < uhi - ulo, c1 = lane + 64u < uhi - ulo;
        float4 n0, n1;
        if (c0) n0 = load4(rpos, (ulo + lane) << 4);
        if (c1) n1 = load4(rpos, (ulo + lane + 64u) << 4);
        if (c0) {
            v[lane] = n0.x;
            v[kPlaneD + lane] = n0.y;
            v[2 * kPlaneD + lane] = n0.z;
        }
        if (c1) {
            v[lane + 64u] = n1.x;
            v[kPlaneD + lane + 64u] = n1.y;
            v[2 * kPlaneD + lane + 64u] = n1.z;
        }
        wave_lds_sync();
    }
    auto staged = [&](uint32_t j, Quad& q) {
        const float* p = sh.rec[w].v + (j - ulo);
        q.X = slot_quad(p, 0);
        q.Y = slot_quad(p, 1);
        q.Z = slot_quad(p, 2);
    };
    auto gathered = [&](uint32_t j, Quad& q) { load_quad(rpos, j, q.X, q.Y, q.Z); };
    auto staged_one = [&](uint32_t j) {
        const float* p = sh.rec[w].v + (j - ulo);
        return make_float4(p[0], p[kPlaneD], p[2 * kPlaneD], 0.0f);
    };
    auto gathered_one = [&](uint32_t j) { return load4(rpos, j << 4); };
    uint32_t m, mh, nkept = 0u;
    float* const kept = sh.rec[w].v + lane;
    if (fit)
        split_trips(staged, pi, sc.h2, lo, hi, m, mh, [](float) {});
    else
        split_trips(gathered, pi, sc.h2, lo, hi, m, mh, [&](float c) {
            if (c < 0.0f) {
                if (nkept < kKept) kept[nkept * kSplitTile] = c;
                ++nkept;
            }
        });
    const uint32_t span = mask_span(lo, hi);
    if (active) {
        a.mask[(size_t)w * a.n + k] = m;
        if (a.mask_hi && span > 32u) a.mask_hi[(size_t)w * a.n + k] = mh;
    }
    // A row the two words do not cover counts as more than any list holds.
    const uint32_t cnt = span > 64u ? kRowOver : (uint32_t)__popc(m) + (uint32_t)__popc(mh);
    reinterpret_cast<uint8_t*>(sh.count)[(((uint32_t)w >> 2) * kSplitTile + lane) * 4u + ((uint32_t)w & 3u)] = (uint8_t)cnt;
    __syncthreads();
    // Where this row's neighbours go in the list, and how many there are.
    uint32_t base = 0u, total = 0u;
#pragma unroll
    for (int g = 0; g < 3; ++g) {
        const uint32_t c = sh.count[g][lane];
        const uint32_t before = w >= 4 * g + 4 ? 0xffffffffu : w > 4 * g ? (1u << (8 * (w - 4 * g))) - 1u : 0u;
        base = __builtin_amdgcn_sad_u8(c & before, 0u, base);
        total = __builtin_amdgcn_sad_u8(g == 2 ? c & 0xffu : c, 0u, total);
    }
    // A corner row has the fewest neighbours to list.
    if (w == kRows - 1) {
        float wr = 0.0f;
        const float pk[3] = {pi.x, pi.y, pi.z};
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            wr += wall_rho((pk[d] - sc.bmin[d]) * sc.inv_h);
            wr += wall_rho((sc.wmax[d] - pk[d]) * sc.inv_h);
        }
        sh.wall[lane] = wr;
    }
    // Lists go through LDS kChunk entries at a time (nearly always once).
    // The list for the force pass leaves the particle itself out; its term is
    // in the sum.
    const uint32_t most = wave_umax(total);  // the same in every wave, and so is the branch on it
    const bool over = most > kListMax + 1u;
    const uint32_t listed = total ? total - 1u : 0u;
    float sum = 0.0f;
    auto list = [&](uint32_t first, auto all) {
        constexpr bool kAll = decltype(all)::value;  // every entry is in this chunk
        uint32_t at = base - first, i = 0u;
        auto put = [&](uint32_t j, float c) {
            if (kAll || at < kChunk) sh.term[at][lane] = c;
            // Candidates past k come one place earlier in the list (rows go
            // in ascending order).
            const uint32_t e = j == k ? kChunk : at - (j > k ? 1u : 0u);
            if (kAll || e <= kChunk) sh.id[e][lane] = (uint16_t)j;
            ++at;
        };
        auto bits = [&](uint32_t r, uint32_t j0) {
            if (fit)
                split_bits(r, j0, staged_one,
                           [&](uint32_t j, const float4& pj) { put(j, split_term(pi, sc.h2, pj.x, pj.y, pj.z)); });
            else
                for (; r; r &= r - 1u, ++i) {
                    const uint32_t j = j0 + (uint32_t)__builtin_ctz(r);
                    float c;
                    if (i < kKept) {
                        c = kept[i * kSplitTile];
                    } else {
                        const float4 pj = gathered_one(j);
                        c = split_term(pi, sc.h2, pj.x, pj.y, pj.z);
                    }
                    put(j, c);
                }
        };
        if (__ballot(mh != 0u)) bits(mask_ascending(mh, span, 32u), row_first(lo, hi, 2u));
        bits(mask_ascending(m, span, 0u), row_first(lo, hi));
    };
    for (uint32_t first = 0u;; first += kChunk) {
        if (most <= kChunk)
            list(0u, Bool<true>());
        else if (!over)
            list(first, Bool<false>());
        __syncthreads();
        if (over) {
            // The first wave runs every row itself; the force pass walks masks.
            if (w != 0) return;
#pragma unroll 1
            for (int r = 0; r < kRows; ++r) {
                split_window(rcs, sc, pi, r % 3 - 1, r / 3 - 1, lo, hi);
                if (!active) lo = hi = 0u;
                split_trips(gathered, pi, sc.h2, lo, hi, m, mh, [&](float c) { sum = fmaf(c * c, -c, sum); });
            }
            if (active) {
                a.ncount[k] = kListOver;
                density_finish(a, sc, k, sum, sh.wall[lane]);
            }
            return;
        }
        if (w != 0) {
            if (active) {
                if (w == 1 && first == 0u) a.ncount[k] = listed;
                for (uint32_t q = (uint32_t)w - 1u; q < kChunk / 4u && first + 4u * q < listed; q += (uint32_t)kRows - 1u)
                    reinterpret_cast<uint2*>(a.nlist)[(size_t)(first / 4u + q) * a.n + k] =
                        make_uint2(sh.id[4u * q][lane] | ((uint32_t)sh.id[4u * q + 1u][lane] << 16),
                                   sh.id[4u * q + 2u][lane] | ((uint32_t)sh.id[4u * q + 3u][lane] << 16));
            }
        } else {
            // Eight terms at a time, the next four loaded while four are
            // added; terms past the list's end count as 0, which adds nothing.
            const uint32_t left = total > first ? min(total - first, kChunk) : 0u;
            float c[4], d[4];
            auto four = [&](uint32_t i, float* v) {
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = sh.term[i + u][lane];
            };
            auto add = [&](uint32_t i, const float* v) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float t = i + (uint32_t)u < left ? v[u] : 0.0f;
                    sum = fmaf(t * t, -t, sum);
                }
            };
            four(0u, c);
            for (uint32_t i = 0; i < left; i += 8u) {
                four(i + 4u, d);
                add(i, c);
                four(min(i + 8u, kChunk), c);
                add(i + 4u, d);
            }
        }
        if (most <= first + kChunk) break;
        __syncthreads();
    }
    if (w == 0 && active) density_finish(a, sc, k, sum, sh.wall[lane]);
}

// Force, split form.  Four waves per 64 particles take the list in rounds of
// 32 neighbours, eight per wave, whose records are gathered together; each
// leaves its pairs' factors in LDS, and two waves then add them in list order
// (force_pair's sums, one the pressure terms and one the viscosity terms)
// while a third takes the walls.  One wave doing all of it waited for each
// few neighbours' gathers (24k: walk 8200 of 17000 cycles, and 3900 for the
// walls, integration and stores after it).
constexpr uint32_t kRound = 32;
constexpr int kForceWaves = 4;
constexpr int kPerWave = (int)kRound / kForceWaves;

struct ForceSplitShared {
    float4 press[kRound][kSplitTile];  // s, dx, dy, dz of a pair
    float4 visc[kRound][kSplitTile];   // vv, dvx, dvy, dvz
    float sum[3][kSplitTile];          // the viscosity sums
    float wall[3][kSplitTile];         // the walls' differences
    uint32_t id[kSplitTile];
};

__global__ __launch_bounds__(64 * kForceWaves) void force_split_kernel(StepArgs a) {
    if (a.frame && a.frame[0]) return;
    __shared__ ForceSplitShared sh;
    const __amdgpu_buffer_rsrc_t rpos = buffer_of(a.pos_s, a.n);
    const __amdgpu_buffer_rsrc_t rvel = buffer_of(a.vel_s, a.n);
    const __amdgpu_buffer_rsrc_t rl = buffer_of(a.nlist, kListMax * a.n);
    const uint2 ti = tile_at(a.tiles, xcd_block(blockIdx.x, gridDim.x));
    const SceneConst sc = scene_at(a.scenes, ti.x);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t k = ti.y + lane;
    const bool active = k < sc.p_end;
    // Entries past a list's end hold any index; their pairs are not added.
    auto ids = [&](uint32_t q) { return __builtin_amdgcn_raw_buffer_load_b64(rl, (int)((q * a.n + k) << 3), 0, 0); };
    u32x2 q0 = ids(2u * (uint32_t)w), q1 = ids(2u * (uint32_t)w + 1u);
    const float4 pi = load4(rpos, k << 4), vi = load4(rvel, k << 4);
    const uint32_t count = active ? a.ncount[k] : 0u;
    const uint32_t id = w == 2 && active ? a.id_s[k] : 0u;
    float4 pj[kPerWave], vj[kPerWave];
    auto gather = [&]() {
        const uint32_t j[kPerWave] = {q0.x & 0xffffu, q0.x >> 16, q0.y & 0xffffu, q0.y >> 16,
                                      q1.x & 0xffffu, q1.x >> 16, q1.y & 0xffffu, q1.y >> 16};
#pragma unroll
        for (int u = 0; u < kPerWave; ++u) pj[u] = load4(rpos, j[u] << 4);
#pragma unroll
        for (int u = 0; u < kPerWave; ++u) vj[u] = load4(rvel, j[u] << 4);
    };
    gather();  // before the counts are known: any index stays inside the buffers' bounds checks
    if (__ballot(count > kListMax) != 0u) {  // the same in every wave
        if (w != 0) return;
        Moved to = {0u, 0.0f};
        if (active) to = force_one(a, sc, k, rpos, rvel, buffer_of(a.cstart, a.ncells + 1u));
        finish_particle(a, k, to, active);
        return;
    }
    float f[3] = {0.f, 0.f, 0.f};
    for (uint32_t first = 0u;; first += kRound) {
        if (__ballot(count > first + (uint32_t)(kPerWave * w)) != 0u) {
            if (first != 0u) {
                q0 = ids(first / 4u + 2u * (uint32_t)w);
                q1 = ids(first / 4u + 2u * (uint32_t)w + 1u);
                gather();
            }
#pragma unroll
            for (int u = 0; u < kPerWave; ++u) {
                // force_pair's factors.
                const float dx = pi.x - pj[u].x, dy = pi.y - pj[u].y, dz = pi.z - pj[u].z;
                const float d2 = dist2(dx, dy, dz);
                const float inv_r = __builtin_amdgcn_rsqf(fmaxf(d2, 1e-30f));
                const float r = d2 * inv_r;
                const float hr = sc.h - r;
                const float s = ((pi.w + pj[u].w) * (hr * hr)) * inv_r;
                sh.press[kPerWave * w + u][lane] = make_float4(s, dx, dy, dz);
                sh.visc[kPerWave * w + u][lane] =
                    make_float4(hr * vj[u].w, vj[u].x - vi.x, vj[u].y - vi.y, vj[u].z - vi.z);
            }
        }
        __syncthreads();
        const uint32_t left = count > first ? min(count - first, kRound) : 0u;
        if (w < 2) {
            auto chain = [&](const float4(&t)[kRound][kSplitTile]) {
                // Four pairs at a time, the next four loaded meanwhile.
                float4 c[4], n[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) c[u] = t[u][lane];
#pragma unroll 2
                for (uint32_t i = 0; i < left; i += 4u) {
                    const uint32_t in = min(i + 4u, kRound - 4u);
#pragma unroll
                    for (int u = 0; u < 4; ++u) n[u] = t[in + u][lane];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (i + (uint32_t)u < left) {
                            f[0] = fmaf(c[u].x, c[u].y, f[0]);
                            f[1] = fmaf(c[u].x, c[u].z, f[1]);
                            f[2] = fmaf(c[u].x, c[u].w, f[2]);
                        }
                        c[u] = n[u];
                    }
                }
            };
            if (w == 0)
                chain(sh.press);
            else
                chain(sh.visc);
        } else if (w == 2 && first == 0u) {
            const float p[3] = {pi.x, pi.y, pi.z};
#pragma unroll
            for (int d = 0; d < 3; ++d)
                sh.wall[d][lane] = wall_j((p[d] - sc.bmin[d]) * sc.inv_h) - wall_j((sc.wmax[d] - p[d]) * sc.inv_h);
            sh.id[lane] = id;
        }
        if (__ballot(count > first + kRound) == 0u) break;
        __syncthreads();
    }
    if (w == 1) {
#pragma unroll
        for (int d = 0; d < 3; ++d) sh.sum[d][lane] = f[d];
    }
    __syncthreads();
    if (w != 0) return;
    Moved to = {0u, 0.0f};
    if (active) {
        const ForceAcc acc = {f[0], f[1], f[2], sh.sum[0][lane], sh.sum[1][lane], sh.sum[2][lane]};
        const float wj[3] = {sh.wall[0][lane], sh.wall[1][lane], sh.wall[2][lane]};
        to = force_finish(a, sc, k, pi, vi, acc, wj, sh.id[lane]);
    }
    finish_particle(a, k, to, active);
}

// Uploads come in any order, a lattice's fastest axis often across the
// cells' rows, so a wave's particles can lie in as many tiles as it has lanes
// and one atomic per run would queue on the few tile sums of a small grid: a
// block counts them in LDS first (grids of up to kHashTiles tiles).
constexpr uint32_t kHashTiles = 2048;

// The tile sums of one block's particles: add() for every lane of the block,
// flush() once at its end.
struct BlockTileSums {
    uint32_t* tsum;
    uint32_t shift, tiles;
    uint32_t* local;  // kHashTiles words of LDS; null: straight to memory
    __device__ __forceinline__ BlockTileSums(uint32_t* head, uint32_t ncells, uint32_t shift_, uint32_t* lds)
        : tsum(head + ncells), shift(shift_), tiles(scan_tiles(ncells, shift_)) {
        local = tiles <= kHashTiles ? lds : nullptr;
        if (local) {
            for (uint32_t i = threadIdx.x; i < tiles; i += blockDim.x) local[i] = 0u;
            __syncthreads();
        }
    }
    __device__ __forceinline__ void add(uint32_t key, bool active) {
        if (!local)
            add_tile_sums(tsum, shift, key, active);
        else if (active)
            atomicAdd(local + (key >> shift), 1u);
    }
    __device__ __forceinline__ void flush() {
        if (!local) return;
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < tiles; i += blockDim.x)
            if (local[i]) atomicAdd(tsum + i, local[i]);
    }
};

__global__ void hash_kernel(const float4* __restrict__ pos, const float4* __restrict__ vel,
                            uint32_t* __restrict__ key0, uint32_t* __restrict__ next, uint32_t* __restrict__ head,
                            uint32_t ncells, uint32_t tile_shift, uint32_t* __restrict__ vmax2,
                            const SceneConst* __restrict__ scenes, const uint2* __restrict__ tiles, uint32_t ntiles) {
    __shared__ uint32_t s_sum[kHashTiles];
    BlockTileSums sums(head, ncells, tile_shift, s_sum);
    uint32_t t0, t1;
    tile_span(ntiles, t0, t1);
    for (uint32_t t = t0; t < t1; ++t) {
        const uint2 ti = tile_at(tiles, t);
        const SceneConst sc = scene_at(scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        const bool active = k < sc.p_end;
        uint32_t key = 0;
        if (active) {
            const float4 p = pos[k];
            key = cell_key(sc, p.x, p.y, p.z);
        }
        push_run(head, next, key, k, active);
        sums.add(key, active);
        if (active) key0[k] = key;
        if (vmax2) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (active) v = vel[k];
            wave_max_v2(vmax2, speed2(v.x, v.y, v.z));
        }
    }
    sums.flush();
}

// pack3, the identity ids and the hash of one scene of n particles in one
// pass; vel_in may be null (zero velocity).
__global__ __launch_bounds__(256) void upload_hash_kernel(const float* __restrict__ xyz, const float* __restrict__ vel_in,
                                                          float4* __restrict__ pos, float4* __restrict__ vel,
                                                          uint32_t* __restrict__ id, uint32_t* __restrict__ key0,
                                                          uint32_t* __restrict__ next, uint32_t* __restrict__ head,
                                                          uint32_t n, uint32_t ncells, uint32_t tile_shift,
                                                          SceneConst sc) {
    __shared__ uint32_t s_sum[kHashTiles];
    BlockTileSums sums(head, ncells, tile_shift, s_sum);
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = k < n;
    uint32_t key = 0;
    if (active) {
        const float4 p = make_float4(xyz[3 * (size_t)k], xyz[3 * (size_t)k + 1], xyz[3 * (size_t)k + 2], 0.0f);
        pos[k] = p;
        vel[k] = vel_in ? make_float4(vel_in[3 * (size_t)k], vel_in[3 * (size_t)k + 1], vel_in[3 * (size_t)k + 2], 0.0f)
                        : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        id[k] = k;
        key = cell_key(sc, p.x, p.y, p.z);
        key0[k] = key;
    }
    push_run(head, next, key, k, active);
    sums.add(key, active);
    sums.flush();
}

// Neighbour sets exactly as force_one iterates them (self included).
template <int FILL>
__global__ void neighbors_kernel(StepArgs a, const uint32_t* __restrict__ offsets,
                                 uint32_t* __restrict__ out) {
    const __amdgpu_buffer_rsrc_t rcs = buffer_of(a.cstart, a.ncells + 1u);
    uint32_t t0, t1;
    tile_span(a.ntiles, t0, t1);
    for (uint32_t t = t0; t < t1; ++t) {
        const uint2 ti = tile_at(a.tiles, t);
        const SceneConst sc = scene_at(a.scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        if (k >= sc.p_end) continue;
        const float4 pi = a.pos_s[k];
        const RowGeom g = row_geom(sc, pi.x, pi.y, pi.z);
        uint32_t c = 0;
        const uint32_t o = FILL ? offsets[k] : 0u;
        for (int row = 0; row < kRows; ++row) {
            uint32_t lo, hi;
            row_window(rcs, sc, g, row % 3 - 1, row / 3 - 1, lo, hi);
            row_neighbors(
                lo, hi, a.mask[(size_t)row * a.n + k],
                [&](uint32_t j) {
                    const float4 pj = a.pos_s[j];
                    return dist2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z) < sc.h2;
                },
                [&](uint32_t j) {
                    if (FILL) out[o + c] = j;
                    ++c;
                });
        }
        if (!FILL) out[k] = c;
    }
}

// Keys of the sorted positions (the cell-count sort does not store them).
__global__ void sorted_keys_kernel(const float4* __restrict__ pos_s, uint32_t* __restrict__ skey,
                                   const SceneConst* __restrict__ scenes, const uint2* __restrict__ tiles) {
    const uint2 ti = tile_at(tiles, blockIdx.x);
    const SceneConst sc = scene_at(scenes, ti.x);
    const uint32_t k = ti.y + threadIdx.x;
    if (k < sc.p_end) skey[k] = cell_key(sc, pos_s[k].x, pos_s[k].y, pos_s[k].z);
}

__global__ void frame_reset_kernel(uint32_t* __restrict__ frame) {
    if (threadIdx.x < (uint32_t)kFrameWords) frame[threadIdx.x] = 0u;
}

__global__ void fill_u32_kernel(uint32_t* __restrict__ p, uint32_t v, size_t count) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void unpermute3_kernel(uint32_t n, const float4* __restrict__ src,
                                  const uint32_t* __restrict__ id, float* __restrict__ out) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const float4 v = src[k];
    const uint32_t i = id[k];
    out[3 * (size_t)i] = v.x;
    out[3 * (size_t)i + 1] = v.y;
    out[3 * (size_t)i + 2] = v.z;
}

// 16 bytes per lane (both buffers start 256-byte aligned), the rest and the
// flag by the first lanes.
__global__ void copy_out_kernel(const uint32_t* __restrict__ src, size_t words, const uint32_t* __restrict__ flag,
                                uint32_t* __restrict__ dst) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t quads = words / 4;
    if (i < quads) reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
    if (i < words % 4) dst[4 * quads + i] = src[4 * quads + i];
    if (i == 0) dst[words] = *flag;
}

__global__ __launch_bounds__(1024) void read_small_kernel(uint32_t n, const float4* __restrict__ src4,
                                                          const float* __restrict__ src1,
                                                          const uint32_t* __restrict__ id,
                                                          const uint32_t* __restrict__ flag, float* __restrict__ dst) {
    __shared__ float s[3 * kReadSmall];
    for (uint32_t k = threadIdx.x; k < n; k += 1024u) {
        const uint32_t i = id[k];
        if (i >= n) continue;
        if (src4) {
            const float4 v = src4[k];
            s[3u * i] = v.x;
            s[3u * i + 1u] = v.y;
            s[3u * i + 2u] = v.z;
        } else {
            s[i] = src1[k];
        }
    }
    __syncthreads();
    const uint32_t words = src4 ? 3u * n : n;
    for (uint32_t i = threadIdx.x; i < words; i += 1024u) dst[i] = s[i];
    if (threadIdx.x == 0) reinterpret_cast<uint32_t*>(dst)[words] = *flag;
}

__global__ void unpermute1_kernel(uint32_t n, const float* __restrict__ src,
                                  const uint32_t* __restrict__ id, float* __restrict__ out) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    out[id[k]] = src[k];
}

// One launch where three copies by the runtime took 12 us of a small handle's
// checkpoint.
__global__ void copy_state_kernel(uint32_t n, float4* __restrict__ dp, float4* __restrict__ dv,
                                  uint32_t* __restrict__ di, const float4* __restrict__ sp,
                                  const float4* __restrict__ sv, const uint32_t* __restrict__ si) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    dp[k] = sp[k];
    dv[k] = sv[k];
    di[k] = si[k];
}

__global__ void pack3_kernel(uint32_t n, const float* __restrict__ src, float4* __restrict__ dst) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    dst[k] = src ? make_float4(src[3 * (size_t)k], src[3 * (size_t)k + 1], src[3 * (size_t)k + 2], 0.0f)
                 : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

inline uint32_t blocks_for(size_t n, int b) { return (uint32_t)((n + b - 1) / b); }

}  // namespace

#define SPH_DISPATCH_BLOCK(KERNEL, block, grid, st, ...)                                       \
    switch (block) {                                                                          \
        case 64: hipLaunchKernelGGL(KERNEL<64>, dim3(grid), dim3(64), 0, st, __VA_ARGS__); break;   \
        case 128: hipLaunchKernelGGL(KERNEL<128>, dim3(grid), dim3(128), 0, st, __VA_ARGS__); break; \
        case 512: hipLaunchKernelGGL(KERNEL<512>, dim3(grid), dim3(512), 0, st, __VA_ARGS__); break; \
        default: hipLaunchKernelGGL(KERNEL<256>, dim3(grid), dim3(256), 0, st, __VA_ARGS__); break;  \
    }

hipError_t launch_density(hipStream_t st, int block, uint32_t grid, const StepArgs& a, int staged) {
    if (grid == 0) return hipSuccess;
    if (staged) {
        SPH_DISPATCH_BLOCK(density_staged_kernel, block, grid, st, a);
    } else {
        SPH_DISPATCH_BLOCK(density_kernel, block, grid, st, a);
    }
    return hipGetLastError();
}

hipError_t launch_force(hipStream_t st, int block, uint32_t grid, const StepArgs& a, int staged) {
    if (grid == 0) return hipSuccess;
    if (staged) {
        SPH_DISPATCH_BLOCK(force_staged_kernel, block, grid, st, a);
    } else {
        SPH_DISPATCH_BLOCK(force_kernel, block, grid, st, a);
    }
    return hipGetLastError();
}

hipError_t launch_density_split(hipStream_t st, const StepArgs& a) {
    if (a.ntiles == 0) return hipSuccess;
    hipLaunchKernelGGL(density_split_kernel, dim3(a.ntiles), dim3(64 * kRows), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_force_split(hipStream_t st, const StepArgs& a) {
    if (a.ntiles == 0) return hipSuccess;
    hipLaunchKernelGGL(force_split_kernel, dim3(a.ntiles), dim3(64 * kForceWaves), 0, st, a);
    return hipGetLastError();
}

template <class K>
static int occupancy(K kernel, int block) {
    int nb = 0;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, block, 0) == hipSuccess ? nb : 0;
}

int force_blocks_per_cu(int block, int staged) {
    // Looked up once per form and block size; 0 = not yet (stores nb + 1).
    static std::atomic<int> cache[2][4];
    const int b = block == 64 ? 0 : block == 128 ? 1 : block == 512 ? 3 : 2;
    std::atomic<int>& c = cache[staged ? 1 : 0][b];
    const int known = c.load(std::memory_order_relaxed);
    if (known > 0) return known - 1;
    int nb = 0;
    switch (b) {
        case 0: nb = staged ? occupancy(force_staged_kernel<64>, 64) : occupancy(force_kernel<64>, 64); break;
        case 1: nb = staged ? occupancy(force_staged_kernel<128>, 128) : occupancy(force_kernel<128>, 128); break;
        case 3: nb = staged ? occupancy(force_staged_kernel<512>, 512) : occupancy(force_kernel<512>, 512); break;
        default: nb = staged ? occupancy(force_staged_kernel<256>, 256) : occupancy(force_kernel<256>, 256); break;
    }
    c.store(nb + 1, std::memory_order_relaxed);
    return nb;
}

hipError_t launch_hash(hipStream_t st, int block, uint32_t grid, const float4* pos, const float4* vel,
                       uint32_t* key0, uint32_t* next, uint32_t* head, uint32_t ncells, uint32_t tile_shift,
                       uint32_t* vmax2, const SceneConst* scenes, const uint2* tiles, uint32_t ntiles) {
    if (grid == 0) return hipSuccess;
    hipLaunchKernelGGL(hash_kernel, dim3(grid), dim3(block), 0, st, pos, vel, key0, next, head, ncells,
                       tile_shift, vmax2, scenes, tiles, ntiles);
    return hipGetLastError();
}

hipError_t launch_upload_hash(hipStream_t st, const float* xyz, const float* vel_in, float4* pos, float4* vel,
                              uint32_t* id, uint32_t* key0, uint32_t* next, uint32_t* head, uint32_t n,
                              uint32_t ncells, uint32_t tile_shift, const SceneConst& sc) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(upload_hash_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, xyz, vel_in, pos, vel, id, key0,
                       next, head, n, ncells, tile_shift, sc);
    return hipGetLastError();
}

hipError_t launch_neighbors(hipStream_t st, int block, uint32_t grid, const StepArgs& a,
                            const uint32_t* offsets, uint32_t* out, int fill) {
    if (grid == 0) return hipSuccess;
    if (fill)
        hipLaunchKernelGGL(neighbors_kernel<1>, dim3(grid), dim3(block), 0, st, a, offsets, out);
    else
        hipLaunchKernelGGL(neighbors_kernel<0>, dim3(grid), dim3(block), 0, st, a, offsets, out);
    return hipGetLastError();
}

hipError_t launch_sorted_keys(hipStream_t st, int block, uint32_t ntiles, const float4* pos_s, uint32_t* skey,
                              const SceneConst* scenes, const uint2* tiles) {
    if (ntiles == 0) return hipSuccess;
    hipLaunchKernelGGL(sorted_keys_kernel, dim3(ntiles), dim3(block), 0, st, pos_s, skey, scenes, tiles);
    return hipGetLastError();
}

hipError_t launch_frame_reset(hipStream_t st, uint32_t* frame) {
    hipLaunchKernelGGL(frame_reset_kernel, dim3(1), dim3(64), 0, st, frame);
    return hipGetLastError();
}

hipError_t launch_fill_u32(hipStream_t st, uint32_t* p, uint32_t value, size_t count) {
    if (count == 0) return hipSuccess;
    const uint32_t g = blocks_for(count, 256) < 4096 ? blocks_for(count, 256) : 4096;
    hipLaunchKernelGGL(fill_u32_kernel, dim3(g), dim3(256), 0, st, p, value, count);
    return hipGetLastError();
}

hipError_t launch_unpermute3(hipStream_t st, uint32_t n, const float4* src, const uint32_t* id, float* out) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(unpermute3_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, src, id, out);
    return hipGetLastError();
}

hipError_t launch_copy_out(hipStream_t st, const uint32_t* src, size_t words, const uint32_t* flag, uint32_t* dst) {
    const size_t lanes = words / 4 > 64 ? words / 4 : 64;
    hipLaunchKernelGGL(copy_out_kernel, dim3(blocks_for(lanes, 256)), dim3(256), 0, st, src, words, flag, dst);
    return hipGetLastError();
}

hipError_t launch_read_small(hipStream_t st, uint32_t n, const float4* src4, const float* src1, const uint32_t* id,
                             const uint32_t* flag, float* dst) {
    if (n == 0 || n > kReadSmall) return hipErrorInvalidValue;
    hipLaunchKernelGGL(read_small_kernel, dim3(1), dim3(1024), 0, st, n, src4, src1, id, flag, dst);
    return hipGetLastError();
}

hipError_t launch_unpermute1(hipStream_t st, uint32_t n, const float* src, const uint32_t* id, float* out) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(unpermute1_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, src, id, out);
    return hipGetLastError();
}

hipError_t launch_copy_state(hipStream_t st, uint32_t n, float4* dp, float4* dv, uint32_t* di, const float4* sp,
                             const float4* sv, const uint32_t* si) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(copy_state_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, dp, dv, di, sp, sv, si);
    return hipGetLastError();
}

hipError_t launch_pack3(hipStream_t st, uint32_t n, const float* src, float4* dst) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(pack3_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, n, src, dst);
    return hipGetLastError();
}

}  // namespace sph
