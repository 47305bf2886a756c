// Hand-written reverse pass of one SPH step (gather form, no float atomics).
//
// Forward, per sorted particle i with neighbours j != i, r = x_i - x_j,
// d = |r|, hr = h - d, t = h^2 - d^2, P = p/rho^2, q = 1/rho:
//   rho_i = cD sum_j t^3                          (self included)
//   a_i   = cP sum (P_i+P_j) hr^2/d r + cV q_i sum q_j hr (v_j - v_i) + g
//   v' = v + dt a ; x~ = x + dt v' ; clamp(x~, v') -> (x', v'')
// Reverse, given xbar', vbar'' (output order = this step's sorted order):
//   adj_integrate: clamp masks, xbar~ , vbar' = vbar'' (or -e vbar'' where the
//                  velocity was reflected) + dt xbar~, abar = dt vbar'
//   adj_force:     xbar_i += sum cP(P_i+P_j)[phi da + (phi'/d)(da.r) r]
//                           + cV q_i q_j (psi'/d)(da.dv) r
//                  vbar_i += sum cV q_i q_j hr (abar_j - abar_i)
//                  Pbar_i = sum cP phi da.r ; qbar_i = sum cV q_j hr da.dv
//                  rhobar_i = Pbar_i (p' q^2 - 2 p q^3) - qbar_i q^2
//                  with da = abar_i - abar_j, dv = v_j - v_i, phi = hr^2/d,
//                  phi'/d = -t/d^3, psi' = -1; per-particle dL/dB and dL/dmu terms
//   adj_density:   xbar_i += sum -6 cD t^2 (rhobar_i + rhobar_j) r, then
//                  scatter both adjoints back to the step's input order, through
//                  adj_integrate of the step before
// Walls, per axis d (u_lo = (x_d - box_min_d)/h, u_hi = (box_max_d - x_d)/h;
// forward: rho_i += rho0 wall_rho(u), a_i,d += cW P_i (wall_j(u_lo) - wall_j(u_hi))):
//   adj_integrate: xbar_i,d += cW P_i abar_i,d (wall_j'(u_lo) + wall_j'(u_hi)) / h,
//                  and cW abar_i,d (wall_j(u_lo) - wall_j(u_hi)) in abar.w, where
//   adj_force      starts Pbar_i from it (the term involves particle i alone)
//   adj_density:   xbar_i,d += rhobar_i rho0 (wall_rho'(u_lo) - wall_rho'(u_hi)) / h
// Each kernel reads neighbour values written by the previous kernel only.
// adj_force and adj_density come in three forms with identical results: the
// neighbours' records gathered from global memory, each row's candidates
// staged in LDS by the wave first, or split over several waves (as the forward
// passes).
#include "sph_internal.hpp"

namespace sph {

namespace {

__device__ __forceinline__ void tile_span(uint32_t ntiles, uint32_t& t0, uint32_t& t1) {
    const uint32_t lb = xcd_block(blockIdx.x, gridDim.x);
    const uint32_t per = (ntiles + gridDim.x - 1) / gridDim.x;
    t0 = lb * per;
    t1 = t0 + per < ntiles ? t0 + per : ntiles;
}

// Visit the neighbours j != k the forward force pass visited, in its order.
template <class F>
__device__ __forceinline__ void for_each_neighbor(const AdjArgs& a, const SceneConst& sc, uint32_t k,
                                                  const float4& pi, F&& f) {
    const __amdgpu_buffer_rsrc_t rcs = buffer_of(a.cstart, a.ncells + 1u);
    const RowGeom g = row_geom(sc, pi.x, pi.y, pi.z);
#pragma unroll
    for (int row = 0; row < kRows; ++row) {
        uint32_t lo, hi;
        row_window(rcs, sc, g, row % 3 - 1, row / 3 - 1, lo, hi);
        uint32_t m = a.mask[(size_t)row * a.n + k];
        if (row == 4) {
            const uint32_t b = mask_bit(lo, hi, k);
            if (b < (uint32_t)kMaskBits) m &= ~(1u << b);
        }
        row_neighbors(
            lo, hi, m,
            [&](uint32_t j) {
                const float4 pj = a.pos_s[j];
                return j != k && dist2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z) < sc.h2;
            },
            f);
    }
}

// The reverse of clamp and symplectic Euler for output k of a step whose sorted
// state is x0, v0 and acceleration ac: xb, vb the adjoint of that output; writes
// what the step's force pass starts from.
// (wj, wd: the walls' differences and slopes at x0, adj_walls).
__device__ __forceinline__ void adj_walls(const SceneConst& sc, const float4& x0, float wj[3], float wd[3]) {
    const float xa[3] = {x0.x, x0.y, x0.z};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float ul = (xa[d] - sc.bmin[d]) * sc.inv_h, uh = (sc.wmax[d] - xa[d]) * sc.inv_h;
        wj[d] = wall_j(ul) - wall_j(uh);
        wd[d] = sc.inv_h * (wall_j_du(ul) + wall_j_du(uh));
    }
}
__device__ __forceinline__ void adj_integrate_one(const AdjArgs& a, const SceneConst& sc, uint32_t k, const float4& x0,
                                                  const float4& v0, const float4& ac, const float4& xb,
                                                  const float4& vb, const float wj[3], const float wd[3]) {
    const float xa[3] = {x0.x, x0.y, x0.z}, va[3] = {v0.x, v0.y, v0.z}, aa[3] = {ac.x, ac.y, ac.z};
    const float xba[3] = {xb.x, xb.y, xb.z}, vba[3] = {vb.x, vb.y, vb.z};
    float xo[3], vo[3], ab[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float v1 = va[d] + sc.dt * aa[d];
        const float xt = xa[d] + sc.dt * v1;
        float xbt = xba[d], vb1 = vba[d];
        if (xt < sc.lo[d]) {
            xbt = 0.0f;
            if (v1 < 0.0f) vb1 = -sc.e * vb1;
        } else if (xt > sc.hi[d]) {
            xbt = 0.0f;
            if (v1 > 0.0f) vb1 = -sc.e * vb1;
        }
        vb1 += sc.dt * xbt;
        xo[d] = xbt;
        vo[d] = vb1;
        ab[d] = sc.dt * vb1;
    }
    // Walls: their pressure term depends on this particle alone, so its
    // reverse (Pbar share in abar.w, xbar here) is elementwise.
    float pw = 0.0f;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        pw += sc.cW * ab[d] * wj[d];
        xo[d] += ((sc.cW * x0.w) * ab[d]) * wd[d];
    }
    a.xbar_o[k] = make_float4(xo[0], xo[1], xo[2], 0.0f);
    a.vbar_o[k] = make_float4(vo[0], vo[1], vo[2], 0.0f);
    a.abar[k] = make_float4(sc.scale_a * ab[0], sc.scale_a * ab[1], sc.scale_a * ab[2], sc.scale_a * pw);
}

// The last step of a segment (the others' is done by the density pass of the
// step after them).
__global__ void adj_integrate_kernel(AdjArgs a) {
    uint32_t t0, t1;
    tile_span(a.ntiles, t0, t1);
    for (uint32_t t = t0; t < t1; ++t) {
        const uint2 ti = tile_at(a.tiles, t);
        const SceneConst sc = scene_at(a.scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        if (k >= sc.p_end) continue;
        const float4 x0 = a.pos_s[k];
        float wj[3], wd[3];
        adj_walls(sc, x0, wj, wd);
        adj_integrate_one(a, sc, k, x0, a.vel_s[k], a.acc[k], a.xbar[k], a.vbar[k], wj, wd);
    }
}

// Per-particle sums of the adjoint force pass, without their constant factors
// (adj_finish_* apply those): g without cP, h without -cV q_i, Pb without cP,
// qb without cV; these four by scale_a, as abar is in memory.  Without the
// scale, seeds whose gradients were far inside the float range lost bits of
// their pairs' terms at its end (h = 0.0056, seeds of 1e-23: 1e-5).
struct AdjForceAcc {
    float gx, gy, gz, hx, hy, hz, Pb, qb, Ax, Ay, Az;
};

__device__ __forceinline__ float dot3(float ax, float ay, float az, float bx, float by, float bz) {
    return fmaf(az, bz, fmaf(ay, by, ax * bx));
}

// One neighbour's terms of the adjoint force pass (pos.w = p/rho^2, vel.w =
// 1/rho); vp = cV q_i / cP.  The passes are bound by this arithmetic: a wave
// walks each row for as long as its longest lane, some 58 pairs a lane where
// 32 count, at four cycles an instruction.  With multiply-adds and the sums'
// constants taken out it has 53 instructions where it had 78: staged force
// pass of 16 x 32k particles 72.1 -> 63.8 us, gathered of 7k 23.5 -> 21.0.
struct AdjFactors {
    float coefr, rx, ry, rz, pphi, dax, day, daz, w, dvx, dvy, dvz, phi, dar, dav;
};
__device__ __forceinline__ AdjFactors adj_force_factors(const SceneConst& sc, const float4& pi, const float4& vi,
                                                        const float4& abi, float vp, const float4& pj,
                                                        const float4& vj, const float4& abj) {
    AdjFactors f;
    f.rx = pi.x - pj.x, f.ry = pi.y - pj.y, f.rz = pi.z - pj.z;
    const float d2 = dist2(f.rx, f.ry, f.rz);
    const float inv_r = d2 > 0.0f ? __builtin_amdgcn_rsqf(d2) : 0.0f;
    const float hr = fmaf(-d2, inv_r, sc.h);
    const float tt = sc.h2 - d2;
    f.phi = hr * hr * inv_r;
    const float dphi_r = -tt * inv_r * inv_r * inv_r;
    f.w = hr * vj.w;
    f.dax = abi.x - abj.x, f.day = abi.y - abj.y, f.daz = abi.z - abj.z;
    f.dvx = vj.x - vi.x, f.dvy = vj.y - vi.y, f.dvz = vj.z - vi.z;
    const float PP = pi.w + pj.w;
    f.dar = dot3(f.dax, f.day, f.daz, f.rx, f.ry, f.rz);
    f.dav = dot3(f.dax, f.day, f.daz, f.dvx, f.dvy, f.dvz);
    f.coefr = fmaf(PP * dphi_r, f.dar, -((vp * vj.w) * inv_r) * f.dav);
    f.pphi = PP * f.phi;
    return f;
}
__device__ __forceinline__ void adj_force_pair(const SceneConst& sc, const float4& pi, const float4& vi,
                                               const float4& abi, float vp, const float4& pj, const float4& vj,
                                               const float4& abj, AdjForceAcc& c) {
    const AdjFactors f = adj_force_factors(sc, pi, vi, abi, vp, pj, vj, abj);
    c.gx = fmaf(f.coefr, f.rx, fmaf(f.pphi, f.dax, c.gx));
    c.gy = fmaf(f.coefr, f.ry, fmaf(f.pphi, f.day, c.gy));
    c.gz = fmaf(f.coefr, f.rz, fmaf(f.pphi, f.daz, c.gz));
    c.hx = fmaf(f.w, f.dax, c.hx);
    c.hy = fmaf(f.w, f.day, c.hy);
    c.hz = fmaf(f.w, f.daz, c.hz);
    c.Pb = fmaf(f.phi, f.dar, c.Pb);
    c.qb = fmaf(f.w, f.dav, c.qb);
    c.Ax = fmaf(f.w, f.dvx, c.Ax);
    c.Ay = fmaf(f.w, f.dvy, c.Ay);
    c.Az = fmaf(f.w, f.dvz, c.Az);
}

// Factor of the viscosity terms against the pressure terms' cP.
__device__ __forceinline__ float visc_ratio(const SceneConst& sc, const float4& vi) { return (sc.cV * vi.w) / sc.cP; }

// The sums' ends: the position adjoint ...
__device__ __forceinline__ float4 adj_finish_x(const SceneConst& sc, float4 xs, float gx, float gy, float gz) {
    const float c = sc.cP * sc.unscale_a;
    xs.x = fmaf(c, gx, xs.x); xs.y = fmaf(c, gy, xs.y); xs.z = fmaf(c, gz, xs.z);
    return xs;
}
// ... the velocity adjoint, ...
__device__ __forceinline__ float4 adj_finish_v(const SceneConst& sc, float4 vs, float qi, float hx, float hy, float hz) {
    const float cvq = sc.cV * qi * sc.unscale_a;
    vs.x = fmaf(-cvq, hx, vs.x); vs.y = fmaf(-cvq, hy, vs.y); vs.z = fmaf(-cvq, hz, vs.z);
    return vs;
}
// ... the dL/dmu term, ...
__device__ __forceinline__ float adj_finish_mu(const SceneConst& sc, float qi, const float4& abi, float Ax, float Ay,
                                               float Az) {
    return sc.cP * qi * (abi.x * Ax + abi.y * Ay + abi.z * Az) * sc.unscale_a;
}
// ... and the EOS reverse: the density adjoint (by scale_r) and the dL/dB term.
__device__ __forceinline__ float adj_finish_rho(const SceneConst& sc, float rho, float qi, const float4& abi, float Pbs,
                                                float qbs, float& rhobar) {
    const float Pb = fmaf(sc.cP * sc.unscale_a, Pbs, abi.w * sc.unscale_a), qb = sc.cV * sc.unscale_a * qbs;
    // EOS derivatives (clamped Tait, exponent 7).
    const float x = rho * sc.inv_rho0;
    const float x2 = x * x, x4 = x2 * x2, x6 = x4 * x2, x7 = x6 * x;
    const float praw = sc.B * (x7 - 1.0f);
    const float sgn = praw < 0.0f ? (sc.attractive ? sc.attr : 0.0f) : 1.0f;
    const float p = praw * sgn;
    const float dp_drho = sgn * sc.B * 7.0f * x6 * sc.inv_rho0;
    const float dp_dB = sgn * (x7 - 1.0f);
    rhobar = sc.scale_r * (Pb * (dp_drho * qi * qi - 2.0f * p * qi * qi * qi) - qb * qi * qi);
    return Pb * qi * qi * dp_dB;
}

// The stores of particle k; returns its (dL/dB, dL/dmu) terms.
__device__ __forceinline__ double2 adj_force_finish(const AdjArgs& a, const SceneConst& sc, uint32_t k,
                                                    const float4& vi, const float4& abi, const AdjForceAcc& c) {
    float rhobar;
    const float bpart = adj_finish_rho(sc, a.rho[k], vi.w, abi, c.Pb, c.qb, rhobar);
    a.rhobar[k] = rhobar;
    const float mpart = adj_finish_mu(sc, vi.w, abi, c.Ax, c.Ay, c.Az);
    a.xbar[k] = adj_finish_x(sc, a.xbar[k], c.gx, c.gy, c.gz);
    a.vbar[k] = adj_finish_v(sc, a.vbar[k], vi.w, c.hx, c.hy, c.hz);
    return make_double2((double)bpart, (double)mpart);
}

// One particle of the adjoint force pass; returns its (dL/dB, dL/dmu) terms.
__device__ __forceinline__ double2 adj_force_one(const AdjArgs& a, const SceneConst& sc, uint32_t k) {
    const float4 pi = a.pos_s[k], vi = a.vel_s[k], abi = a.abar[k];
    AdjForceAcc c = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const float vp = visc_ratio(sc, vi);
    for_each_neighbor(a, sc, k, pi, [&](uint32_t j) {
        adj_force_pair(sc, pi, vi, abi, vp, a.pos_s[j], a.vel_s[j], a.abar[j], c);
    });
    return adj_force_finish(a, sc, k, vi, abi, c);
}

// Staged forms of the adjoint force and density passes: the forward passes'
// staging applied to the reverse walk.  All nine windows and masks are formed
// first; per row the wave copies the union of its lanes' windows into its LDS
// slot (coalesced) and every lane walks its own mask over the slot; a wider
// union is read from global memory.  Same neighbours, same order, same
// arithmetic: the gathered kernels' results bit for bit.  Every lane of the
// wave takes part; inactive lanes have empty windows and store nothing.
constexpr uint32_t kStageA = 96;
static_assert(kStageA <= 128, "the copy into a slot takes two records per lane");
struct AdjForceSlot {
    float4 pos[kStageA];
    float4 vel[kStageA];
    float4 abar[kStageA];
};
struct AdjDensitySlot {
    float4 pos[kStageA];
    float rb[kStageA];
};

struct AdjRows {
    uint32_t lo[kRows], hi[kRows], mk[kRows];
};

__device__ __forceinline__ void adj_rows(const AdjArgs& a, const SceneConst& sc, uint32_t k, bool active,
                                         const float4& pi, AdjRows& r) {
    const __amdgpu_buffer_rsrc_t rcs = buffer_of(a.cstart, a.ncells + 1u);
    const RowGeom g = row_geom(sc, pi.x, pi.y, pi.z);
#pragma unroll
    for (int row = 0; row < kRows; ++row) {
        row_window(rcs, sc, g, row % 3 - 1, row / 3 - 1, r.lo[row], r.hi[row]);
        r.mk[row] = active ? a.mask[(size_t)row * a.n + k] : 0u;
        if (!active) r.lo[row] = r.hi[row] = 0u;
    }
    const uint32_t b = mask_bit(r.lo[4], r.hi[4], k);
    if (active && b < (uint32_t)kMaskBits) r.mk[4] &= ~(1u << b);
}

// kv: a particle of the tile (the lane's own when active) whose values the
// inactive lanes load in place of theirs.
__device__ __forceinline__ double2 adj_force_one_staged(const AdjArgs& a, const SceneConst& sc, uint32_t k,
                                                        bool active, uint32_t kv, AdjForceSlot& slot) {
    const float4 pi = a.pos_s[kv], vi = a.vel_s[kv], abi = a.abar[kv];
    AdjRows r;
    adj_rows(a, sc, k, active, pi, r);
    AdjForceAcc c = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const float vp = visc_ratio(sc, vi);
    const uint32_t lane = threadIdx.x & 63u;
#pragma unroll
    for (int row = 0; row < kRows; ++row) {
        const bool has = r.hi[row] > r.lo[row];
        const uint32_t ulo = wave_umin(has ? r.lo[row] : 0xffffffffu);
        const uint32_t uhi = wave_umax(has ? r.hi[row] : 0u);
        if (ulo >= uhi) continue;
        if (uhi - ulo <= kStageA) {
            // Both halves of the copy (a union holds at most 2 x 64 records)
            // are loaded before either is stored, so their latencies overlap.
            const uint32_t span = uhi - ulo;
            const bool c0 = lane < span, c1 = lane + 64u < span;
            float4 p0 = make_float4(0.f, 0.f, 0.f, 0.f), v0 = p0, b0 = p0, p1 = p0, v1 = p0, b1 = p0;
            if (c0) {
                p0 = a.pos_s[ulo + lane];
                v0 = a.vel_s[ulo + lane];
                b0 = a.abar[ulo + lane];
            }
            if (c1) {
                p1 = a.pos_s[ulo + lane + 64u];
                v1 = a.vel_s[ulo + lane + 64u];
                b1 = a.abar[ulo + lane + 64u];
            }
            if (c0) {
                slot.pos[lane] = p0;
                slot.vel[lane] = v0;
                slot.abar[lane] = b0;
            }
            if (c1) {
                slot.pos[lane + 64u] = p1;
                slot.vel[lane + 64u] = v1;
                slot.abar[lane + 64u] = b1;
            }
            wave_lds_sync();
            const uint32_t e0 = row_first(r.lo[row], r.hi[row]) - ulo;
            row_neighbors_from(
                r.lo[row], r.hi[row], r.mk[row],
                [&](uint32_t j) {
                    const float4 pj = slot.pos[j - ulo];
                    return j != k && dist2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z) < sc.h2;
                },
                [&](uint32_t j) {
                    const uint32_t e = j - ulo;
                    adj_force_pair(sc, pi, vi, abi, vp, slot.pos[e], slot.vel[e], slot.abar[e], c);
                },
                [&](uint32_t i) {
                    adj_force_pair(sc, pi, vi, abi, vp, slot.pos[e0 + i], slot.vel[e0 + i], slot.abar[e0 + i], c);
                });
            wave_lds_sync();
        } else {
            row_neighbors(
                r.lo[row], r.hi[row], r.mk[row],
                [&](uint32_t j) {
                    const float4 pj = a.pos_s[j];
                    return j != k && dist2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z) < sc.h2;
                },
                [&](uint32_t j) { adj_force_pair(sc, pi, vi, abi, vp, a.pos_s[j], a.vel_s[j], a.abar[j], c); });
        }
    }
    return active ? adj_force_finish(a, sc, k, vi, abi, c) : make_double2(0.0, 0.0);
}

// Adds the terms of a tile of blockDim.x particles to its running sums, in
// the order of a tree over the lanes (halves of the tile first): its halves
// above a wave by wave 0, the wave by shuffles.  One barrier, where the tree
// in LDS had nine (the second one only for a block with another tile to go).
__device__ __forceinline__ void add_wave_terms(double2* __restrict__ acc, double x, double y) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        x += __shfl_down(x, o, 64);
        y += __shfl_down(y, o, 64);
    }
    if ((threadIdx.x & 63u) == 0u) {
        double2 sum = *acc;
        sum.x += x;
        sum.y += y;
        *acc = sum;
    }
}
__device__ __forceinline__ void add_tile_terms(const AdjArgs& a, uint32_t t, double2 part, double2* red) {
    red[threadIdx.x] = part;
    __syncthreads();
    if (threadIdx.x < 64u) {
        double x = part.x, y = part.y;
        const uint32_t i = threadIdx.x;
        if (blockDim.x == 256u) {
            x = (x + red[i + 128u].x) + (red[i + 64u].x + red[i + 192u].x);
            y = (y + red[i + 128u].y) + (red[i + 64u].y + red[i + 192u].y);
        } else if (blockDim.x == 128u) {
            x += red[i + 64u].x;
            y += red[i + 64u].y;
        }
        add_wave_terms(a.tile_acc + t, x, y);
    }
    __syncthreads();
}

// Eight waves per SIMD (64 VGPRs, three spilled): the backward pass was
// 3 % faster than without the bound (47.0 against 48.3 ms, 16 x 32k
// particles x 200 steps, with the walls' reverse still in this kernel).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) void adj_force_kernel(AdjArgs a) {
    uint32_t t0, t1;
    tile_span(a.ntiles, t0, t1);
    // Per-tile (dL/dB, dL/dmu) of this step, reduced in double in a fixed
    // tree and added to the tile's running sum: deterministic, no atomics.
    __shared__ double2 red[256];
    for (uint32_t t = t0; t < t1; ++t) {
        const uint2 ti = tile_at(a.tiles, t);
        const SceneConst sc = scene_at(a.scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        double2 part = make_double2(0.0, 0.0);
        if (k < sc.p_end) part = adj_force_one(a, sc, k);
        add_tile_terms(a, t, part, red);
    }
}

// adj_force_kernel with the rows staged in LDS (4.5 KB per wave).
__global__ __launch_bounds__(256) void adj_force_staged_kernel(AdjArgs a) {
    uint32_t t0, t1;
    tile_span(a.ntiles, t0, t1);
    __shared__ double2 red[256];
    __shared__ AdjForceSlot s_slot[256 / 64];
    AdjForceSlot& slot = s_slot[threadIdx.x >> 6];
    for (uint32_t t = t0; t < t1; ++t) {
        const uint2 ti = tile_at(a.tiles, t);
        const SceneConst sc = scene_at(a.scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        const bool active = k < sc.p_end;
        const double2 part = adj_force_one_staged(a, sc, k, active, active ? k : ti.y, slot);
        add_tile_terms(a, t, part, red);
    }
}

__device__ __forceinline__ float adj_density_factor(const SceneConst& sc, float rx, float ry, float rz, float rbi,
                                                    float rbj) {
    const float tt = sc.h2 - dist2(rx, ry, rz);
    return (tt * tt) * (rbi + rbj);
}
// One neighbour's term of the adjoint density pass, without its factor -6 cD
// (adj_scatter applies it), by scale_r as the density adjoint is.
__device__ __forceinline__ void adj_density_pair(const SceneConst& sc, const float4& pi, float rbi, const float4& pj,
                                                 float rbj, float& gx, float& gy, float& gz) {
    const float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
    const float s = adj_density_factor(sc, rx, ry, rz, rbi, rbj);
    gx = fmaf(s, rx, gx);
    gy = fmaf(s, ry, gy);
    gz = fmaf(s, rz, gz);
}

// The walls' density reverse, and the adjoints of particle k scattered back
// to the step's input order: the step before's output, whose integration is
// reversed right away where that step is on the tape (a pass of its own read
// and wrote 64 bytes a particle more and took 13 us for 16 x 32k particles, 5
// for 7k).
struct AdjMove {
    uint32_t src;
    float4 xs, vs, x0, v0, ac;
};
__device__ __forceinline__ AdjMove adj_move(const AdjArgs& a, uint32_t k) {
    AdjMove m;
    m.src = a.perm[k];
    m.xs = a.xbar[k];
    m.vs = a.vbar[k];
    m.x0 = m.v0 = m.ac = make_float4(0.f, 0.f, 0.f, 0.f);
    if (a.pos_p) {
        m.x0 = a.pos_p[m.src];
        m.v0 = a.vel_p[m.src];
        m.ac = a.acc_p[m.src];
    }
    return m;
}
__device__ __forceinline__ void adj_density_walls(const SceneConst& sc, const float4& pi, float rbi, float gw[3]) {
    const float pk[3] = {pi.x, pi.y, pi.z};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float ul = (pk[d] - sc.bmin[d]) * sc.inv_h, uh = (sc.wmax[d] - pk[d]) * sc.inv_h;
        gw[d] = (rbi * sc.unscale_r * sc.rho0) * (sc.inv_h * (wall_rho_du(ul) - wall_rho_du(uh)));
    }
}
__device__ __forceinline__ void adj_scatter(const AdjArgs& a, const SceneConst& sc, AdjMove& m, float gx, float gy,
                                            float gz, const float gw[3], const float wj[3], const float wd[3]) {
    const float cg = -6.0f * sc.cD * sc.unscale_r;
    m.xs.x += fmaf(cg, gx, gw[0]);
    m.xs.y += fmaf(cg, gy, gw[1]);
    m.xs.z += fmaf(cg, gz, gw[2]);
    if (a.pos_p) {
        adj_integrate_one(a, sc, m.src, m.x0, m.v0, m.ac, m.xs, m.vs, wj, wd);
    } else {
        a.xbar_o[m.src] = m.xs;
        a.vbar_o[m.src] = m.vs;
    }
}
__device__ __forceinline__ void adj_density_finish(const AdjArgs& a, const SceneConst& sc, uint32_t k,
                                                   const float4& pi, float rbi, float gx, float gy, float gz) {
    float gw[3], wj[3], wd[3];
    adj_density_walls(sc, pi, rbi, gw);
    AdjMove m = adj_move(a, k);
    adj_walls(sc, m.x0, wj, wd);
    adj_scatter(a, sc, m, gx, gy, gz, gw, wj, wd);
}

// adj_density_kernel with the rows staged in LDS (1.9 KB per wave).
// Eight waves per SIMD: the bound fits it in 64 VGPRs (25 SGPRs in lanes).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) void adj_density_staged_kernel(AdjArgs a) {
    uint32_t t0, t1;
    tile_span(a.ntiles, t0, t1);
    __shared__ AdjDensitySlot s_slot[256 / 64];
    AdjDensitySlot& slot = s_slot[threadIdx.x >> 6];
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t t = t0; t < t1; ++t) {
        const uint2 ti = tile_at(a.tiles, t);
        const SceneConst sc = scene_at(a.scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        const bool active = k < sc.p_end;
        const uint32_t kv = active ? k : ti.y;
        const float4 pi = a.pos_s[kv];
        const float rbi = a.rhobar[kv];
        AdjRows r;
        adj_rows(a, sc, k, active, pi, r);
        float gx = 0, gy = 0, gz = 0;
#pragma unroll
        for (int row = 0; row < kRows; ++row) {
            const bool has = r.hi[row] > r.lo[row];
            const uint32_t ulo = wave_umin(has ? r.lo[row] : 0xffffffffu);
            const uint32_t uhi = wave_umax(has ? r.hi[row] : 0u);
            if (ulo >= uhi) continue;
            if (uhi - ulo <= kStageA) {
                // Both halves of the copy are loaded before either is stored.
                const uint32_t span = uhi - ulo;
                const bool c0 = lane < span, c1 = lane + 64u < span;
                float4 p0 = make_float4(0.f, 0.f, 0.f, 0.f), p1 = p0;
                float q0 = 0.f, q1 = 0.f;
                if (c0) {
                    p0 = a.pos_s[ulo + lane];
                    q0 = a.rhobar[ulo + lane];
                }
                if (c1) {
                    p1 = a.pos_s[ulo + lane + 64u];
                    q1 = a.rhobar[ulo + lane + 64u];
                }
                if (c0) {
                    slot.pos[lane] = p0;
                    slot.rb[lane] = q0;
                }
                if (c1) {
                    slot.pos[lane + 64u] = p1;
                    slot.rb[lane + 64u] = q1;
                }
                wave_lds_sync();
                const uint32_t e0 = row_first(r.lo[row], r.hi[row]) - ulo;
                row_neighbors_from(
                    r.lo[row], r.hi[row], r.mk[row],
                    [&](uint32_t j) {
                        const float4 pj = slot.pos[j - ulo];
                        return j != k && dist2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z) < sc.h2;
                    },
                    [&](uint32_t j) {
                        const uint32_t e = j - ulo;
                        adj_density_pair(sc, pi, rbi, slot.pos[e], slot.rb[e], gx, gy, gz);
                    },
                    [&](uint32_t i) { adj_density_pair(sc, pi, rbi, slot.pos[e0 + i], slot.rb[e0 + i], gx, gy, gz); });
                wave_lds_sync();
            } else {
                row_neighbors(
                    r.lo[row], r.hi[row], r.mk[row],
                    [&](uint32_t j) {
                        const float4 pj = a.pos_s[j];
                        return j != k && dist2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z) < sc.h2;
                    },
                    [&](uint32_t j) { adj_density_pair(sc, pi, rbi, a.pos_s[j], a.rhobar[j], gx, gy, gz); });
            }
        }
        if (active) adj_density_finish(a, sc, k, pi, rbi, gx, gy, gz);
    }
}

__global__ void adj_density_kernel(AdjArgs a) {
    uint32_t t0, t1;
    tile_span(a.ntiles, t0, t1);
    for (uint32_t t = t0; t < t1; ++t) {
        const uint2 ti = tile_at(a.tiles, t);
        const SceneConst sc = scene_at(a.scenes, ti.x);
        const uint32_t k = ti.y + threadIdx.x;
        if (k >= sc.p_end) continue;
        const float4 pi = a.pos_s[k];
        const float rbi = a.rhobar[k];
        float gx = 0, gy = 0, gz = 0;
        for_each_neighbor(a, sc, k, pi, [&](uint32_t j) {
            adj_density_pair(sc, pi, rbi, a.pos_s[j], a.rhobar[j], gx, gy, gz);
        });
        adj_density_finish(a, sc, k, pi, rbi, gx, gy, gz);
    }
}

// ------------------------------------------------------------- split form
//
// As in the forward step, a small handle's pass lasts as long as one wave's
// chain (7k particles, 113 waves: force 21.0 us, density 13.5; in this form
// 7.8 and 5.5, bound by the latency of the windows, the gathers and the
// in-order sums one after the other).  Force: nine
// waves per 64 particles list the neighbours, one row each, from the step's
// masks; eight of them gather the pairs of kAdjRound list entries and leave
// their factors in LDS; then three waves add them in list order, each its
// share of the sums, and finish that share.  The density pass takes the list
// over, four waves per 64 particles.  The sums' order and arithmetic are the
// other forms', bit for bit.
constexpr int kAdjRound = 16;  // two blocks of 77 KB fit a CU

struct AdjForceShared {
    float4 f1[kAdjRound][kSplitTile];    // coefr, r
    float4 f2[kAdjRound][kSplitTile];    // (P_i + P_j) phi, da
    float4 f3[kAdjRound][kSplitTile];    // w, dv
    float2 f4[kAdjRound][kSplitTile];    // phi, da.r
    float f5[kAdjRound][kSplitTile];     // da.dv
    uint16_t id[kListMax][kSplitTile];   // the neighbours, without the particle itself
    uint32_t count[3][kSplitTile];       // neighbours per row, one byte a row
};
static_assert(2 * sizeof(AdjForceShared) <= 160 * 1024, "two blocks per CU");

__global__ __launch_bounds__(64 * kRows) void adj_force_split_kernel(AdjArgs a) {
    __shared__ AdjForceShared sh;
    const __amdgpu_buffer_rsrc_t rpos = buffer_of(a.pos_s, a.n);
    const __amdgpu_buffer_rsrc_t rvel = buffer_of(a.vel_s, a.n);
    const __amdgpu_buffer_rsrc_t rab = buffer_of((const float4*)a.abar, a.n);
    const __amdgpu_buffer_rsrc_t rcs = buffer_of(a.cstart, a.ncells + 1u);
    const uint2 ti = tile_at(a.tiles, xcd_block(blockIdx.x, gridDim.x));
    const SceneConst sc = scene_at(a.scenes, ti.x);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t k = ti.y + lane;
    const bool active = k < sc.p_end;
    // Zeros past the buffers' ends.
    const float4 pi = load4(rpos, k << 4), vi = load4(rvel, k << 4), abi = load4(rab, k << 4);
    uint32_t m = active ? a.mask[(size_t)w * a.n + k] : 0u;
    // What the finishing waves add their sums to.
    float4 own = make_float4(0.f, 0.f, 0.f, 0.f);
    if (active) {
        if (w == 0) own = a.xbar[k];
        if (w == 1) own = a.vbar[k];
        if (w == 2) own.x = a.rho[k];
    }
    uint32_t lo, hi;
    split_window(rcs, sc, pi, w % 3 - 1, w / 3 - 1, lo, hi);
    if (!active) lo = hi = 0u;
    if (w == 4 && active) m = without_self(m, lo, hi, k, 0u);
    // The mask's slots as ascending bits, and the 32 before them, tested again.
    const uint32_t span = mask_span(lo, hi);
    const uint32_t j1 = row_first(lo, hi, 2u), j0 = row_first(lo, hi);
    const uint32_t r = mask_ascending(m, span, 0u);
    uint32_t rh = 0u;
    for (uint32_t j = j1; j < j0; ++j) {
        const float4 pj = load4(rpos, j << 4);
        if (j != k && dist2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z) < sc.h2) rh |= 1u << (j - j1);
    }
    const uint32_t cnt = span > 64u ? kRowOver : (uint32_t)__popc(r) + (uint32_t)__popc(rh);
    reinterpret_cast<uint8_t*>(sh.count)[(((uint32_t)w >> 2) * kSplitTile + lane) * 4u + ((uint32_t)w & 3u)] = (uint8_t)cnt;
    __syncthreads();
    uint32_t at = 0u, total = 0u;
#pragma unroll
    for (int g = 0; g < 3; ++g) {
        const uint32_t c = sh.count[g][lane];
        const uint32_t before = w >= 4 * g + 4 ? 0xffffffffu : w > 4 * g ? (1u << (8 * (w - 4 * g))) - 1u : 0u;
        at = __builtin_amdgcn_sad_u8(c & before, 0u, at);
        total = __builtin_amdgcn_sad_u8(g == 2 ? c & 0xffu : c, 0u, total);
    }
    const uint32_t most = wave_umax(total);  // the same in every wave
    if (most > kListMax) {
        if (w == 0 && active) {
            a.ncount[k] = kListOver;
            a.part[k] = adj_force_one(a, sc, k);
        }
        return;
    }
    for (uint32_t q = rh; q; q &= q - 1u) sh.id[at++][lane] = (uint16_t)(j1 + (uint32_t)__builtin_ctz(q));
    for (uint32_t q = r; q; q &= q - 1u) sh.id[at++][lane] = (uint16_t)(j0 + (uint32_t)__builtin_ctz(q));
    __syncthreads();
    const float vp = visc_ratio(sc, vi);
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f, s4 = 0.f, s5 = 0.f;
    for (uint32_t first = 0u;; first += kAdjRound) {
        if (w < 8) {
            const uint32_t e = 2u * (uint32_t)w;
            if (__ballot(total > first + e) != 0u) {
                float4 pj[2], vj[2], bj[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const uint32_t i = first + e + (uint32_t)u;
                    const uint32_t j = i < total ? (uint32_t)sh.id[i][lane] : k;  // past the list: not added
                    pj[u] = load4(rpos, j << 4);
                    vj[u] = load4(rvel, j << 4);
                    bj[u] = load4(rab, j << 4);
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const AdjFactors f = adj_force_factors(sc, pi, vi, abi, vp, pj[u], vj[u], bj[u]);
                    sh.f1[e + (uint32_t)u][lane] = make_float4(f.coefr, f.rx, f.ry, f.rz);
                    sh.f2[e + (uint32_t)u][lane] = make_float4(f.pphi, f.dax, f.day, f.daz);
                    sh.f3[e + (uint32_t)u][lane] = make_float4(f.w, f.dvx, f.dvy, f.dvz);
                    sh.f4[e + (uint32_t)u][lane] = make_float2(f.phi, f.dar);
                    sh.f5[e + (uint32_t)u][lane] = f.dav;
                }
            }
        } else if (first == 0u && active) {
            // The list, for the density pass.
            a.ncount[k] = total;
            for (uint32_t q = 0; 4u * q < total; ++q)
                reinterpret_cast<uint2*>(a.nlist)[(size_t)q * a.n + k] =
                    make_uint2(sh.id[4u * q][lane] | ((uint32_t)sh.id[4u * q + 1u][lane] << 16),
                               sh.id[4u * q + 2u][lane] | ((uint32_t)sh.id[4u * q + 3u][lane] << 16));
        }
        __syncthreads();
        const uint32_t left = total > first ? min(total - first, (uint32_t)kAdjRound) : 0u;
        if (w == 0) {
#pragma unroll 4
            for (uint32_t i = 0; i < left; ++i) {
                const float4 f1 = sh.f1[i][lane], f2 = sh.f2[i][lane];
                s0 = fmaf(f1.x, f1.y, fmaf(f2.x, f2.y, s0));
                s1 = fmaf(f1.x, f1.z, fmaf(f2.x, f2.z, s1));
                s2 = fmaf(f1.x, f1.w, fmaf(f2.x, f2.w, s2));
            }
        } else if (w == 1) {
#pragma unroll 4
            for (uint32_t i = 0; i < left; ++i) {
                const float4 f2 = sh.f2[i][lane], f3 = sh.f3[i][lane];
                s0 = fmaf(f3.x, f2.y, s0);
                s1 = fmaf(f3.x, f2.z, s1);
                s2 = fmaf(f3.x, f2.w, s2);
                s3 = fmaf(f3.x, f3.y, s3);
                s4 = fmaf(f3.x, f3.z, s4);
                s5 = fmaf(f3.x, f3.w, s5);
            }
        } else if (w == 2) {
#pragma unroll 4
            for (uint32_t i = 0; i < left; ++i) {
                const float2 f4 = sh.f4[i][lane];
                s0 = fmaf(f4.x, f4.y, s0);
                s1 = fmaf(sh.f3[i][lane].x, sh.f5[i][lane], s1);
            }
        }
        if (most <= first + (uint32_t)kAdjRound) break;
        __syncthreads();
    }
    if (!active) return;
    double* const part = reinterpret_cast<double*>(a.part + k);
    if (w == 0) a.xbar[k] = adj_finish_x(sc, own, s0, s1, s2);
    if (w == 1) {
        a.vbar[k] = adj_finish_v(sc, own, vi.w, s0, s1, s2);
        part[1] = (double)adj_finish_mu(sc, vi.w, abi, s3, s4, s5);
    }
    if (w == 2) {
        float rhobar;
        part[0] = (double)adj_finish_rho(sc, own.x, vi.w, abi, s0, s1, rhobar);
        a.rhobar[k] = rhobar;
    }
}

constexpr uint32_t kAdjDensityRound = 32;
constexpr int kAdjDensityWaves = 4;
constexpr int kAdjPerWave = (int)kAdjDensityRound / kAdjDensityWaves;

struct AdjDensityShared {
    float4 f[kAdjDensityRound][kSplitTile];  // s, r
    float gw[3][kSplitTile];                 // the walls' density term
    float wj[3][kSplitTile], wd[3][kSplitTile];
};

__global__ __launch_bounds__(64 * kAdjDensityWaves) void adj_density_split_kernel(AdjArgs a) {
    __shared__ AdjDensityShared sh;
    const __amdgpu_buffer_rsrc_t rpos = buffer_of(a.pos_s, a.n);
    const __amdgpu_buffer_rsrc_t rrb = buffer_of((const float*)a.rhobar, a.n);
    const __amdgpu_buffer_rsrc_t rl = buffer_of((const uint16_t*)a.nlist, kListMax * a.n);
    const uint2 ti = tile_at(a.tiles, xcd_block(blockIdx.x, gridDim.x));
    const SceneConst sc = scene_at(a.scenes, ti.x);
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t k = ti.y + lane;
    const bool active = k < sc.p_end;
    // Entries past a list's end hold any index; their pairs are not added.
    auto ids = [&](uint32_t q) { return __builtin_amdgcn_raw_buffer_load_b64(rl, (int)((q * a.n + k) << 3), 0, 0); };
    u32x2 q0 = ids(2u * (uint32_t)w), q1 = ids(2u * (uint32_t)w + 1u);
    const float4 pi = load4(rpos, k << 4);
    const float rbi = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rrb, (int)(k << 2), 0, 0));
    const uint32_t count = active ? a.ncount[k] : 0u;
    float4 pj[kAdjPerWave];
    float rj[kAdjPerWave];
    auto gather = [&]() {
        const uint32_t j[kAdjPerWave] = {q0.x & 0xffffu, q0.x >> 16, q0.y & 0xffffu, q0.y >> 16,
                                         q1.x & 0xffffu, q1.x >> 16, q1.y & 0xffffu, q1.y >> 16};
#pragma unroll
        for (int u = 0; u < kAdjPerWave; ++u) {
            pj[u] = load4(rpos, j[u] << 4);
            rj[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rrb, (int)(j[u] << 2), 0, 0));
        }
    };
    gather();  // before the counts are known: any index stays inside the buffers' bounds checks
    AdjMove mv;
    if (w == 0 && active) mv = adj_move(a, k);
    if (w == 3 && ((ti.y - sc.p_begin) & 255u) == 0u) {
        // The step's terms of 256 particles into their tile's running sums,
        // added in add_tile_terms' order.
        double2 p[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            p[i] = make_double2(0.0, 0.0);
            if (k + 64u * i < sc.p_end) p[i] = a.part[k + 64u * i];
        }
        double x = (p[0].x + p[2].x) + (p[1].x + p[3].x), y = (p[0].y + p[2].y) + (p[1].y + p[3].y);
        add_wave_terms(a.tile_acc + (a.tile_first[ti.x] + ((ti.y - sc.p_begin) >> 8)), x, y);
    }
    if (__ballot(count > kListMax) != 0u) {  // the same in every wave
        if (w == 0 && active) {
            float gx = 0.f, gy = 0.f, gz = 0.f;
            for_each_neighbor(a, sc, k, pi, [&](uint32_t j) {
                adj_density_pair(sc, pi, rbi, a.pos_s[j], a.rhobar[j], gx, gy, gz);
            });
            adj_density_finish(a, sc, k, pi, rbi, gx, gy, gz);
        }
        return;
    }
    float gx = 0.f, gy = 0.f, gz = 0.f;
    for (uint32_t first = 0u;; first += kAdjDensityRound) {
        if (__ballot(count > first + (uint32_t)(kAdjPerWave * w)) != 0u) {
            if (first != 0u) {
                q0 = ids(first / 4u + 2u * (uint32_t)w);
                q1 = ids(first / 4u + 2u * (uint32_t)w + 1u);
                gather();
            }
#pragma unroll
            for (int u = 0; u < kAdjPerWave; ++u) {
                const float rx = pi.x - pj[u].x, ry = pi.y - pj[u].y, rz = pi.z - pj[u].z;
                sh.f[kAdjPerWave * w + u][lane] =
                    make_float4(adj_density_factor(sc, rx, ry, rz, rbi, rj[u]), rx, ry, rz);
            }
        }
        if (first == 0u && active) {
            float t[3], u[3];
            if (w == 1) {
                adj_density_walls(sc, pi, rbi, t);
#pragma unroll
                for (int d = 0; d < 3; ++d) sh.gw[d][lane] = t[d];
            } else if (w == 2 && a.pos_p) {
                adj_walls(sc, a.pos_p[a.perm[k]], t, u);
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    sh.wj[d][lane] = t[d];
                    sh.wd[d][lane] = u[d];
                }
            }
        }
        __syncthreads();
        const uint32_t left = count > first ? min(count - first, kAdjDensityRound) : 0u;
        if (w == 0) {
#pragma unroll 4
            for (uint32_t i = 0; i < left; ++i) {
                const float4 f = sh.f[i][lane];
                gx = fmaf(f.x, f.y, gx);
                gy = fmaf(f.x, f.z, gy);
                gz = fmaf(f.x, f.w, gz);
            }
        }
        if (__ballot(count > first + kAdjDensityRound) == 0u) break;
        __syncthreads();
    }
    if (w != 0 || !active) return;
    const float gw[3] = {sh.gw[0][lane], sh.gw[1][lane], sh.gw[2][lane]};
    float wj[3] = {0.f, 0.f, 0.f}, wd[3] = {0.f, 0.f, 0.f};
    if (a.pos_p) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            wj[d] = sh.wj[d][lane];
            wd[d] = sh.wd[d][lane];
        }
    }
    adj_scatter(a, sc, mv, gx, gy, gz, gw, wj, wd);
}

// Per-scene totals of the per-tile accumulators: block s sums tiles
// [tile_first[s], tile_first[s + 1]) in a fixed order (threads stride, then
// a tree), so the result is the same run to run.
__global__ __launch_bounds__(256) void scene_tiles_kernel(const uint32_t* __restrict__ tile_first,
                                                          const double2* __restrict__ tile_acc,
                                                          double* __restrict__ acc_a, double* __restrict__ acc_b) {
    __shared__ double sa[256], sb[256];
    const uint32_t s = blockIdx.x;
    const uint32_t beg = tile_first[s], end = tile_first[s + 1];
    double va = 0.0, vb = 0.0;
    for (uint32_t i = beg + threadIdx.x; i < end; i += 256) {
        va += tile_acc[i].x;
        vb += tile_acc[i].y;
    }
    sa[threadIdx.x] = va;
    sb[threadIdx.x] = vb;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            sa[threadIdx.x] += sa[threadIdx.x + o];
            sb[threadIdx.x] += sb[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        acc_a[s] = sa[0];
        acc_b[s] = sb[0];
    }
}

__global__ void gather3_kernel(uint32_t n, const float* __restrict__ g, const uint32_t* __restrict__ id,
                               float4* __restrict__ out) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const size_t i = id[k];
    out[k] = make_float4(g[3 * i], g[3 * i + 1], g[3 * i + 2], 0.0f);
}

}  // namespace

hipError_t launch_adj_integrate(hipStream_t st, int block, uint32_t grid, const AdjArgs& a) {
    if (grid == 0) return hipSuccess;
    hipLaunchKernelGGL(adj_integrate_kernel, dim3(grid), dim3(block), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_adj_force(hipStream_t st, int block, uint32_t grid, const AdjArgs& a, int staged) {
    if (grid == 0) return hipSuccess;
    // __launch_bounds__(256), and whole waves whose terms add_tile_terms adds.
    if (block != 64 && block != 128 && block != 256) return hipErrorInvalidValue;
    if (staged)
        hipLaunchKernelGGL(adj_force_staged_kernel, dim3(grid), dim3(block), 0, st, a);
    else
        hipLaunchKernelGGL(adj_force_kernel, dim3(grid), dim3(block), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_adj_density(hipStream_t st, int block, uint32_t grid, const AdjArgs& a, int staged) {
    if (grid == 0) return hipSuccess;
    if (staged && (block > 256 || block % 64)) return hipErrorInvalidValue;
    if (staged)
        hipLaunchKernelGGL(adj_density_staged_kernel, dim3(grid), dim3(block), 0, st, a);
    else
        hipLaunchKernelGGL(adj_density_kernel, dim3(grid), dim3(block), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_adj_force_split(hipStream_t st, const AdjArgs& a) {
    if (a.ntiles == 0) return hipSuccess;
    hipLaunchKernelGGL(adj_force_split_kernel, dim3(a.ntiles), dim3(64 * kRows), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_adj_density_split(hipStream_t st, const AdjArgs& a) {
    if (a.ntiles == 0) return hipSuccess;
    hipLaunchKernelGGL(adj_density_split_kernel, dim3(a.ntiles), dim3(64 * kAdjDensityWaves), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_scene_tile_sums(hipStream_t st, uint32_t nscenes, const uint32_t* tile_first,
                                  const double2* tile_acc, double* acc_a, double* acc_b) {
    if (nscenes == 0) return hipSuccess;
    hipLaunchKernelGGL(scene_tiles_kernel, dim3(nscenes), dim3(256), 0, st, tile_first, tile_acc, acc_a, acc_b);
    return hipGetLastError();
}

hipError_t launch_gather3(hipStream_t st, uint32_t n, const float* g, const uint32_t* id, float4* out) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(gather3_kernel, dim3((n + 255) / 256), dim3(256), 0, st, n, g, id, out);
    return hipGetLastError();
}

}  // namespace sph
