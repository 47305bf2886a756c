// Autotuner: picks the block size of the density and force passes (and, of
// the radix sort, the gather's block and the keys per thread of the digit passes), whether density and force
// run as persistent blocks over tile queues and whether the force and
// density passes stage their rows in LDS, by timing each candidate
// with HIP events on the handle's own state.  The state is saved first and
// restored before every trial, so all candidates run the same steps.
// Results are cached per process, keyed by device arch, particle-count
// bucket (power of two), scene count, x subdivision and sort mode (which is
// the handle's own: its buffers are allocated for it).  A handle small enough
// for the split form runs density and force in that, which has no shape to
// choose; its sort has one in radix mode.
#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <string>

#include "sph_engine.hpp"

using namespace sph;

namespace {

std::mutex g_mu;
std::map<std::string, Tuning> g_cache;

std::string cache_key(const sph_handle* h, bool split) {
    int bucket = 0;
    while ((1u << bucket) < h->n && bucket < 31) ++bucket;
    return h->arch + ":" + std::to_string(bucket) + ":" + std::to_string(h->sc_h.size()) + ":" +
           std::to_string(h->xsub) + ":" + std::to_string(h->tune.sort_mode) + (split ? ":split" : h->wide_rows ? ":wide" : "");
}

struct Saved {
    DevBuf<float4> pos, vel;
    DevBuf<uint32_t> id;
};

}  // namespace

extern "C" int sph_autotune(sph_handle* h) {
    BudgetScope budget_scope(h ? &h->mem : nullptr);
    if (!h) return SPH_E_INVALID;
    if (!h->ready) return fail(h, SPH_E_NOT_READY, "call sph_make_ready first");
    const Tuning before = h->tune;  // stays where tuning fails
    h->tune.split = 1;
    const bool radix = h->tune.sort_mode == kSortRadix;
    if (split_form(h) && !radix) {  // no shape to choose
        invalidate_graph(h);
        return SPH_OK;
    }
    {
        std::lock_guard<std::mutex> lk(g_mu);
        auto it = g_cache.find(cache_key(h, split_form(h)));
        if (it != g_cache.end()) {
            const int mode = h->tune.sort_mode;
            h->tune = it->second;
            h->tune.sort_mode = mode;
            invalidate_graph(h);
            return SPH_OK;
        }
    }
    const size_t n = h->n;
    Saved sv;
    hipError_t e = sv.pos.ensure(n);
    if (e == hipSuccess) e = sv.vel.ensure(n);
    if (e == hipSuccess) e = sv.id.ensure(n);
    if (e == hipSuccess) e = hipMemcpyAsync(sv.pos.p, h->pos.p, n * sizeof(float4), hipMemcpyDeviceToDevice, h->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(sv.vel.p, h->vel.p, n * sizeof(float4), hipMemcpyDeviceToDevice, h->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(sv.id.p, h->id.p, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, h->stream);
    if (e != hipSuccess) {
        h->tune = before;
        return hip_fail(h, e, "autotune save");
    }
    const bool split = split_form(h);  // still, with the state saved
    const std::string key = cache_key(h, split);

    const bool prof_was = h->prof;
    auto restore = [&]() -> hipError_t {
        hipError_t x = hipMemcpyAsync(h->pos.p, sv.pos.p, n * sizeof(float4), hipMemcpyDeviceToDevice, h->stream);
        if (x == hipSuccess) x = hipMemcpyAsync(h->vel.p, sv.vel.p, n * sizeof(float4), hipMemcpyDeviceToDevice, h->stream);
        if (x == hipSuccess) x = hipMemcpyAsync(h->id.p, sv.id.p, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, h->stream);
        h->keys_valid = false;
        return x;
    };
    // Mean milliseconds per pass over `steps` profiled steps from the saved state.
    auto trial = [&](double* ms) -> int {
        if (restore() != hipSuccess) return SPH_E_HIP;
        h->prof = false;
        int rc = enqueue_step(h, h->work, false);  // warm-up (hash, caches)
        if (rc != SPH_OK) return rc;
        double tmp[SPH_NUM_PASSES];
        uint32_t cnt = 0;
        rc = sph_profile_read(h, tmp, &cnt);
        if (rc != SPH_OK) return rc;
        const int steps = 4;
        for (int s = 0; s < steps; ++s) {
            rc = enqueue_step(h, h->work, true);
            if (rc != SPH_OK) return rc;
        }
        rc = sph_profile_read(h, ms, &cnt);
        if (rc != SPH_OK) return rc;
        for (int p = 0; p < SPH_NUM_PASSES; ++p) ms[p] /= std::max(1u, cnt);
        return check_device_error(h);
    };

    // The form of the handle's size: its blocks are timed first, and it stays
    // unless the other is 5 % faster.
    const int of_size = staged_by_size(h);
    const int blocks[] = {64, 128, 256, 512};
    const int items[] = {4, 8, 12, 16};
    Tuning best = h->tune;
    if (!split) {
        best.by_size = 0;
        best.force_staged = best.density_staged = of_size;
    }
    double ms[SPH_NUM_PASSES];
    int rc = SPH_OK;
    // Takes the candidate with the least time in a pass (or two) as the field's value.
    auto choose = [&](int& field, const int* cand, int ncand, int pass) {
        double best_ms = 1e30;
        int best_v = field;
        for (int c = 0; c < ncand && rc == SPH_OK; ++c) {
            field = cand[c];
            h->tune = best;
            rc = trial(ms);
            if (rc == SPH_OK && ms[pass] < best_ms) { best_ms = ms[pass]; best_v = cand[c]; }
        }
        field = best_v;
    };
    if (!split) {
        choose(best.density_block, blocks, 4, SPH_PASS_DENSITY);
        choose(best.force_block, blocks, 4, SPH_PASS_FORCE);
    }
    // The gather's block and the keys per thread only shape the radix sort.
    if (radix) {
        choose(best.reorder_block, blocks, 4, SPH_PASS_REORDER);
        choose(best.sort_items, items, 4, SPH_PASS_SORT);
    }
    // Staged or gathered: the trials are a few steps from the state as it is,
    // often a fresh one, whose forms can lie within the trials' noise of each
    // other while compression and the reverse pass, which takes the force
    // pass's form, favour the size's: 16 scenes of 32,768 particles reverse 200
    // steps in 36.0 ms staged and in 41.9 where a trial preferred the gathered
    // force.  t[form]: each form's least time.
    auto form = [&](const double (&t)[2]) { return t[!of_size] < 0.95 * t[of_size] ? !of_size : of_size; };
    if (!split) {
        // Launch form of density and force (persistent or one block per tile;
        // force rows staged in LDS or gathered), judged on their summed time.
        double t[2] = {1e30, 1e30};
        int persistent[2] = {0, 0};
        for (int c = 0; c < 4 && rc == SPH_OK; ++c) {
            best.persistent = c & 1;
            best.force_staged = c >> 1;
            h->tune = best;
            rc = trial(ms);
            const double sum = ms[SPH_PASS_DENSITY] + ms[SPH_PASS_FORCE];
            if (rc == SPH_OK && sum < t[c >> 1]) { t[c >> 1] = sum; persistent[c >> 1] = c & 1; }
        }
        best.force_staged = form(t);
        best.persistent = persistent[best.force_staged];
        // Density rows staged in LDS or read from global memory.
        double d[2] = {1e30, 1e30};
        for (int c = 0; c < 2 && rc == SPH_OK; ++c) {
            best.density_staged = c;
            h->tune = best;
            rc = trial(ms);
            if (rc == SPH_OK) d[c] = ms[SPH_PASS_DENSITY];
        }
        best.density_staged = form(d);
        // A form other than the blocks were timed in gets its own.
        if (best.density_staged != of_size) choose(best.density_block, blocks, 4, SPH_PASS_DENSITY);
        if (best.force_staged != of_size) choose(best.force_block, blocks, 4, SPH_PASS_FORCE);
    }
    h->tune = rc == SPH_OK ? best : before;
    h->prof = prof_was;
    const hipError_t re = restore();
    invalidate_graph(h);
    if (rc != SPH_OK) return rc;
    if (re != hipSuccess) return hip_fail(h, re, "autotune restore");
    rc = sync(h);
    if (rc != SPH_OK) return rc;
    std::lock_guard<std::mutex> lk(g_mu);
    g_cache[key] = best;
    return SPH_OK;
}
