// The engine's host code without a GPU: this program defines the HIP runtime
// calls the library makes (its own definitions win over the runtime's), with
// host memory for device memory and kernels that do nothing but are noted by
// name.  Each check, named on the command line, drives the C ABI into a state
// that is hard to reach on a GPU and looks at what the host code asked for.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "sph_engine.h"

namespace fake {

// Host stub -> kernel name.  The library registers its kernels before this
// program's own objects are built.
std::map<const void*, std::string>& kernels() {
    static std::map<const void*, std::string> m;
    return m;
}
std::vector<std::string> launched;
std::map<void*, std::string>& events() {  // what was launched last before the event
    static std::map<void*, std::string> m;
    return m;
}
std::set<void*> held;      // device allocations
uint64_t frees = 0;        // device allocations given back so far
bool capturing = false;
std::map<void*, uint64_t> graphs;  // executable graph -> frees when it was captured
uint64_t captured_at = 0;
bool stale = false;        // a graph ran after a buffer it may name was given back
uint64_t device_left = ~0ull;  // bytes hipMalloc still hands out
std::map<void*, uint64_t> sizes;

int count(const char* what) {
    int n = 0;
    for (const std::string& s : launched) n += s.find(what) != std::string::npos;
    return n;
}

}  // namespace fake

#define API extern "C" __attribute__((visibility("default")))

API void** __hipRegisterFatBinary(const void*) { static void* m; return &m; }
API void __hipUnregisterFatBinary(void**) {}
API void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                               int*) {
    fake::kernels()[host] = name;
}
API void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
API hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
API hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
    *g = dim3(1);
    *b = dim3(1);
    *s = 0;
    *st = nullptr;
    return hipSuccess;
}
API hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
    fake::launched.push_back(fake::kernels()[f]);
    return hipSuccess;
}
API hipError_t hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (n > fake::device_left) return hipErrorOutOfMemory;
    fake::device_left -= n;
    *p = std::calloc(1, n);
    fake::held.insert(*p);
    fake::sizes[*p] = n;
    return hipSuccess;
}
API hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    if (!fake::held.erase(p)) {
        std::printf("hipFree of memory that is not held\n");
        std::exit(3);
    }
    fake::device_left += fake::sizes[p];
    ++fake::frees;
    std::free(p);
    return hipSuccess;
}
API hipError_t hipHostMalloc(void** p, size_t n, unsigned) { *p = std::calloc(1, n); return hipSuccess; }
API hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
API hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
API hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
API hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
API hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
API hipError_t hipSetDevice(int) { return hipSuccess; }
API hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
API const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
API hipError_t hipGetLastError() { return hipSuccess; }
API hipError_t hipGetSymbolAddress(void** p, const void* s) { *p = const_cast<void*>(s); return hipSuccess; }
API hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 4; return hipSuccess; }
API hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
API hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
API hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
API hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
API hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
API hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
API hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
API hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    fake::events()[e] = fake::launched.empty() ? "" : fake::launched.back();
    return hipSuccess;
}
API hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
API hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    fake::capturing = true;
    fake::captured_at = fake::frees;
    return hipSuccess;
}
API hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    fake::capturing = false;
    *g = reinterpret_cast<hipGraph_t>(std::malloc(1));
    return hipSuccess;
}
API hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *x = reinterpret_cast<hipGraphExec_t>(std::malloc(1));
    fake::graphs[*x] = fake::captured_at;
    return hipSuccess;
}
API hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
    fake::graphs.erase(x);
    std::free(x);
    return hipSuccess;
}
API hipError_t hipGraphDestroy(hipGraph_t g) { std::free(g); return hipSuccess; }
API hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t) {
    fake::launched.push_back("graph");
    fake::stale |= fake::graphs.at(x) != fake::frees;
    return hipSuccess;
}

// Milliseconds between two events: the caller's, by what was launched last
// before the later one.
namespace fake {
float (*pass_ms)(const std::string& kernel) = nullptr;
}
API hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t e) {
    *ms = fake::pass_ms ? fake::pass_ms(fake::events()[e]) : 0.005f;
    return hipSuccess;
}

// ------------------------------------------------------------------ checks

namespace {

#define CHECK(c)                                                      \
    do {                                                              \
        if (!(c)) {                                                   \
            std::printf("%s:%d: %s\n", __FILE__, __LINE__, #c);       \
            return 1;                                                 \
        }                                                             \
    } while (0)

// ratio: the support in particle radii.
sph_handle* make(uint32_t n, float ratio = 4.0f) {
    sph_params p;
    sph_params_default(&p);
    p.particle_radius = 0.005f;
    p.kernel_radius = ratio * 0.005f;
    sph_handle* e = nullptr;
    if (sph_create(&p, &e) != SPH_OK) std::exit(4);
    std::vector<float> x(3 * (size_t)n, 0.1f);
    if (sph_set_particles(e, x.data(), nullptr, n) != SPH_OK || sph_make_ready(e) != SPH_OK) std::exit(5);
    return e;
}

// A process's autotuned shapes are shared by handles of the same size bucket;
// how a handle sorts is its own.
int autotune_keeps_the_sort() {
    for (int first : {SPH_SORT_RADIX, SPH_SORT_CELL_COUNT}) {
        const uint32_t n = first == SPH_SORT_RADIX ? 50000u : 100000u;  // a bucket each
        sph_handle* e[2] = {make(n), make(n)};
        const int mode[2] = {first, first == SPH_SORT_RADIX ? SPH_SORT_CELL_COUNT : SPH_SORT_RADIX};
        for (int i = 0; i < 2; ++i) {
            CHECK(sph_set_sort_mode(e[i], mode[i]) == SPH_OK);
            CHECK(sph_autotune(e[i]) == SPH_OK);
            CHECK(sph_get_sort_mode(e[i]) == mode[i]);
            fake::launched.clear();
            CHECK(sph_set_use_graph(e[i], 0) == SPH_OK);
            CHECK(sph_advance_steps(e[i], 1) == SPH_OK);
            CHECK((fake::count("radix_pass") > 0) == (mode[i] == SPH_SORT_RADIX));
        }
        for (sph_handle* h : e) sph_destroy(h);
    }
    return 0;
}

// A step whose tables do not fit fails, and with room for them the next one
// hashes the state as if that one had not been asked for.
int hash_without_its_table_fails() {
    const uint32_t n = 5000;
    const uint64_t spares = n * (9ull * 4 + 128 * 2 + 4);
    sph_handle* full = make(n);
    uint64_t used = 0;
    CHECK(sph_device_memory_used(full, &used) == SPH_OK);
    sph_destroy(full);
    for (int frame = 0; frame < 2; ++frame) {
        sph_params p;
        sph_params_default(&p);
        p.kernel_radius = 0.02f;
        p.particle_radius = 0.005f;
        p.cfl_number = frame ? 0.3f : 0.0f;
        sph_handle* e = nullptr;
        CHECK(sph_create(&p, &e) == SPH_OK);
        CHECK(sph_set_device_memory_limit(e, used - spares) == SPH_OK);
        std::vector<float> x(3 * n, 0.1f);
        CHECK(sph_set_particles(e, x.data(), nullptr, n) == SPH_OK && sph_make_ready(e) == SPH_OK);
        const int cfg[5] = {64, 64, 256, 8, 0};
        CHECK(sph_set_tuning(e, cfg) == SPH_OK);
        // Room for the step's table of 64-particle tiles, not for the hash's of
        // 256; the frame loop hashes first.
        CHECK(sph_set_device_memory_limit(e, used - spares + (frame ? 0 : (n + 63) / 64 * 8)) == SPH_OK);
        fake::launched.clear();
        const int rc = frame ? sph_run_frame(e, nullptr, nullptr) : sph_advance_steps(e, 1);
        CHECK(rc == SPH_E_OOM);
        CHECK(fake::count("force") == 0 && fake::count("graph") == 0);
        CHECK(sph_set_device_memory_limit(e, 0) == SPH_OK);
        fake::launched.clear();
        CHECK(sph_advance_steps(e, 1) == SPH_OK);
        CHECK(fake::count("hash_kernel") == 1 && fake::count("force") == 1);
        sph_destroy(e);
    }
    return 0;
}

// Making a handle ready again when there is more room gives it the neighbour
// lists it did without: no graph that names the buffers before runs on.
int new_spares_drop_the_graphs() {
    const uint32_t n = 5000;
    const uint64_t lists = n * (128ull * 2 + 4);
    sph_handle* full = make(n);
    uint64_t used = 0;
    CHECK(sph_device_memory_used(full, &used) == SPH_OK);
    sph_destroy(full);
    sph_params p;
    sph_params_default(&p);
    p.kernel_radius = 0.02f;
    p.particle_radius = 0.005f;
    sph_handle* e = nullptr;
    CHECK(sph_create(&p, &e) == SPH_OK);
    CHECK(sph_set_device_memory_limit(e, used - lists) == SPH_OK);
    std::vector<float> x(3 * n, 0.1f);
    CHECK(sph_set_particles(e, x.data(), nullptr, n) == SPH_OK && sph_make_ready(e) == SPH_OK);
    CHECK(sph_set_device_memory_limit(e, used) == SPH_OK);  // the tile tables
    fake::launched.clear();
    CHECK(sph_advance_steps(e, 2) == SPH_OK);  // the second one's is a graph
    CHECK(fake::count("split") == 0 && fake::count("graph") == 1);
    CHECK(sph_set_device_memory_limit(e, 0) == SPH_OK);
    CHECK(sph_make_ready(e) == SPH_OK);
    fake::launched.clear();
    fake::stale = false;
    CHECK(sph_advance_steps(e, 1) == SPH_OK);
    CHECK(fake::count("graph") == 1 && !fake::stale);
    CHECK(fake::count("force_split") == 1);  // captured anew, with the lists
    sph_destroy(e);
    return 0;
}

// The forms that hold a row's candidates or a particle's neighbours in room of
// a fixed size are left to supports whose rows and neighbours fit them.
int wide_rows_are_gathered() {
    for (uint32_t n : {5000u, 200000u})
        for (float ratio : {4.0f, 6.0f, 7.0f, 12.0f}) {
            sph_handle* e = make(n, ratio);
            CHECK(sph_set_use_graph(e, 0) == SPH_OK);
            fake::launched.clear();
            CHECK(sph_advance_steps(e, 1) == SPH_OK);
            const bool wide = ratio > 6.5f;
            CHECK(fake::count("density_kernel") == wide && fake::count("force_kernel") == wide);
            CHECK(fake::count("split") == (!wide && n == 5000u ? 2 : 0));
            CHECK(fake::count("staged") == (!wide && n == 200000u ? 2 : 0));
            sph_destroy(e);
        }
    return 0;
}

// sph_get_tuning says what runs, and setting that changes nothing: small, in
// between, large, tuned and set handles.
int tuning_round_trip() {
    struct {
        uint32_t n;
        float ratio;
        int form;  // launch form an untuned handle reports
    } const kinds[] = {{5000u, 4.0f, 8}, {40960u, 4.0f, 8}, {40961u, 4.0f, 0}, {131071u, 4.0f, 0},
                       {131072u, 4.0f, 6}, {5000u, 8.0f, 0}, {200000u, 8.0f, 0}};
    for (const auto& kind : kinds)
        for (int how = 0; how < 3; ++how) {  // untuned, autotuned, set to other forms
            sph_handle* e = make(kind.n, kind.ratio);
            CHECK(sph_set_use_graph(e, 0) == SPH_OK);
            if (how == 1) CHECK(sph_autotune(e) == SPH_OK);
            const int other[5] = {128, 64, 256, 8, 4};
            if (how == 2) CHECK(sph_set_tuning(e, other) == SPH_OK);
            int cfg[5], again[5];
            CHECK(sph_get_tuning(e, cfg) == SPH_OK);
            if (how == 0) CHECK(cfg[4] == kind.form);
            if (how == 2) CHECK(std::memcmp(cfg, other, sizeof(cfg)) == 0);
            CHECK(sph_advance_steps(e, 1) == SPH_OK);
            fake::launched.clear();
            CHECK(sph_advance_steps(e, 1) == SPH_OK);
            const std::vector<std::string> before = fake::launched;
            CHECK(fake::count("split") == ((cfg[4] & 8) ? 2 : 0));
            if (!(cfg[4] & 8)) {
                CHECK(fake::count("force_staged") == ((cfg[4] >> 1) & 1));
                CHECK(fake::count("density_staged") == ((cfg[4] >> 2) & 1));
            }
            CHECK(sph_set_tuning(e, cfg) == SPH_OK);
            CHECK(sph_get_tuning(e, again) == SPH_OK && std::memcmp(cfg, again, sizeof(cfg)) == 0);
            fake::launched.clear();
            CHECK(sph_advance_steps(e, 1) == SPH_OK);
            CHECK(fake::launched == before);
            const int bad[5] = {256, 256, 256, 8, 16};
            CHECK(sph_set_tuning(e, bad) == SPH_E_INVALID);
            sph_destroy(e);
        }
    return 0;
}

// Small handles have no density and force shapes to choose, but the radix
// sort's are timed for them as for others, for each a set of its own.
int autotune_times_the_radix_sort() {
    for (uint32_t n : {5000u, 33000u, 60000u}) {  // two of one size bucket
        sph_handle* e = make(n);
        CHECK(sph_set_sort_mode(e, SPH_SORT_RADIX) == SPH_OK);
        fake::launched.clear();
        CHECK(sph_autotune(e) == SPH_OK);
        for (const char* kernel : {"radix_pass_kernelILi4E", "radix_pass_kernelILi16E"}) CHECK(fake::count(kernel) > 0);
        CHECK((fake::count("split") > 0) == (n < 40960u));
        CHECK((fake::count("staged") > 0) == (n > 40960u));
        sph_destroy(e);
        e = make(n);  // cell counts: nothing to time where the form has no shape
        fake::launched.clear();
        CHECK(sph_autotune(e) == SPH_OK);
        CHECK((fake::launched.size() > 0) == (n > 40960u));
        sph_destroy(e);
    }
    return 0;
}

// The blocks are timed in the form that runs, and a form other than the size's
// has to be 5 % faster than the size's, not than what it was compared with last.
float blocks_of_forms(const std::string& k) {
    auto has = [&](const char* s) { return k.find(s) != std::string::npos; };
    if (has("force_staged")) return has("Li64E") ? 0.9f : 1.0f;
    if (has("force_kernel")) return has("Li512E") ? 1.2f : 1.5f;  // the gathered form's best block is another
    if (has("density_staged")) return has("Li128E") ? 0.9f : 1.0f;
    if (has("density_kernel")) return has("Li256E") ? 1.2f : 1.5f;
    return 0.005f;
}
bool persistent_gathers_win(const sph_handle* h) {
    int cfg[5];
    return sph_get_tuning(h, cfg) == SPH_OK && (cfg[4] & 3) == 1;
}
const sph_handle* timed = nullptr;
float persistent_gather(const std::string& k) {
    if (k.find("force") == std::string::npos) return 0.001f;
    if (k.find("staged") != std::string::npos) return 1.0f;
    return persistent_gathers_win(timed) ? 0.90f : 0.94f;  // both 5 % faster, the second by less over the first
}
int autotune_compares_forms() {
    sph_handle* e = make(1u << 18);
    fake::pass_ms = blocks_of_forms;
    CHECK(sph_autotune(e) == SPH_OK);
    int cfg[5];
    CHECK(sph_get_tuning(e, cfg) == SPH_OK);
    CHECK(cfg[0] == 128 && cfg[1] == 64 && (cfg[4] & 6) == 6);
    sph_destroy(e);
    timed = e = make(1u << 19);
    fake::pass_ms = persistent_gather;
    CHECK(sph_autotune(e) == SPH_OK);
    CHECK(sph_get_tuning(e, cfg) == SPH_OK);
    CHECK((cfg[4] & 3) == 1);
    fake::pass_ms = nullptr;
    sph_destroy(e);
    return 0;
}

// A tuning that fails leaves the shapes as they were.
int failed_autotune_changes_nothing() {
    const uint32_t n = 30000;
    sph_handle* e = make(n);
    uint64_t used = 0;
    CHECK(sph_device_memory_used(e, &used) == SPH_OK);
    sph_params p;
    CHECK(sph_get_params(e, &p) == SPH_OK);
    sph_destroy(e);
    // No room for the spares, nor for the state to be saved.
    CHECK(sph_create(&p, &e) == SPH_OK);
    CHECK(sph_set_device_memory_limit(e, used - n * (9ull * 4 + 128 * 2 + 4) + 1000) == SPH_OK);
    std::vector<float> x(3 * n, 0.1f);
    CHECK(sph_set_particles(e, x.data(), nullptr, n) == SPH_OK && sph_make_ready(e) == SPH_OK);
    const int other[5] = {128, 64, 256, 8, 4};
    CHECK(sph_set_tuning(e, other) == SPH_OK);
    CHECK(sph_autotune(e) == SPH_E_OOM);
    CHECK(sph_set_device_memory_limit(e, 0) == SPH_OK);
    CHECK(sph_make_ready(e) == SPH_OK);  // with its spares again
    int cfg[5];
    CHECK(sph_get_tuning(e, cfg) == SPH_OK && std::memcmp(cfg, other, sizeof(cfg)) == 0);
    sph_destroy(e);
    return 0;
}

// What a handle can do without makes room for another handle's buffers.
int spares_make_room_for_others() {
    sph_handle* a = make(30000);
    CHECK(sph_advance_steps(a, 2) == SPH_OK);
    fake::launched.clear();
    CHECK(sph_advance_steps(a, 1) == SPH_OK && fake::count("graph") == 1);
    uint64_t used = 0, after = 0;
    CHECK(sph_device_memory_used(a, &used) == SPH_OK);
    sph_handle* b = make(20000);
    uint64_t need = 0;
    CHECK(sph_device_memory_used(b, &need) == SPH_OK);
    sph_destroy(b);
    const uint64_t spares_a = 30000ull * (9 * 4 + 128 * 2 + 4), spares_b = 20000ull * (9 * 4 + 128 * 2 + 4);
    // Room for all but a kilobyte of b's own buffers.
    fake::device_left = need - spares_b - 1024;
    b = make(20000);
    CHECK(sph_device_memory_used(a, &after) == SPH_OK && after == used - spares_a);
    fake::device_left = ~0ull >> 1;
    fake::stale = false;
    for (sph_handle* h : {a, b}) CHECK(sph_advance_steps(h, 2) == SPH_OK);
    CHECK(!fake::stale);
    // Spares alone take nothing from other handles.
    CHECK(sph_make_ready(a) == SPH_OK && sph_device_memory_used(a, &after) == SPH_OK && after >= used);
    fake::device_left = 0;
    CHECK(sph_make_ready(b) == SPH_OK && sph_device_memory_used(a, &used) == SPH_OK && used == after);
    sph_destroy(a);
    sph_destroy(b);
    return 0;
}

struct Check {
    const char* name;
    int (*run)();
};
const Check kChecks[] = {
    {"autotune_keeps_the_sort", autotune_keeps_the_sort},
    {"hash_without_its_table_fails", hash_without_its_table_fails},
    {"new_spares_drop_the_graphs", new_spares_drop_the_graphs},
    {"wide_rows_are_gathered", wide_rows_are_gathered},
    {"tuning_round_trip", tuning_round_trip},
    {"autotune_times_the_radix_sort", autotune_times_the_radix_sort},
    {"autotune_compares_forms", autotune_compares_forms},
    {"failed_autotune_changes_nothing", failed_autotune_changes_nothing},
    {"spares_make_room_for_others", spares_make_room_for_others},
};

}  // namespace

int main(int argc, char** argv) {
    for (const Check& c : kChecks)
        if (argc == 2 && std::strcmp(argv[1], c.name) == 0) return c.run();
    std::printf("no such check\n");
    return 2;
}
