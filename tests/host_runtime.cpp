// host_runtime.cpp — the library's host code on a machine without a GPU: a stand-in for the HIP runtime
// and rocFFT (device memory is host memory, copies are made at once, launched kernels are noted but not run),
// and scenarios that look at what the host code queues. The program's definitions of the runtime's
// functions come before the real runtime's. Usage: host_runtime SCENARIO; prints "name value" lines.
#include <hip/hip_runtime_api.h>
#include <rocfft/rocfft.h>
#include <unistd.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "lagpm.h"

struct ihipEvent_t {
    size_t at = 0;
};

namespace {
struct launch {
    std::string kernel;
    dim3 grid;
};
std::mutex mu;
// the library registers its kernels before this program's own variables are set up
std::map<const void*, std::string>& kernels() {
    static auto* k = new std::map<const void*, std::string>;
    return *k;
}
std::vector<launch> launches;
thread_local dim3 call_grid, call_block;
thread_local size_t call_lds;
thread_local hipStream_t call_stream;
char stream_mem[64];
std::atomic<int> nstream{0};
std::atomic<int> ncapture{0}, npinned{0};  // graph captures; pinned buffers of a megabyte and more
std::atomic<size_t> nuploaded{0};          // bytes copied to the device
uint32_t plant_nodes = 0;                  // tree builds find this many nodes, and that they do not fit
int malloc_fails = 0, nbad = 0;            // device allocations fail; launches of empty grids or with null node arrays
thread_local int slow_new = 0;             // allocations of this thread take this many microseconds
thread_local int fail_new = 0;             // the fail_new-th allocation of this thread from here on fails

struct own {  // the stand-in's own allocations neither fail nor count
    int f = fail_new;
    own() { fail_new = 0; }
    ~own() { fail_new = f; }
};

size_t count(const char* name) {  // launches so far of kernels of this name
    std::lock_guard<std::mutex> lk(mu);
    size_t c = 0;
    for (const launch& l : launches) c += l.kernel.find(name) != std::string::npos;
    return c;
}
}  // namespace

void* operator new(size_t n) {
    if (slow_new) usleep((useconds_t)slow_new);
    if (fail_new && --fail_new == 0) throw std::bad_alloc();
    if (void* p = malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

extern "C" {
void** __hipRegisterFatBinary(const void*) { return (void**)calloc(1, sizeof(void*)); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    call_grid = g; call_block = b; call_lds = lds; call_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = call_grid; *b = call_block; *lds = call_lds; *s = call_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void** args, size_t, hipStream_t) {
    own quiet;
    std::lock_guard<std::mutex> lk(mu);
    launches.push_back({kernels()[f], g});
    const std::string& name = launches.back().kernel;
    auto pointer = [&](int i) { return *(void**)args[i]; };
    if (g.x == 0 || g.y == 0 || g.z == 0) nbad++;
    if (name.find("tree_rows_kernel") != std::string::npos) {  // (sizes: nodes first, overflow fourth)
        ((uint32_t*)pointer(5))[0] = plant_nodes;
        ((uint32_t*)pointer(5))[3] = plant_nodes ? 1u : 0u;
    }
    if (name.find("tree_emit_kernel") != std::string::npos)  // the node arrays that it writes
        for (int i : {5, 8, 9, 10, 11, 12})
            if (!pointer(i)) nbad++;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 8;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error of the stand-in"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = calloc(1, 1 << 20); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
    if (malloc_fails) return hipErrorOutOfMemory;
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (n >= 1 << 20) npinned++;
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t) {
    memcpy(d, s, n);
    if (kind == hipMemcpyHostToDevice) nuploaded += n;
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)(stream_mem + nstream++); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { ncapture++; return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipEventCreate(hipEvent_t* e) { own quiet; *e = new ihipEvent_t; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    std::lock_guard<std::mutex> lk(mu);
    e->at = launches.size();
    return hipSuccess;
}
// "time" is the number of kernels queued between the two events
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) {
    *ms = (float)((double)b->at - (double)a->at);
    return hipSuccess;
}

rocfft_status rocfft_setup() { return rocfft_status_success; }
rocfft_status rocfft_plan_description_create(rocfft_plan_description* d) { *d = (rocfft_plan_description)stream_mem; return rocfft_status_success; }
rocfft_status rocfft_plan_description_destroy(rocfft_plan_description) { return rocfft_status_success; }
rocfft_status rocfft_plan_description_set_data_layout(rocfft_plan_description, rocfft_array_type, rocfft_array_type, const size_t*,
                                                      const size_t*, size_t, const size_t*, size_t, size_t, const size_t*, size_t) {
    return rocfft_status_success;
}
rocfft_status rocfft_plan_create(rocfft_plan* p, rocfft_result_placement, rocfft_transform_type, rocfft_precision, size_t,
                                 const size_t*, size_t, const rocfft_plan_description) {
    *p = (rocfft_plan)stream_mem;
    return rocfft_status_success;
}
rocfft_status rocfft_plan_destroy(rocfft_plan) { return rocfft_status_success; }
rocfft_status rocfft_plan_get_work_buffer_size(const rocfft_plan, size_t* n) { *n = 0; return rocfft_status_success; }
rocfft_status rocfft_execution_info_create(rocfft_execution_info* i) { *i = (rocfft_execution_info)stream_mem; return rocfft_status_success; }
rocfft_status rocfft_execution_info_destroy(rocfft_execution_info) { return rocfft_status_success; }
rocfft_status rocfft_execution_info_set_work_buffer(rocfft_execution_info, void*, size_t) { return rocfft_status_success; }
rocfft_status rocfft_execution_info_set_stream(rocfft_execution_info, void*) { return rocfft_status_success; }
rocfft_status rocfft_execute(const rocfft_plan, void**, void**, rocfft_execution_info) { return rocfft_status_success; }
}

namespace {
lagpm_ctx* ctx;

void must(int rc, const char* what) {
    if (rc == LAGPM_OK) return;
    printf("failed %s: %d %s\n", what, rc, lagpm_last_error(ctx));
    exit(2);
}
#define MUST(call) must((call), #call)

lagpm_params params(int n) {
    lagpm_params p{};
    p.n = n; p.law = LAGPM_LAW_ERFC; p.precision = LAGPM_PREC_FP32; p.deconvolve = 1;
    p.mass = 1.0; p.efold = 2.5; p.epsilon = 0.1; p.rsphere = 5.625; p.theta = 0.5;
    p.amax = 48.0; p.omep = 0.26; p.omeplam = 0.74;
    return p;
}
lagpm_box* new_box(int n, size_t np) {
    const lagpm_params p = params(n);
    lagpm_box* b = nullptr;
    MUST(lagpm_box_create(ctx, &p, np, &b));
    const std::vector<double> x(np, 1.0);
    MUST(lagpm_box_upload(ctx, b, x.data(), x.data(), x.data(), nullptr, nullptr, nullptr));
    return b;
}

// Key bits in order: a build that may split deeper than the last sort's bits must sort again. Prints
// the sorts queued by the tree correction in question.
void resort() {
    lagpm_evolfact ef{};
    ef.fact1 = ef.fact2 = 1.0f;
    lagpm_box* b = new_box(32, 1000);
    MUST(lagpm_treecorrection(ctx, b, &ef));  // full sort; the (empty) tree's depth becomes the limit
    MUST(lagpm_drift(ctx, b, 0.0));
    MUST(lagpm_tsc(ctx, b, nullptr));  // sorts the bits of that limit
    size_t before = count("keys_kernel");
    MUST(lagpm_treecorrection(ctx, b, &ef));
    printf("same_tuning %zu\n", count("keys_kernel") - before);
    MUST(lagpm_box_set_tuning(b, 4, 8));  // the depth is to be found again
    before = count("keys_kernel");
    MUST(lagpm_treecorrection(ctx, b, &ef));
    printf("other_tuning %zu\n", count("keys_kernel") - before);
    before = count("keys_kernel");
    MUST(lagpm_treecorrection(ctx, b, &ef));
    printf("again %zu\n", count("keys_kernel") - before);
    MUST(lagpm_drift(ctx, b, 0.0));
    MUST(lagpm_tsc(ctx, b, nullptr));
    before = count("keys_kernel");
    MUST(lagpm_box_set_tuning(b, 16, 64));
    const int64_t id = 0;
    double acc[3];
    MUST(lagpm_tree_accel_sample(ctx, b, &id, 1, acc));
    printf("sample %zu\n", count("keys_kernel") - before);
    MUST(lagpm_box_destroy(ctx, b));
}

// Whole steps launch their kernels, whatever lagpm_set_step_graphs was told. The first one is left out: its
// tree is built to the full depth, with a launch more a level.
void steps() {
    lagpm_box* b = new_box(32, 1000);
    const int on[4] = {0, 1, 1, 0};
    for (int i = 0; i < 4; i++) {
        MUST(lagpm_set_step_graphs(ctx, on[i]));
        const size_t before = launches.size();
        MUST(lagpm_kdk_step(ctx, b, 1.0 + 0.1 * i, 0.1));
        if (i) printf("step%d %zu\n", i, launches.size() - before);
    }
    printf("captures %d\n", ncapture.load());
    MUST(lagpm_box_destroy(ctx, b));
}

// The first large copies of a context, by two threads at once on boxes of their own.
void first_copies() {
    const size_t np = 100000;  // three arrays of 0.8 MB: through the pinned slots
    const lagpm_params p = params(32);
    lagpm_box* b[2];
    for (lagpm_box*& q : b) MUST(lagpm_box_create(ctx, &p, np, &q));
    const std::vector<double> x(np, 1.0);
    std::atomic<int> ready{0};
    std::thread t[2];
    int rc[2];
    for (int i = 0; i < 2; i++)
        t[i] = std::thread([&, i] {
            ready++;
            while (ready < 2) {}
            slow_new = 20000;
            rc[i] = lagpm_box_upload(ctx, b[i], x.data(), x.data(), x.data(), nullptr, nullptr, nullptr);
            slow_new = 0;
        });
    for (std::thread& q : t) q.join();
    must(rc[0], "upload of thread 0");
    must(rc[1], "upload of thread 1");
    printf("pinned %d\n", npinned.load());
    for (lagpm_box* q : b) MUST(lagpm_box_destroy(ctx, q));
}

// A large copy with each allocation that it makes on the host failing in turn: it says so, or does
// without, and a copy that reports success has moved every byte.
void no_host_memory() {
    const size_t np = 1000000;
    const lagpm_params p = params(32);
    lagpm_box* b = nullptr;
    MUST(lagpm_box_create(ctx, &p, np, &b));
    const std::vector<double> x(np, 1.0);
    int refused = 0, done = 0, other = 0, partial = 0;
    for (int k = 1; k <= 40; k++) {
        const size_t before = nuploaded;
        fail_new = k;
        const int rc = lagpm_box_upload(ctx, b, x.data(), x.data(), x.data(), nullptr, nullptr, nullptr);
        fail_new = 0;
        (rc == LAGPM_OK ? done : rc == LAGPM_E_NOMEM ? refused : other)++;
        if (rc == LAGPM_OK && nuploaded - before != 3 * np * sizeof(double)) partial++;
    }
    printf("refused %d\ndone_some %d\nother %d\npartial %d\n", refused > 0, done > 20, other, partial);
    MUST(lagpm_box_destroy(ctx, b));
}

// The tree times of a step cover the tree build alone, with the other phases' events recorded or not,
// for one box and for boxes of a batch.
void build_times() {
    lagpm_box* b[3] = {new_box(32, 1000), new_box(32, 1000), new_box(32, 1000)};
    const double a[3] = {1.0, 1.0, 1.0}, da[3] = {0.1, 0.1, 0.1};
    for (lagpm_box* q : b) MUST(lagpm_kdk_step(ctx, q, 1.0, 0.1));  // (full depth the first time)
    for (int events : {0, 1}) {
        MUST(lagpm_set_step_graphs(ctx, !events));
        for (int nbox : {1, 3}) {
            MUST(lagpm_batch_step(ctx, b, nbox, a, da));
            lagpm_timings t;
            lagpm_tree_stats s;
            MUST(lagpm_box_timings(ctx, b[0], &t));
            MUST(lagpm_tree_stats_get(b[0], &s));
            printf("events%d_boxes%d_timings %g\nevents%d_boxes%d_stats %g\n", events, nbox, t.ms_build, events, nbox, s.ms_build);
        }
    }
    for (lagpm_box* q : b) MUST(lagpm_box_destroy(ctx, q));
}

// Node arrays that cannot be grown: the call fails, and later ones find arrays or make them.
void no_device_memory() {
    lagpm_evolfact ef{};
    ef.fact1 = ef.fact2 = 1.0f;
    lagpm_box* b = new_box(32, 1000);
    MUST(lagpm_treecorrection(ctx, b, &ef));
    plant_nodes = 100000;
    malloc_fails = 1;
    printf("grow %d\n", lagpm_treecorrection(ctx, b, &ef) != LAGPM_OK);
    plant_nodes = 0;
    printf("still_none %d\n", lagpm_treecorrection(ctx, b, &ef) != LAGPM_OK);
    malloc_fails = 0;
    printf("again %d\n", lagpm_treecorrection(ctx, b, &ef));
    // the descriptors of a walk over many boxes
    const std::vector<double> a(70, 1.0), da(70, 0.1);
    std::vector<lagpm_box*> many;
    for (int i = 0; i < 70; i++) many.push_back(new_box(24, 10));
    MUST(lagpm_set_batch_pipeline(ctx, 1, 0));
    MUST(lagpm_batch_step(ctx, many.data(), 2, a.data(), da.data()));
    malloc_fails = 1;
    printf("many %d\n", lagpm_batch_step(ctx, many.data(), 70, a.data(), da.data()) != LAGPM_OK);
    malloc_fails = 0;
    printf("many_again %d\n", lagpm_batch_step(ctx, many.data(), 2, a.data(), da.data()));
    printf("bad_launches %d\n", nbad);
    for (lagpm_box* q : many) MUST(lagpm_box_destroy(ctx, q));
    MUST(lagpm_box_destroy(ctx, b));
}
}  // namespace

int main(int argc, char** argv) {
    setvbuf(stdout, nullptr, _IONBF, 0);
    const std::string what = argc > 1 ? argv[1] : "";
    must(lagpm_create(&ctx, 0), "lagpm_create");
    if (what == "resort") resort();
    else if (what == "steps") steps();
    else if (what == "first_copies") first_copies();
    else if (what == "no_host_memory") no_host_memory();
    else if (what == "build_times") build_times();
    else if (what == "no_device_memory") no_device_memory();
    else return 3;
    lagpm_destroy(ctx);
    printf("end 0\n");
    return 0;
}
