// The library's host side without a GPU: this program defines the HIP calls that
// libastc_mi355x.so makes (the dynamic linker takes an executable's definitions
// first), with host memory for device memory and launches that are written down
// instead of run.  Each scenario (argv[1]) drives entry points and prints what the
// host queued; test_host_queueing.py says what that has to be.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "astc_mi355x.h"

namespace {

// What a launch, in stream order and through events, is known to follow.
using Ops = std::set<int>;
struct Stream { Ops before; };
struct Event { Ops before; int queries = 0; };
struct Launch {
    std::string kernel;
    unsigned grid;
    size_t lds;
    Stream* stream;
    Ops before;
    std::vector<uint8_t> args;  // the kernel's first argument, if it is a copy list
};

struct CopyList {  // as the copy kernel takes it
    struct { void* dst; const void* src; int64_t bytes; } range[64];
    int first[64];
    int count;
};

std::map<const void*, std::string>& kernels() {
    static std::map<const void*, std::string> k;
    return k;
}
std::vector<Launch> launches;
Stream null_stream;
int fail_alloc_after = -1;  // allocations until one fails; -1: none does
struct { dim3 grid, block; size_t lds; hipStream_t stream; } pushed;

Stream* of(hipStream_t s) { return s ? reinterpret_cast<Stream*>(s) : &null_stream; }
bool allocation_fails() { return fail_alloc_after >= 0 && fail_alloc_after-- == 0; }
hipError_t allocate(void** p, size_t n) {
    *p = nullptr;
    if (allocation_fails()) return hipErrorOutOfMemory;
    *p = std::aligned_alloc(4096, (n + 4095) / 4096 * 4096);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}

}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    pushed = {g, b, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = pushed.grid; *b = pushed.block; *lds = pushed.lds; *s = pushed.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void** args, size_t lds, hipStream_t s) {
    Launch l{kernels()[f], g.x, lds, of(s), of(s)->before, {}};
    if (l.kernel.find("copy_kernel") != std::string::npos) {
        l.args.resize(sizeof(CopyList));
        std::memcpy(l.args.data(), args[0], sizeof(CopyList));
    }
    of(s)->before.insert(int(launches.size()));
    launches.push_back(l);
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return allocate(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return allocate(p, n); }
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { return allocate(p, 4 << 20); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = reinterpret_cast<hipStream_t>(new Stream()); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete of(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st) { *st = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    const Ops& b = reinterpret_cast<Event*>(e)->before;
    of(s)->before.insert(b.begin(), b.end());
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = reinterpret_cast<hipEvent_t>(new Event()); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event*>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    *reinterpret_cast<Event*>(e) = {of(s)->before, 0};
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
// a batch takes a few polls, so that every slot has one in flight
hipError_t hipEventQuery(hipEvent_t e) { return ++reinterpret_cast<Event*>(e)->queries > 5 ? hipSuccess : hipErrorNotReady; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1; return hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = nullptr; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { *e = nullptr; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"

namespace {

astc_ctx* make_context() {
    astc_ctx* ctx = nullptr;
    if (astc_ctx_create(0, &ctx) != ASTC_OK) std::exit(3);
    return ctx;
}
astc_server* make_server(astc_ctx* ctx, int slots, int per_batch) {
    astc_server_config cfg{64 << 20, slots, per_batch, {4, 2, 1, 0, 1}};
    astc_server* sv = nullptr;
    if (astc_server_create(ctx, &cfg, &sv) != ASTC_OK) std::exit(3);
    return sv;
}

// Six requests, two a batch, three batches in flight; `same`: with one destination.
// Prints how many pairs of the trace's launches on different streams are ordered.
void overlapping_trace(bool same) {
    astc_ctx* ctx = make_context();
    astc_server* sv = make_server(ctx, 3, 2);
    const astc_image_desc d{64, 64, 256, ASTC_FMT_RGBA8, 4, ASTC_FLAG_ALPHA};
    std::vector<uint8_t> src(6 * 16384), dst(6 * 4096 + 16);
    uint8_t* aligned = dst.data() + (16 - reinterpret_cast<uintptr_t>(dst.data()) % 16) % 16;
    std::vector<astc_request> reqs;
    for (int i = 0; i < 6; ++i) {
        astc_request r{};
        r.images = &d;
        r.nimages = 1;
        r.src_dev = src.data() + 16384 * i;
        r.dst_dev = aligned + (same ? 0 : 4096 * i);
        reqs.push_back(r);
    }
    launches.clear();
    double latency[6];
    astc_server_stats st{};
    const int rc = astc_server_run_trace(sv, reqs.data(), 6, latency, &st);
    int ordered = 0, unordered = 0;
    for (size_t a = 0; a < launches.size(); ++a)
        for (size_t b = a + 1; b < launches.size(); ++b)
            if (launches[a].stream != launches[b].stream) ++(launches[b].before.count(int(a)) ? ordered : unordered);
    std::printf("rc %d batches %lld peak_inflight %d ordered %d unordered %d\n", rc, (long long)st.batches,
                st.peak_inflight, ordered, unordered);
    astc_server_destroy(sv);
    astc_ctx_destroy(ctx);
}

// A request of more images than the slots' work lists have room for, with the k-th
// allocation of the growth failing, then again with none: prints the return codes.
void growth_fails(int k) {
    astc_ctx* ctx = make_context();
    astc_server* sv = make_server(ctx, 2, 2);
    const std::vector<astc_image_desc> images(5000, astc_image_desc{4, 4, 16, ASTC_FMT_RGBA8, 4, 0});
    std::vector<uint8_t> src(5000 * 256);
    astc_request r{};
    r.images = images.data();
    r.nimages = int(images.size());
    r.src_dev = src.data();
    double latency;
    fail_alloc_after = k;
    const int first = astc_server_run_trace(sv, &r, 1, &latency, nullptr);
    fail_alloc_after = -1;
    const int second = astc_server_run_trace(sv, &r, 1, &latency, nullptr);
    std::printf("first %d second %d\n", first, second);
    astc_server_destroy(sv);
    astc_ctx_destroy(ctx);
}

// A batch of one image of 400 x 250 blocks for each of the three kernels: each
// launch's workgroups and LDS beside its own.
void batch_tuning(const astc_tuning& t) {
    astc_ctx* ctx = make_context();
    const astc_image_desc descs[3] = {{2400, 1500, 9600, ASTC_FMT_RGBA8, 6, ASTC_FLAG_ALPHA},
                                      {1600, 1000, 6400, ASTC_FMT_RGBA8, 4, ASTC_FLAG_ALPHA},
                                      {1600, 1000, 4800, ASTC_FMT_RGB8, 4, 0}};
    const void* srcs[3] = {reinterpret_cast<void*>(4096), reinterpret_cast<void*>(4096), reinterpret_cast<void*>(4096)};
    void* dsts[3] = {reinterpret_cast<void*>(4096), reinterpret_cast<void*>(4096), reinterpret_cast<void*>(4096)};
    astc_batch* b = nullptr;
    if (astc_batch_create(ctx, descs, srcs, dsts, 3, &b) != ASTC_OK || astc_batch_set_tuning(b, &t) != ASTC_OK) std::exit(3);
    launches.clear();
    const int rc = astc_batch_launch(b, nullptr);
    std::printf("rc %d\n", rc);
    for (const Launch& l : launches) std::printf("grid %u lds %zu\n", l.grid, l.lds);
    astc_batch_destroy(b);
    astc_ctx_destroy(ctx);
}

// The workgroups of a plain launch over an RGBA8 image of `blocks` x 1 blocks.
void plain_grid(int dim, int blocks, uint32_t flags, const astc_plain_tuning& t) {
    astc_ctx* ctx = make_context();
    const astc_image_desc d{dim * blocks, dim, 4 * dim * blocks, ASTC_FMT_RGBA8, dim, flags};
    launches.clear();
    const int rc = astc_encode_tuned(ctx, &d, reinterpret_cast<void*>(4096), reinterpret_cast<void*>(4096), &t, nullptr);
    std::printf("rc %d grid %u\n", rc, launches.empty() ? 0 : launches[0].grid);
    astc_ctx_destroy(ctx);
}

// The autotuner over a batch of one image of blocks x 1 blocks: its launches (each
// candidate's, one to warm up and three timed) and what it keeps.
void autotune(int dim, int blocks) {
    astc_ctx* ctx = make_context();
    const astc_image_desc d{dim * blocks, dim, 4 * dim * blocks, ASTC_FMT_RGBA8, dim, 0};
    const void* src = reinterpret_cast<void*>(4096);
    void* dst = reinterpret_cast<void*>(4096);
    astc_batch* b = nullptr;
    astc_tuning best{};
    if (astc_batch_create(ctx, &d, &src, &dst, 1, &b) != ASTC_OK) std::exit(3);
    launches.clear();
    const int rc = astc_batch_autotune(b, nullptr, 3, &best);
    std::printf("rc %d launches %zu blocks_per_lane %d prefetch %d lanes %d\n", rc, launches.size(), best.blocks_per_lane,
                best.prefetch, best.lanes_per_block);
    astc_batch_destroy(b);
    astc_ctx_destroy(ctx);
}

// A batch of one image of columns x rows blocks: its return code and work items.
void batch_items(int columns, int rows) {
    astc_ctx* ctx = make_context();
    const astc_image_desc d{4 * columns, 4 * rows, 16 * columns, ASTC_FMT_RGBA8, 4, 0};
    const void* src = reinterpret_cast<void*>(4096);
    void* dst = reinterpret_cast<void*>(4096);
    astc_batch* b = nullptr;
    const int rc = astc_batch_create(ctx, &d, &src, &dst, 1, &b);
    int64_t blocks = 0, texels = 0;
    int32_t items = 0;
    if (b) astc_batch_info(b, &blocks, &texels, &items);
    std::printf("rc %d blocks %lld items %d\n", rc, (long long)blocks, items);
    astc_batch_destroy(b);
    astc_ctx_destroy(ctx);
}

}  // namespace

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "one_destination") overlapping_trace(true);
    else if (what == "own_destinations") overlapping_trace(false);
    else if (what == "growth_fails") growth_fails(std::atoi(argv[2]));
    else if (what == "batch_tuning")
        batch_tuning({std::atoi(argv[2]), std::atoi(argv[3]), std::atoi(argv[4]), std::atoi(argv[5]), std::atoi(argv[6])});
    else if (what == "plain_grid")
        plain_grid(std::atoi(argv[2]), std::atoi(argv[3]), unsigned(std::atoi(argv[4])),
                   {std::atoi(argv[5]), std::atoi(argv[6]), std::atoi(argv[7]), std::atoi(argv[8]), std::atoi(argv[9])});
    else if (what == "autotune") autotune(std::atoi(argv[2]), std::atoi(argv[3]));
    else if (what == "batch_items") batch_items(std::atoi(argv[2]), std::atoi(argv[3]));
    else return 2;
    return 0;
}
