// Run by tests/test_host.py: the workspaces of split wide rows (vxs_api.cpp) over a HIP runtime and a
// sampler of this file's own, which run nothing and only keep the order: a stream has the work queued on
// it, an event the work queued before its record, and waiting ends that work. Checks that no workspace is
// ever handed to a launch while one that it is not ordered after may still be using it.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
using std::max;
using std::min;
#include "../voxwerk_amd/csrc/vxs_api.cpp"

namespace {

struct Use {  // of a workspace by a queued kernel or fill
    void* ws;
    hipStream_t stream;
    bool done;
};
std::vector<Use> uses;
std::map<hipEvent_t, std::vector<size_t>> events;  // the uses an event's last record covers
hipError_t last_error = hipSuccess;                // sticky until read
bool record_fails = false;
int launches = 0, failures = 0, allocations = 0, mallocs_fail = 0;
void* launched_with = nullptr;

hipStream_t stream(int i) { return reinterpret_cast<hipStream_t>(uintptr_t(0x1000 + 16 * i)); }
void finish(hipStream_t s) {
    for (Use& u : uses) u.done |= u.stream == s;
}
void use(void* ws, hipStream_t s) {
    for (const Use& u : uses)
        if (u.ws == ws && !u.done && u.stream != s) {
            std::printf("  a workspace in use on another stream was handed out\n");
            failures++;
        }
    uses.push_back({ws, s, false});
}
void expect(bool ok, const char* what) {
    if (ok) return;
    std::printf("  expected: %s\n", what);
    failures++;
}

}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() {
    for (Use& u : uses) u.done = true;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = stream(0), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return finish(s), hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* c) { return *c = hipStreamCaptureStatusNone, hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    for (size_t i : events[e])
        if (!uses[i].done) uses[i].stream = s;  // (ordered before what follows on s)
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = reinterpret_cast<hipEvent_t>(std::malloc(1)), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (record_fails) return last_error = hipErrorOutOfMemory;
    events[e].clear();
    for (size_t i = 0; i < uses.size(); i++)
        if (uses[i].stream == s && !uses[i].done) events[e].push_back(i);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    for (size_t i : events[e])
        if (!uses[i].done) return hipErrorNotReady;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    for (size_t i : events[e]) uses[i].done = true;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    allocations++;
    if (mallocs_fail > 0 && mallocs_fail--) return last_error = hipErrorOutOfMemory;
    return *p = std::malloc(n), hipSuccess;
}
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::malloc(n), hipSuccess; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* p, unsigned) { return *d = p, hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy2DAsync(void*, size_t, const void*, size_t, size_t, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int, size_t, hipStream_t s) { return use(p, s), hipSuccess; }
}

namespace vxs {
hipError_t launch_sample(const SampleArgs&, hipStream_t s, void* ws) {
    launches++;
    launched_with = ws;
    if (ws) use(ws, s);
    return hipGetLastError();  // (as the sampler's: whatever error the thread holds)
}
size_t split_workspace_bytes() { return 64; }
bool split_wanted(const SampleArgs&) { return true; }
hipError_t noalloc_scratch(int, void** out) { return *out = nullptr, hipSuccess; }
std::mutex& noalloc_lock(int) {
    static std::mutex m;
    return m;
}
hipError_t launch_draw_sequence(int32_t*, int, double*, hipStream_t) { return hipSuccess; }
hipError_t launch_embed(const EmbedArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_frame_embed(const FrameEmbedArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_head(const HeadArgs&, hipStream_t) { return hipSuccess; }
hipError_t launch_head_pack_int8(int, int, const uint16_t*, int64_t, int8_t*, int64_t, float*, hipStream_t) { return hipSuccess; }
}  // namespace vxs

namespace {

int sample_on(vxs_ctx* ctx, int s) {
    static float x[1];
    static vxs_params p[1];
    static int32_t id[1];
    static double u[1];
    vxs_set_stream(ctx, s ? stream(s) : nullptr);
    return vxs_sample_device(ctx, 1, 30000, x, 30000, nullptr, nullptr, p, 1, u, id, nullptr, nullptr, 0);
}

void streams_in_turn(vxs_ctx* ctx) {
    std::set<void*> seen;
    for (int s = 0; s <= kSplitStreams; s++) {
        expect(sample_on(ctx, s) == VXS_OK, "a call's status");
        seen.insert(launched_with);
    }
    expect(seen.size() == kSplitStreams + 1 && !seen.count(nullptr), "a workspace for each of the first streams");
    sample_on(ctx, 9);
    expect(launched_with == nullptr, "no workspace for a stream too many");
    finish(stream(2));
    sample_on(ctx, 9);
    expect(launched_with != nullptr, "an idle stream's workspace for another");
    sample_on(ctx, 9);
    expect(launched_with != nullptr, "a stream's own workspace again");
}

// A launch that reports an error the program left behind is queued like any other.
void older_error(vxs_ctx* ctx) {
    last_error = hipErrorInvalidDevice;
    expect(sample_on(ctx, 1) == VXS_ERR_HIP, "the older error reported");
    for (int s = 2; s < 8; s++) sample_on(ctx, s);
    (void)hipDeviceSynchronize();
    sample_on(ctx, 1);
    last_error = hipErrorInvalidDevice;
    sample_on(ctx, 1);  // again, with the stream's workspace recorded before
    for (int s = 2; s < 8; s++) sample_on(ctx, s);
}

// An event that cannot be recorded: the call waits instead.
void record_error(vxs_ctx* ctx) {
    record_fails = true;
    expect(sample_on(ctx, 1) == VXS_OK, "a call's status");
    record_fails = false;
    for (int s = 2; s < 8; s++) expect(sample_on(ctx, s) == VXS_OK, "a call's status");
}

void split_wait(vxs_ctx* ctx) {
    expect(vxs_set_split_wait(nullptr, 1) == VXS_ERR_INVALID_ARG, "no context");
    expect(vxs_set_split_wait(ctx, 10000000) == VXS_OK, "the longest wait");
    expect(vxs_set_split_wait(ctx, 10000001) == VXS_ERR_INVALID_ARG, "a wait too long");
}

// No memory for a workspace: the calls take one workgroup per row, and few of them try to allocate.
void no_memory(vxs_ctx* ctx) {
    sample_on(ctx, 1);  // (the other buffers of a call are there)
    const int before = allocations;
    mallocs_fail = 1 << 30;
    for (int i = 0; i < 200; i++) {
        expect(sample_on(ctx, i % 2 ? 0 : 2) == VXS_OK, "a call's status");
        expect(launched_with == nullptr, "no workspace");
    }
    expect(allocations - before <= 2, "one try, or two, in 200 calls");
    sample_on(ctx, 1);
    expect(launched_with != nullptr, "a stream's own workspace");
    mallocs_fail = 0;
    for (int i = 0; i < 300; i++) sample_on(ctx, 0);
    expect(launched_with != nullptr, "a workspace once there is memory again");
}

void run(const char* name, void (*test)(vxs_ctx*)) {
    std::printf("%s\n", name);
    vxs_ctx* ctx = nullptr;
    expect(vxs_create(&ctx, 0, 0, 0, 0) == VXS_OK, "a context");
    test(ctx);
    vxs_set_stream(ctx, nullptr);
    vxs_destroy(ctx);
    uses.clear();
    events.clear();
    last_error = hipSuccess;
}

}  // namespace

int main() {
    run("streams in turn", streams_in_turn);
    run("an older error", older_error);
    run("an event that cannot be recorded", record_error);
    run("no memory", no_memory);
    run("the wait of split rows", split_wait);
    std::printf("%d launches, %d failures\n", launches, failures);
    return failures != 0;
}
