// The density network's entry points against a stand-in for the HIP runtime in
// this executable (its symbols come before the library's in the loader's order):
// device memory is host memory, asynchronous copies and kernels wait in their
// stream's queue until something synchronises it, kernels do nothing, and the
// k-th launch fails.  Whichever launch that is, an entry point may return only
// when its queues are empty: what it leaves queued would read and write buffers
// that go with it, and the next pass's workspace.
//   failed_launches <deck_dir> <name>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/sq_amd.h"

namespace {
struct Op { hipStream_t st; void *dst; const void *src; size_t n; };
std::vector<Op> queue;
long launches = 0, fail_at = -1;
hipError_t last = hipSuccess;
int events = 0;
hipStream_t pushed = nullptr;

void drain(hipStream_t st, bool all)
{
    std::vector<Op> rest;
    for (const Op &o : queue) {
        if (!all && o.st != st) { rest.push_back(o); continue; }
        if (o.dst) memcpy(o.dst, o.src, o.n);
    }
    queue.swap(rest);
}
}  // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t st) { pushed = st; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, hipStream_t *s)
{
    *g = dim3(1);
    *b = dim3(1);
    *l = 0;
    *s = pushed;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t st)
{
    if (launches++ == fail_at) return last = hipErrorLaunchFailure;
    queue.push_back({st, nullptr, nullptr, 0});
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { drain(nullptr, true); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)(size_t)++events; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { drain(nullptr, true); return hipSuccess; }
hipError_t hipFree(void *p) { drain(nullptr, true); free(p); return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 160 * 1024;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipGetSymbolAddress(void **p, const void *) { static char room[256]; *p = room; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipErrorUnknown; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorUnknown; }
hipError_t hipMalloc(void **p, size_t n) { *p = calloc(1, std::max<size_t>(n, 1)); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipMemGetAddressRange(hipDeviceptr_t *, size_t *, hipDeviceptr_t) { return hipErrorUnknown; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) { queue.push_back({st, d, s, n}); return hipSuccess; }
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return hipErrorUnknown; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorUnknown; }
hipError_t hipStreamCreate(hipStream_t *s) { *s = (hipStream_t)(size_t)++events; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorUnknown; }
hipError_t hipStreamSynchronize(hipStream_t st) { drain(st, false); return hipSuccess; }
}

template <typename F>
static int check(const char *name, F call)
{
    for (long k = 0; k < 1000; k++) {
        launches = 0;
        fail_at = k;
        const int rc = call();
        const bool failed = launches > k;   // else every launch went through
        if (!queue.empty()) {
            printf("%s: %zu operations queued after launch %ld failed\n", name, queue.size(), k);
            return 1;
        }
        if (!failed) {
            printf("%s: %ld launches\n", name, k);
            return k == 0;
        }
        if (rc == 0) {
            printf("%s: launch %ld failed unnoticed\n", name, k);
            return 1;
        }
    }
    return 1;
}

int main(int argc, char **argv)
{
    if (argc != 3) return 2;
    sq_options o;
    sq_default_options(&o);
    sq_ctx *c = nullptr;
    sq_info I;
    o.device = -1;
    if (sq_create_from_deck(argv[1], argv[2], &o, &c) || sq_get_info(c, &I)) return 2;
    sq_destroy(c);
    o.device = 0;
    for (int d = 0; d < 3; d++) o.rank_box[3 + d] = I.npts[d] - 1;
    if (sq_create_from_deck(argv[1], argv[2], &o, &c)) {
        printf("context: %s\n", sq_last_error());
        return 2;
    }
    drain(nullptr, true);
    sq_mlp *m = nullptr;
    if (sq_mlp_create(0, 1, &m)) return 2;
    const long n = 100;
    std::vector<float> x(32 * n, 0.5f), t(n, 0.25f), y(n);
    std::vector<double> g(1 << 14), rho((size_t)(I.npts[0] - 1) * (I.npts[1] - 1) * (I.npts[2] - 1));
    double loss;
    int bad = 0;
    bad |= check("forward", [&] { return sq_mlp_forward(m, x.data(), n, 1, 1, y.data()); });
    bad |= check("loss_grad", [&] { return sq_mlp_loss_grad(m, x.data(), t.data(), n, &loss, g.data()); });
    bad |= check("guess", [&] { return sq_mlp_guess(m, c, 1, rho.data()); });
    bad |= check("descriptors", [&] {
        std::vector<float> f(32 * rho.size());
        return sq_mlp_descriptors(c, f.data());
    });
    fail_at = -1;
    sq_mlp_destroy(m);
    sq_destroy(c);
    printf(bad ? "failed\n" : "all queues empty\n");
    return bad;
}
