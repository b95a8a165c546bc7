// A HIP runtime without a GPU, for tests of the host code: loaded before
// libimexlb.so (RTLD_GLOBAL), its functions take the place of libamdhip64's.  Device
// memory is address space that stays empty until it is touched, of a size that the
// test sets; launches are recorded, refused where HIP refuses them, and advance a
// clock by a time that the test sets per kernel; the one kernel that is carried
// out is k_copy_out.
#include <hip/hip_runtime.h>

#include <sys/mman.h>
#include <unistd.h>

#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../imexlb_amd/csrc/kernels.h"

namespace {
struct Launch {
    std::string name;
    uint64_t grid, block;
};
struct Event {
    double at = 0;
};
struct Graph {
    double ms = 0;
};
std::mutex m;
std::map<const void *, std::string> names;
std::vector<Launch> launches;
std::vector<std::pair<std::string, double>> costs;
std::map<const void *, size_t> held, pinned;
size_t room = size_t(288) << 30, used = 0, most_pinned = 0;
uint64_t next_range = uint64_t(1) << 44;
double now = 0, captured = 0;
bool capturing = false;
useconds_t copy_delay = 0;
thread_local struct {
    dim3 grid, block;
    size_t shared;
    hipStream_t st;
} call;

hipError_t take(void **p, size_t n)
{
    std::lock_guard<std::mutex> l(m);
    if (n > room - used) return hipErrorOutOfMemory;
    void *q = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (q == MAP_FAILED) return hipErrorOutOfMemory;
    held[q] = n;
    used += n;
    *p = q;
    return hipSuccess;
}

void copy_out(const imx::CopyOut &c)
{
    for (int k = 0; k < 4; ++k)
        if (c.bytes[k]) std::memcpy(c.dst + c.at[k] * 16, c.src[k], c.bytes[k]);
    if (copy_delay) usleep(copy_delay);
}
}  // namespace

extern "C" {
// ---- what a test sets and reads
void fake_room(size_t bytes) { room = bytes; }
size_t fake_used() { return used; }
size_t fake_most_pinned() { return most_pinned; }
void fake_copy_delay(unsigned us) { copy_delay = us; }
void fake_cost(const char *part, double ms) { costs.insert(costs.begin(), {part, ms}); }
// every allocation of at most `bytes` holds a value of its own, in all its doubles
void fake_paint(size_t bytes)
{
    std::lock_guard<std::mutex> l(m);
    double v = 0;
    for (auto &h : held)
        if (++v, h.second <= bytes)
            for (size_t k = 0; k < h.second / sizeof v; ++k) ((double *)h.first)[k] = v;
}
void fake_forget() { launches.clear(); }
int fake_launches() { return (int)launches.size(); }
const char *fake_name(int k) { return launches[k].name.c_str(); }
uint64_t fake_grid(int k) { return launches[k].grid; }
uint64_t fake_block(int k) { return launches[k].block; }

// ---- the runtime
void **__hipRegisterFatBinary(const void *) { return new void *; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    names[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st)
{
    call = {g, b, s, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st)
{
    *g = call.grid;
    *b = call.block;
    *s = call.shared;
    *st = call.st;
    return hipSuccess;
}
static thread_local hipError_t last = hipSuccess;
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t)
{
    {
        std::lock_guard<std::mutex> l(m);
        // at most 1024 threads a workgroup, fewer than 2^32 work-items along x
        if (g.x == 0 || b.x == 0 || b.x > 1024 || (uint64_t)g.x * b.x >= (uint64_t(1) << 32))
            return last = hipErrorInvalidConfiguration;
        launches.push_back({names[f], g.x, b.x});
        double ms = 0;
        for (auto &c : costs)
            if (names[f].find(c.first) != std::string::npos) {
                ms = c.second;
                break;
            }
        (capturing ? captured : now) += ms;
        if (names[f].find("k_copy_out") == std::string::npos) return hipSuccess;
    }
    copy_out(*(const imx::CopyOut *)args[0]);
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "ok" : "refused by the fake runtime"; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t)
{
    std::lock_guard<std::mutex> l(m);
    *f = room - used;
    *t = room;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) { return last = take(p, n); }
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> l(m);
    auto it = held.find(p);
    if (it == held.end()) return p ? hipErrorInvalidValue : hipSuccess;
    used -= it->second;
    munmap(p, it->second);
    held.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> l(m);
    *p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
    pinned[*p] = n;
    most_pinned = n > most_pinned ? n : most_pinned;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)  // kept mapped: a late access is a wrong value, not a fault
{
    std::lock_guard<std::mutex> l(m);
    pinned.erase(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *)
{
    std::memset(a, 0, sizeof *a);
    a->type = hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }  // fresh memory is 0
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorInvalidValue; }
hipError_t hipStreamCreate(hipStream_t *s) { return *s = (hipStream_t)1, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t) new Event, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete (Event *)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return ((Event *)e)->at = now, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    *ms = (float)(((Event *)b)->at - ((Event *)a)->at);
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
    capturing = true;
    captured = 0;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    capturing = false;
    *g = (hipGraph_t) new Graph{captured};
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *, char *, size_t)
{
    return *x = (hipGraphExec_t) new Graph(*(Graph *)g), hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete (Graph *)g, hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return delete (Graph *)x, hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t) { return now += ((Graph *)x)->ms, hipSuccess; }
// a window's address range: never touched, only counted
hipError_t hipMemGetAllocationGranularity(size_t *g, const hipMemAllocationProp *, hipMemAllocationGranularity_flags)
{
    return *g = size_t(2) << 20, hipSuccess;
}
hipError_t hipMemAddressReserve(void **p, size_t n, size_t, void *, unsigned long long)
{
    std::lock_guard<std::mutex> l(m);
    *p = (void *)next_range;
    next_range += n + (size_t(1) << 30);
    return hipSuccess;
}
hipError_t hipMemAddressFree(void *, size_t) { return hipSuccess; }
hipError_t hipMemCreate(hipMemGenericAllocationHandle_t *h, size_t n, const hipMemAllocationProp *, unsigned long long)
{
    std::lock_guard<std::mutex> l(m);
    if (n > room - used) return hipErrorOutOfMemory;
    used += n;
    *h = (hipMemGenericAllocationHandle_t) new size_t(n);
    return hipSuccess;
}
hipError_t hipMemRelease(hipMemGenericAllocationHandle_t h)
{
    std::lock_guard<std::mutex> l(m);
    used -= *(size_t *)h;
    delete (size_t *)h;
    return hipSuccess;
}
hipError_t hipMemMap(void *, size_t, size_t, hipMemGenericAllocationHandle_t, unsigned long long) { return hipSuccess; }
hipError_t hipMemUnmap(void *, size_t) { return hipSuccess; }
hipError_t hipMemSetAccess(void *, size_t, const hipMemAccessDesc *, size_t) { return hipSuccess; }
}  // extern "C"
