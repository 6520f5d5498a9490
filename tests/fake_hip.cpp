// A HIP runtime for host-side tests: device memory is host memory with a list of what is allocated, streams run at once, kernels are counted and not run (a captured one when its graph is launched) -- but for the two that carry bytes between
// host and device (csrc/ctx.hip: put_kernel, pin_copy_kernel), which copy.  Loaded in front of the library under test (RTLD_GLOBAL), whose calls it then takes.
// fake_fail(name, n): the n-th call of that name from now on fails; fake_count(name): calls since the last fake_reset(), launches of a kernel also by its name; fake_stray(): bytes that a kernel would have touched outside an allocation.
#include <hip/hip_runtime_api.h>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Alloc { size_t bytes; int device; hipMemoryType type; };
std::map<char *, Alloc> mem;
std::map<std::string, int> count, fail, blocks;
std::map<const void *, std::string> kernels;
int current = 0;
size_t stray = 0, memory = (size_t)288 << 30;
hipError_t last = hipSuccess;
struct Thing { int device; }; // a stream or an event
using Graph = std::vector<std::string>; // the kernels' names
Graph *capturing = nullptr;
hipError_t call(const char *name, hipError_t e = hipSuccess) {
    count[name]++;
    auto f = fail.find(name);
    if (f != fail.end() && --f->second == 0) { fail.erase(f); e = hipErrorUnknown; }
    return e == hipSuccess ? e : last = e;
}
const std::pair<char *const, Alloc> *find(const void *p) {
    auto it = mem.upper_bound((char *)p);
    if (it == mem.begin()) return nullptr;
    --it;
    return (char *)p < it->first + it->second.bytes ? &*it : nullptr;
}
bool fits(const void *p, size_t bytes) {
    auto *a = find(p);
    return a && (char *)p + bytes <= a->first + a->second.bytes;
}
void move(void *dst, const void *src, size_t bytes, bool dst_known, bool src_known) {
    if ((dst_known && !fits(dst, bytes)) || (src_known && !fits(src, bytes))) { stray += bytes; return; }
    memcpy(dst, src, bytes);
}
hipError_t alloc(void **p, size_t bytes, hipMemoryType type) {
    *p = calloc(1, bytes ? bytes : 1);
    mem[(char *)*p] = Alloc{bytes, current, type};
    return hipSuccess;
}
} // namespace

extern "C" {
void fake_reset() { blocks.clear(); count.clear(); fail.clear(); stray = 0; last = hipSuccess; }
void fake_fail(const char *name, int n) { fail[name] = n; }
int fake_count(const char *name) { // (of every name with this in it: a kernel's is mangled)
    int n = 0;
    for (auto &c : count)
        if (c.first.find(name) != std::string::npos) n += c.second;
    return n;
}
size_t fake_stray() { return stray; }
void fake_memory(size_t bytes) { memory = bytes; } // the device's memory in all
size_t fake_held() { // device memory that is allocated
    size_t n = 0;
    for (auto &a : mem) n += a.second.type == hipMemoryTypeDevice ? a.second.bytes : 0;
    return n;
}
int fake_blocks(const char *name) { // work-groups of the last launch of such a kernel
    for (auto &b : blocks)
        if (b.first.find(name) != std::string::npos) return b.second;
    return 0;
}

void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) { kernels[host] = name; }
static struct { dim3 grid, block; size_t lds; hipStream_t st; } config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) { config = {g, b, s, st}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st) { *g = config.grid; *b = config.block; *s = config.lds; *st = config.st; return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t s) {
    if (s && ((Thing *)s)->device != current) return call("hipLaunchKernel", hipErrorInvalidHandle);
    const std::string &n = kernels[f];
    if (n.find("pin_copy_kernel") != std::string::npos) {
        if (call("pin_copy_kernel")) return hipErrorUnknown;
        move(*(void **)args[1], *(void **)args[0], *(size_t *)args[2], true, true);
        return hipSuccess;
    }
    if (n.find("put_kernel") != std::string::npos) { // {dst[4], bytes[4], words}
        if (call("put_kernel")) return hipErrorUnknown;
        char *a = (char *)args[0];
        const unsigned *bytes = (unsigned *)(a + 32);
        const char *v = a + 48;
        for (int i = 0; i < 4; v += (bytes[i] + 3) / 4 * 4, i++)
            if (bytes[i]) move(((void **)a)[i], v, bytes[i], true, false);
        return hipSuccess;
    }
    blocks[n] = (int)(grid.x * grid.y * grid.z);
    if (capturing) { capturing->push_back(n); return hipSuccess; }
    count[n]++;
    return call("hipLaunchKernel");
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { capturing = new Graph; return call("hipStreamBeginCapture"); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = (hipGraph_t)capturing; capturing = nullptr; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) { *e = (hipGraphExec_t) new Graph(*(Graph *)g); return call("hipGraphInstantiate"); }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    for (auto &n : *(Graph *)e) count[n]++;
    return call("hipGraphLaunch");
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete (Graph *)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete (Graph *)e; return hipSuccess; }

hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return call("hipSetDevice"); }
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *, int) { return hipErrorUnknown; }
const char *hipGetErrorString(hipError_t) { return "an error"; }
hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return call("hipGetLastError", e) ? (last = hipSuccess, hipErrorUnknown) : hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return hipSuccess; }

hipError_t hipMalloc(void **p, size_t bytes) {
    const hipError_t e = call("hipMalloc");
    return e != hipSuccess ? e : alloc(p, bytes, hipMemoryTypeDevice);
}
hipError_t hipMemGetInfo(size_t *free, size_t *all) { *free = (size_t)1 << 30; *all = memory; return call("hipMemGetInfo"); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return call("hipHostMalloc") ? hipErrorUnknown : alloc(p, bytes, hipMemoryTypeHost); }
hipError_t hipFree(void *p) { mem.erase((char *)p); free(p); return hipSuccess; }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    auto *f = find(p);
    memset(a, 0, sizeof *a);
    a->type = f ? f->second.type : hipMemoryTypeUnregistered;
    a->device = f ? f->second.device : -2;
    return call("hipPointerGetAttributes", p ? hipSuccess : hipErrorInvalidValue);
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *bytes, hipDeviceptr_t p) {
    auto *f = find(p);
    if (!f) return last = hipErrorNotFound;
    *base = f->first;
    *bytes = f->second.bytes;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t) {
    if (call("hipMemcpyAsync")) return hipErrorUnknown;
    if (!dst || !src || !fits(kind == hipMemcpyHostToDevice ? dst : src, bytes)) return last = hipErrorInvalidValue;
    memmove(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind) { return hipMemcpyAsync(dst, src, bytes, kind, nullptr); }
hipError_t hipMemsetAsync(void *dst, int v, size_t bytes, hipStream_t) { if (!fits(dst, bytes)) return last = hipErrorInvalidValue; memset(dst, v, bytes); return hipSuccess; }
hipError_t hipMemset(void *dst, int v, size_t bytes) { return hipMemsetAsync(dst, v, bytes, nullptr); }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t) new Thing{current}; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete (Thing *)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return call("hipStreamSynchronize"); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t) new Thing{current}; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Thing *)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return call("hipEventRecord", ((Thing *)e)->device == ((Thing *)s)->device ? hipSuccess : hipErrorInvalidHandle); }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return call("hipEventSynchronize"); }
}
