// C-ABI (include/ps_hip.h): context, device memory, stream and events -- the part of the library every model family sits on.
#include "ps_internal.h"

#include <algorithm>
#include <cstdio>
#include <cstring>

// ------------------------------------------------------------------ small data in, results out (ps_internal.h)
namespace {
template <int W> struct PutArgs { unsigned char *dst[4]; unsigned bytes[4]; uint32_t v[W]; }; // the pieces' words one behind the other
template <int W>
__global__ void put_kernel(const PutArgs<W> a) {
    for (unsigned i = threadIdx.x; i < W; i += blockDim.x) {
        unsigned w = i;
        int s = 0;
        while (s < 4 && w >= (a.bytes[s] + 3) / 4) w -= (a.bytes[s++] + 3) / 4;
        if (s == 4) return;
        if (w * 4 + 4 <= a.bytes[s]) ((uint32_t *)a.dst[s])[w] = a.v[i];
        else for (unsigned b = w * 4; b < a.bytes[s]; b++) a.dst[s][b] = (unsigned char)(a.v[i] >> (b % 4 * 8));
    }
}
template <int W>
hipError_t put_launch(hipStream_t st, const ps_piece *p, int n) { // n <= 4 pieces of at most W words in all
    PutArgs<W> a{};
    size_t at = 0;
    for (int i = 0; i < n; i++) {
        a.dst[i] = (unsigned char *)p[i].dst;
        a.bytes[i] = (unsigned)p[i].bytes;
        memcpy(a.v + at, p[i].src, p[i].bytes);
        at += (p[i].bytes + 3) / 4;
    }
    void *args[] = {&a};
    return hipLaunchKernel((const void *)put_kernel<W>, dim3(1), dim3(W < 256 ? 64 : 256), args, 0, st); // (its own result: hipGetLastError may hold somebody else's)
}
__global__ __launch_bounds__(256) void pin_copy_kernel(const char *src, char *dst, size_t bytes) {
    const bool wide = (((uintptr_t)src | (uintptr_t)dst) & 15) == 0;
    const size_t n16 = wide ? bytes / 16 : 0, step = (size_t)gridDim.x * blockDim.x, t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (size_t i = t; i < n16; i += step) ((uint4 *)dst)[i] = ((const uint4 *)src)[i];
    for (size_t i = n16 * 4 + t; i < bytes / 4; i += step) ((uint32_t *)dst)[i] = ((const uint32_t *)src)[i];
}
} // namespace
hipError_t ps_put(hipStream_t st, const ps_piece *p, int n) {
    constexpr size_t CAP = 896;
    size_t total = 0;
    for (int i = 0; i < n; i++) total += p[i].bytes;
    if (total > PS_PUT_MAX) {
        hipError_t e = hipSuccess;
        for (int i = 0; i < n && e == hipSuccess; i++)
            if (p[i].bytes) e = hipMemcpyAsync(p[i].dst, p[i].src, p[i].bytes, hipMemcpyHostToDevice, st);
        const hipError_t w = hipStreamSynchronize(st); // (the sources may be temporaries)
        return e != hipSuccess ? e : w;
    }
    ps_piece q[4];
    int k = 0;
    size_t words = 0;
    auto flush = [&]() {
        const hipError_t e = !k ? hipSuccess : words <= 32 ? put_launch<32>(st, q, k) : put_launch<CAP>(st, q, k);
        k = 0; words = 0;
        return e;
    };
    for (int i = 0; i < n; i++) {
        for (size_t done = 0; done < p[i].bytes;) {
            const size_t b = std::min(p[i].bytes - done, (CAP - words) * 4);
            q[k++] = ps_piece{(char *)p[i].dst + done, (const char *)p[i].src + done, b};
            words += (b + 3) / 4;
            done += b;
            if (k == 4 || words == CAP)
                if (const hipError_t e = flush()) return e;
        }
    }
    return flush();
}
bool ps_pin_ready(ps_hip_ctx *c) {
    if (c->pin) return true;
    if (hipSetDevice(c->device) != hipSuccess) { (void)hipGetLastError(); return false; } // (an event belongs to the device that is current)
    for (auto &e : c->pin_ev)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) { e = nullptr; (void)hipGetLastError(); return false; }
    if (hipHostMalloc((void **)&c->pin, 2 * PS_PIN_HALF, hipHostMallocDefault) != hipSuccess) { c->pin = nullptr; (void)hipGetLastError(); return false; }
    return true;
}
void ps_pin_copy(ps_hip_ctx *c, int half, size_t at, const void *dev, size_t bytes) {
    const unsigned blocks = (unsigned)std::min<size_t>((bytes + 4095) / 4096, 256);
    hipLaunchKernelGGL(pin_copy_kernel, dim3(blocks), dim3(256), 0, c->stream, (const char *)dev, c->pin + half * PS_PIN_HALF + at, bytes);
}

// Whether a caller's copy to the host may be a kernel that reads src: src lies whole in an allocation of the context's device and dst is host memory.  A copy checks its operands and comes back
// with an error, a kernel faults; what is not known to be in order is left to the copy.
static bool kernel_may_copy(const ps_hip_ctx *c, const void *dst, const void *src, size_t bytes) {
    hipPointerAttribute_t s{}, d{};
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    int dev = -1;
    if (!dst || !src || hipGetDevice(&dev) != hipSuccess || dev != c->device) return false; // (a copy may be enqueued whichever device is current, a kernel not)
    if (hipPointerGetAttributes(&s, src) != hipSuccess || s.type != hipMemoryTypeDevice || s.device != c->device || hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)src) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if ((size_t)((const char *)src - (const char *)base) + bytes > size) return false;
    if (hipPointerGetAttributes(&d, dst) != hipSuccess) { (void)hipGetLastError(); return true; } // (pageable memory, to runtimes that do not say so)
    return d.type == hipMemoryTypeUnregistered || d.type == hipMemoryTypeHost;
}

extern "C" {

int ps_hip_abi_version(void) { return PS_HIP_ABI_VERSION; }

int ps_hip_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}


int ps_hip_create(int device, ps_hip_ctx **out) {
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0 || device >= n) return 1;
    if (hipSetDevice(device) != hipSuccess) return 1;
    auto c    = new ps_hip_ctx();
    c->device = device;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) c->n_cu = prop.multiProcessorCount;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) { delete c; return 1; }
    *out = c;
    return 0;
}

void ps_hip_destroy(ps_hip_ctx *c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    if (c->act_buf) (void)hipFree(c->act_buf);
    if (c->i32_buf) (void)hipFree(c->i32_buf);
    if (c->u8_buf) (void)hipFree(c->u8_buf);
    if (c->rope_buf) (void)hipFree(c->rope_buf);
    if (c->pin) (void)hipHostFree(c->pin);
    for (auto e : c->pin_ev) if (e) (void)hipEventDestroy(e);
    (void)hipStreamDestroy(c->stream);
    delete c;
}

const char *ps_hip_last_error(const ps_hip_ctx *c) { return c ? c->err.c_str() : "no context"; }

int ps_hip_device_name(const ps_hip_ctx *c, char *buf, size_t cap) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, c->device) != hipSuccess) return 1;
    snprintf(buf, cap, "%s (%s, %d CUs)", prop.name, prop.gcnArchName, prop.multiProcessorCount);
    return 0;
}

int ps_hip_malloc(ps_hip_ctx *c, size_t bytes, void **dptr) {
    PS_CHECK(c, hipSetDevice(c->device));
    PS_CHECK(c, hipMalloc(dptr, bytes ? bytes : 16));
    return 0;
}
int ps_hip_free(ps_hip_ctx *c, void *dptr) {
    PS_CHECK(c, hipStreamSynchronize(c->stream));
    PS_CHECK(c, hipFree(dptr));
    return 0;
}
int ps_hip_memcpy_h2d(ps_hip_ctx *c, void *dst, const void *src, size_t bytes) {
    PS_CHECK(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
    PS_CHECK(c, hipStreamSynchronize(c->stream));
    return 0;
}
int ps_hip_memcpy_d2h(ps_hip_ctx *c, void *dst, const void *src, size_t bytes) {
    if (bytes && bytes % 4 == 0 && bytes <= PS_PIN_WAITED && ((uintptr_t)src & 3) == 0 && kernel_may_copy(c, dst, src, bytes) && ps_pin_ready(c)) {
        ps_pin_copy(c, 0, 0, src, bytes);
        PS_CHECK(c, hipStreamSynchronize(c->stream));
        memcpy(dst, c->pin, bytes);
        return 0;
    }
    PS_CHECK(c, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c->stream));
    PS_CHECK(c, hipStreamSynchronize(c->stream));
    return 0;
}
int ps_hip_memset(ps_hip_ctx *c, void *dst, int value, size_t bytes) {
    PS_CHECK(c, hipMemsetAsync(dst, value, bytes, c->stream));
    return 0;
}
int ps_hip_sync(ps_hip_ctx *c) {
    PS_CHECK(c, hipStreamSynchronize(c->stream));
    PS_CHECK(c, hipGetLastError());
    return 0;
}
void *ps_hip_stream(ps_hip_ctx *c) { return (void *)c->stream; }

int ps_hip_event_create(ps_hip_ctx *c, void **ev) {
    hipEvent_t e;
    PS_CHECK(c, hipEventCreate(&e));
    *ev = (void *)e;
    return 0;
}
int ps_hip_event_record(ps_hip_ctx *c, void *ev) {
    PS_CHECK(c, hipEventRecord((hipEvent_t)ev, c->stream));
    return 0;
}
int ps_hip_event_elapsed_ms(ps_hip_ctx *c, void *a, void *b, float *ms) {
    PS_CHECK(c, hipEventSynchronize((hipEvent_t)b));
    PS_CHECK(c, hipEventElapsedTime(ms, (hipEvent_t)a, (hipEvent_t)b));
    return 0;
}
int ps_hip_event_destroy(ps_hip_ctx *c, void *ev) {
    PS_CHECK(c, hipEventDestroy((hipEvent_t)ev));
    return 0;
}

} // extern "C"
