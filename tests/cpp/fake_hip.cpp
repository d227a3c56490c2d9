// The HIP runtime functions that libicempm.so calls, for a program without a
// GPU: memory is host memory, launches are recorded and not run (but for the
// few kernels below that only move words), and the answers that a test needs
// can be set.  Linked into a test program with -rdynamic, these definitions
// come before the runtime's own.
#include "fake_hip.h"

#include <sys/mman.h>

#include <cstdlib>
#include <cstring>
#include <string>

namespace fake {

State &state()
{
    static State s;
    return s;
}

}  // namespace fake

using fake::state;

struct ihipStream_t { int device; };
struct ihipEvent_t { int device; unsigned flags; };

namespace {

// A failing call leaves its error for hipGetLastError, as in the runtime.
hipError_t done(hipError_t e)
{
    if (e != hipSuccess) state().last_error = e;
    return e;
}

void *map(size_t bytes)
{
    void *p = mmap(nullptr, bytes ? bytes : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    return p == MAP_FAILED ? nullptr : p;
}

// The largest parts of memory are fresh where a test clears them, and zero.
void clear(void *p, size_t n)
{
    if (n < (size_t(1) << 28)) std::memset(p, 0, n);
}

std::map<const void *, std::string> &kernel_names()
{
    static std::map<const void *, std::string> m;
    return m;
}

thread_local dim3 t_grid, t_block;
thread_local size_t t_shared;
thread_local hipStream_t t_stream;

}  // namespace

extern "C" {

void **__hipRegisterFatBinary(const void *)
{
    static void *module;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    kernel_names()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream)
{
    t_grid = grid;
    t_block = block;
    t_shared = shared;
    t_stream = stream;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream)
{
    *grid = t_grid;
    *block = t_block;
    *shared = t_shared;
    *stream = t_stream;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t, hipStream_t)
{
    const std::string &name = kernel_names()[f];
    fake::Launch l;
    l.name = name;
    l.grid = grid;
    l.block = block;
    if (name.find("k_fill_zero") != std::string::npos) {
        void *p = *(void **)args[0];
        const size_t n16 = *(size_t *)args[1], tail = *(size_t *)args[3];
        l.pointer = p;
        clear(p, n16 * 16 + tail);
    } else if (name.find("k_read") != std::string::npos) {
        std::memcpy(*(void **)args[1], *(void **)args[0], *(int *)args[2] * sizeof(unsigned));
    }
    state().launches.push_back(l);
    return done(hipSuccess);
}

hipError_t hipGetDeviceCount(int *n) { *n = state().n_devices; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = state().device; return hipSuccess; }
hipError_t hipSetDevice(int d) { state().device = d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeWallClockRate ? 100000 : 0;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t)
{
    *n = state().occupancy;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **, const void *) { return done(hipErrorInvalidSymbol); }
hipError_t hipGetLastError(void)
{
    const hipError_t e = state().last_error;
    state().last_error = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "error of the test"; }

hipError_t hipMalloc(void **p, size_t bytes)
{
    if (bytes >= state().malloc_limit) return done(hipErrorOutOfMemory);
    *p = map(bytes);
    state().allocated.push_back(bytes);
    return done(*p ? hipSuccess : hipErrorOutOfMemory);
}
hipError_t hipFree(void *) { return hipSuccess; }   // kept mapped: a later use is no fault of the test
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags)
{
    if (state().host_malloc_fails) return done(hipErrorOutOfMemory);
    state().host_flags.push_back(flags);
    *p = std::aligned_alloc(4096, (bytes + 4095) / 4096 * 4096);
    return done(*p ? hipSuccess : hipErrorOutOfMemory);
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t)
{
    if (v == 0) clear(p, n);
    else std::memset(p, v, n);
    return hipSuccess;
}

hipError_t hipStreamCreate(hipStream_t *s) { *s = new ihipStream_t{state().device}; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags)
{
    *e = new ihipEvent_t{state().device, flags};
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecordWithFlags(hipEvent_t e, hipStream_t s, unsigned)
{
    return done(e->device == s->device ? hipSuccess : hipErrorInvalidHandle);   // an event belongs to its device
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return hipEventRecordWithFlags(e, s, 0); }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1; return hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return done(hipErrorNotSupported); }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return done(hipErrorNotSupported); }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return done(hipErrorNotSupported); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return done(hipErrorNotSupported); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"
