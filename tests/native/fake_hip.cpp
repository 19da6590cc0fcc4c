// A HIP runtime on the host for tests of libgsim's host code: device memory is
// host memory, streams run at once, kernels do nothing but leave their name
// (read_kernel copies, as on the device).  Loaded with RTLD_GLOBAL ahead of
// libgsim.so, it answers that library's HIP calls.  Failures are asked for by
// the fake_* functions.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <thread>

namespace {

std::recursive_mutex mu;
std::map<const void *, std::string> kernels;  // host stub -> device name
std::map<void *, size_t> blocks;              // live device allocations
size_t live = 0, limit = ~(size_t)0;
std::string launches, faults;
std::set<void *> capturing, spoiled;  // streams in capture; captures made invalid
unsigned capture_delay_us = 0, instantiated = 0, refused_graphs = 0;
// Memsets and copies on the device return before they are done; the library's
// streams do not wait for the null stream.
bool null_busy = false;
char token;  // every stream, event and graph but the null stream is some address

void fault(const std::string &what) { faults += what + "\n"; }

void *fresh() { return std::malloc(1); }

template <typename T>
T arg(void **args, int k) {
    return *static_cast<T *>(args[k]);
}

// read_kernel(pos, vel, mass, perm, na, n, pos_out, vel_out, mass_out, stall, stall_out)
void read_particles(void **a) {
    struct F2 {
        float x, y;
    };
    const F2 *pos = arg<const F2 *>(a, 0), *vel = arg<const F2 *>(a, 1);
    const float *mass = arg<const float *>(a, 2);
    const uint32_t *perm = arg<const uint32_t *>(a, 3);
    F2 *po = arg<F2 *>(a, 6), *vo = arg<F2 *>(a, 7);
    float *mo = arg<float *>(a, 8);
    const uint32_t *in = arg<const uint32_t *>(a, 9);
    uint32_t *out = arg<uint32_t *>(a, 10);
    if (!po || !vo || !mo) return fault("read_kernel writes to address 0");
    if (in) *out = *in;
    for (uint32_t k = 0; k < arg<uint32_t>(a, 4); ++k) {
        const uint32_t i = perm ? perm[k] : k;
        if (i >= arg<uint32_t>(a, 5)) continue;
        po[i] = pos[k];
        vo[i] = vel[k];
        mo[i] = mass[k];
    }
}

hipError_t allocate(void **p, size_t n) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    *p = nullptr;
    if (n > limit || live > limit - n) return hipErrorOutOfMemory;
    *p = std::calloc(n ? n : 1, 1);
    if (!*p) return hipErrorOutOfMemory;
    blocks[*p] = n;
    live += n;
    return hipSuccess;
}

hipError_t release(void *p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (!p) return hipSuccess;
    auto it = blocks.find(p);
    if (it == blocks.end()) {
        fault("free of an unknown address");
        return hipErrorInvalidValue;
    }
    live -= it->second;
    blocks.erase(it);
    std::free(p);
    return hipSuccess;
}

hipError_t copy(void *d, const void *s, size_t n) {
    if (n && (!d || !s)) return hipErrorInvalidValue;
    if (n) std::memcpy(d, s, n);
    return hipSuccess;
}

}  // namespace

extern "C" {

static void starts_on(hipStream_t st) {
    if (st && null_busy) fault("work starts beside an unfinished one of the null stream");
}

// ---- what a test asks for and looks at ---------------------------------------
void fake_limit(size_t bytes) { limit = bytes; }  // of device memory held at once
size_t fake_live() { return live; }
void fake_capture_delay(unsigned us) { capture_delay_us = us; }  // a launch under capture
void fake_refuse_graphs(unsigned n) { refused_graphs = n; }  // the next n instantiations
void fake_forget() { launches.clear(); }
const char *fake_launches() { return launches.c_str(); }  // names, a line each
const char *fake_faults() { return faults.c_str(); }
unsigned fake_instantiated() { return instantiated; }

// ---- the runtime ----------------------------------------------------------------
void **__hipRegisterFatBinary(const void *) { return (void **)&token; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
static thread_local Config config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
    config = Config{g, b, sh, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *st) {
    *g = config.grid;
    *b = config.block;
    *sh = config.shared;
    *st = config.stream;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t st) {
    unsigned wait = 0;
    {
        std::lock_guard<std::recursive_mutex> lk(mu);
        const std::string &name = kernels[f];
        launches += name + "\n";
        if (!capturing.count(st)) starts_on(st);
        auto is = [&](const char *k) { return name.find(k) != std::string::npos; };
        if (is("read_kernel")) read_particles(args);
        if ((is("ds_partial_kernel") || is("ds_sym_kernel")) && !arg<void *>(args, 2))
            fault(name + " writes partial sums to address 0");
        if (is("bh_leaf_kernel") && !arg<void *>(args, 0)) fault(name + " reads address 0");
        if (capturing.count(st)) wait = capture_delay_us;
    }
    if (wait) std::this_thread::sleep_for(std::chrono::microseconds(wait));
    return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t n) { return allocate(p, n); }
hipError_t hipFree(void *p) { return release(p); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::calloc(n, 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind kind) {
    null_busy = kind == hipMemcpyDeviceToDevice;  // the others wait for all before
    return copy(d, s, n);
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
    starts_on(st);
    return copy(d, s, n);
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) {
    if (n && !d) return hipErrorInvalidValue;
    starts_on(st);
    if (!st) null_busy = true;
    if (!v && n > ((size_t)64 << 20)) {  // give the pages back instead of touching them
        const uintptr_t p = (uintptr_t)d, a = (p + 4095) / 4096 * 4096, b = (p + n) / 4096 * 4096;
        std::memset(d, 0, a - p);
        madvise((void *)a, b - a, MADV_DONTNEED);
        std::memset((void *)b, 0, p + n - b);
    } else if (n) {
        std::memset(d, v, n);
    }
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { return hipMemsetAsync(d, v, n, nullptr); }

hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    *p = &token;
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = (hipStream_t)fresh();
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (!s) null_busy = false;
    if (!capturing.count(s)) return hipSuccess;
    spoiled.insert(s);
    fault("a stream under capture is waited for");
    return hipErrorStreamCaptureUnsupported;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    capturing.insert(s);
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    capturing.erase(s);
    *g = nullptr;
    if (spoiled.erase(s)) return hipErrorStreamCaptureInvalidated;
    *g = (hipGraph_t)fresh();
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (refused_graphs) {
        --refused_graphs;
        return hipErrorUnknown;
    }
    ++instantiated;
    *e = (hipGraphExec_t)fresh();
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t st) {
    starts_on(st);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    std::free(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    std::free(e);
    return hipSuccess;
}

hipError_t hipEventCreate(hipEvent_t *e) {
    *e = (hipEvent_t)fresh();
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }

}  // extern "C"
