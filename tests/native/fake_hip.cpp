// A HIP runtime without a GPU, for host tests of what the library queues and waits for: linked in front of libamdhip64, it
// answers the calls that the kernel library makes.  Kernels do not run, device memory is address space that nobody can read,
// and what a copy brings to the host is zero.  Queued work is counted per stream, and who is ordered behind what is
// kept as one count per stream (streams of hipStreamCreateWithFlags do not wait for the default stream).
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
typedef std::map<const void*, unsigned long> Seen;      // stream -> items of it that lie behind
struct Alloc {
    size_t bytes;
    int device;
};
std::recursive_mutex mu;
std::map<const void*, Seen> streams;                     // of each stream: what its next item is ordered behind, itself included
Seen host;                                               // what the host has waited for
std::map<const char*, Alloc> memory;
struct Kernel {
    std::string name;                                     // mangled
    unsigned long launched = 0;
};
// by the host's stub; made by the first registration, which comes before this library's own variables are
std::map<const void*, Kernel>& kernels() {
    static std::map<const void*, Kernel> k;
    return k;
}
unsigned long launches = 0, copies = 0, waits = 0;
unsigned long failing = 0;                               // launches that fail from now on
thread_local hipError_t last_error = hipSuccess;
unsigned long limit = ~0ul;                              // bytes of the device's memory
thread_local int device = 0;
char symbol[1 << 24];

void merge(Seen& a, const Seen& b) {
    for (const auto& e : b)
        if (a[e.first] < e.second) a[e.first] = e.second;
}
void push(const void* s) { streams[s][s]++; }
typedef std::lock_guard<std::recursive_mutex> Lock;
const Alloc* block_of(const void* p, const char** base) {
    auto it = memory.upper_bound((const char*)p);
    if (it == memory.begin()) return nullptr;
    --it;
    if ((const char*)p >= it->first + it->second.bytes) return nullptr;
    *base = it->first;
    return &it->second;
}
}  // namespace

extern "C" {
// ---- for the tests
// items of `stream` that the host has not waited for
unsigned long fake_pending(const void* stream) { Lock l(mu); return streams[stream][stream] - host[stream]; }
// streams with work that neither the host nor the default stream has been made to wait for
unsigned long fake_unjoined() {
    Lock l(mu);
    unsigned long n = 0;
    for (auto& s : streams) {
        if (!s.first) continue;
        const unsigned long queued = s.second[s.first];
        if (queued > host[s.first] && queued > streams[nullptr][s.first]) n++;
    }
    return n;
}
// device memory allocated now
unsigned long fake_bytes() {
    Lock l(mu);
    unsigned long n = 0;
    for (auto& a : memory) n += a.second.bytes;
    return n;
}
// no more than `bytes` can be allocated together from now on
void fake_limit(unsigned long bytes) { limit = bytes; }
// the next n launches fail
void fake_fail_launches(unsigned long n) { failing = n; }
unsigned long fake_launches() { return launches; }
// launches of the kernels whose name holds `part`
unsigned long fake_launched(const char* part) {
    Lock l(mu);
    unsigned long n = 0;
    for (auto& k : kernels())
        if (k.second.name.find(part) != std::string::npos) n += k.second.launched;
    return n;
}
unsigned long fake_copies() { return copies; }
// waits of the host for a stream, an event or the device
unsigned long fake_waits() { return waits; }
void fake_queue(const void* stream) { Lock l(mu); push(stream); }

void fake_set_device(int d) { device = d; }

// ---- the runtime
hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
hipError_t hipSetDevice(int d) { device = d; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
hipError_t hipMalloc(void** p, size_t bytes) {
    Lock l(mu);
    bytes = (bytes + 4095) & ~(size_t)4095;
    if (limit != ~0ul && fake_bytes() + bytes > limit) return hipErrorOutOfMemory;
    void* m = mmap(nullptr, bytes, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return hipErrorOutOfMemory;
    memory[(const char*)m] = Alloc{bytes, device};
    *p = m;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    Lock l(mu);
    waits++;
    for (auto& s : streams) merge(host, s.second);
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    Lock l(mu);
    (void)hipDeviceSynchronize();
    auto it = memory.find((const char*)p);
    if (it == memory.end()) return p ? hipErrorInvalidValue : hipSuccess;
    munmap(p, it->second.bytes);
    memory.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { *p = calloc(1, bytes); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s) {
    Lock l(mu);
    if (kind == hipMemcpyDeviceToDevice)                     // inside one block at each end
        for (const void* p : {(const void*)dst, src}) {
            const char* base;
            const Alloc* b = block_of(p, &base);
            if (!b || (const char*)p + bytes > base + b->bytes) return hipErrorInvalidValue;
        }
    push(s);
    copies++;
    if (kind == hipMemcpyDeviceToHost) memset(dst, 0, bytes);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    Lock l(mu);
    const char* base;
    const Alloc* b = block_of(p, &base);
    if (!b) return hipErrorInvalidValue;
    memset(a, 0, sizeof *a);
    a->type = hipMemoryTypeDevice;
    a->device = b->device;
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p) {
    Lock l(mu);
    const char* start;
    const Alloc* b = block_of(p, &start);
    if (!b) return hipErrorInvalidValue;
    *base = (hipDeviceptr_t)start;
    *size = b->bytes;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = symbol; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)malloc(16); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { Lock l(mu); waits++; merge(host, streams[s]); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { Lock l(mu); merge(streams[s], *(Seen*)e); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t) new Seen(); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Seen*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { Lock l(mu); *(Seen*)e = streams[s]; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { Lock l(mu); waits++; merge(host, *(Seen*)e); return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }

thread_local struct { dim3 grid, block; size_t shared; hipStream_t stream; } config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) { config = {g, b, sh, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* s) {
    *g = config.grid;
    *b = config.block;
    *sh = config.shared;
    *s = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* stub, dim3, dim3, void**, size_t, hipStream_t s) {
    Lock l(mu);
    if (failing) {
        failing--;
        return last_error = hipErrorLaunchFailure;
    }
    push(s);
    launches++;
    kernels()[stub].launched++;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { static void* handle; return &handle; }
void __hipRegisterFunction(void**, const void* stub, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { kernels()[stub].name = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}
