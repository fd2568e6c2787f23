// A stand-in for the HIP runtime, preloaded by test_host_runtime.py: device
// memory is host memory, copies are memcpy, launches run nothing but are
// counted and, where their tables can be read, checked.  stub_count(what)
// tells how often a call was made, stub_fail(what, n) makes its n-th call
// from now on fail once, stub_bad() counts what was found wrong.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <chrono>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace {

struct State {
    std::recursive_mutex mu;
    std::map<const void*, std::string> kernel;
    std::map<std::string, long> count, fail;
    std::map<char*, size_t> dev, host;
    size_t dev_bytes = 0;
    long bad = 0;
    int band_rows = 0;   // of the last batched band coherence
    bool capturing = false;
    int sync_ms = 0;     // what a stream synchronisation takes
};
State& st()
{
    static State* s = new State;   // never destroyed: used while others are
    return *s;
}

// counts the call; true: it is to fail
bool called(const char* what)
{
    std::lock_guard<std::recursive_mutex> l(st().mu);
    st().count[what]++;
    auto f = st().fail.find(what);
    return f != st().fail.end() && f->second > 0 && --f->second == 0;
}

void bad(const char* what)
{
    fprintf(stderr, "hip_stub: %s\n", what);
    st().bad++;
}

bool inside(const std::map<char*, size_t>& m, const void* p, size_t n)
{
    auto it = m.upper_bound((char*)p);
    if (it == m.begin()) return false;
    --it;
    return (char*)p + n <= it->first + it->second;
}

struct CohItem {   // tops::CohItem
    const void *m, *s;
    float* coh;
    int w, h;
};
struct Int4 { int x, y, z, w; };

// the batched band coherence: each workgroup's rows lie in its raster and all
// rasters are covered
void check_band_batch(void** a, unsigned grid)
{
    const CohItem* items = *(const CohItem**)a[0];
    const Int4* work = *(const Int4**)a[1];
    const int rows = *(int*)a[5];
    st().band_rows = rows;
    if (!inside(st().dev, work, sizeof(Int4) * grid)) return bad("band table too short");
    std::map<int, long> covered, blocks_x;
    for (unsigned i = 0; i < grid; i++) {
        const CohItem& c = items[work[i].x];
        if (work[i].z * rows >= c.h) return bad("band workgroup past its raster");
        if (work[i].y + 1 > blocks_x[work[i].x]) blocks_x[work[i].x] = work[i].y + 1;
        const int r0 = work[i].z * rows;
        covered[work[i].x] += (r0 + rows < c.h ? r0 + rows : c.h) - r0;
    }
    for (auto& k : covered)
        if (k.second != (long)items[k.first].h * blocks_x[k.first]) bad("raster rows not covered");
}

struct Config { dim3 grid, block; size_t lds; hipStream_t s; };
thread_local std::vector<Config> g_config;

}  // namespace

extern "C" {

long stub_count(const char* what) { return st().count[what]; }
void stub_fail(const char* what, long nth) { st().fail[what] = nth; }
long stub_bad() { return st().bad; }
int stub_band_rows() { return st().band_rows; }
void stub_sync_ms(int ms) { st().sync_ms = ms; }
// what hipDeviceReset does to the memory of the device
void stub_reset()
{
    std::lock_guard<std::recursive_mutex> l(st().mu);
    st().dev.clear();
    st().host.clear();
    st().dev_bytes = 0;
}
size_t stub_device_bytes() { return st().dev_bytes; }
long stub_host_blocks() { return (long)st().host.size(); }

hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    g_config.push_back({g, b, lds, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s)
{
    const Config c = g_config.back();
    g_config.pop_back();
    *g = c.grid;
    *b = c.block;
    *lds = c.lds;
    *s = c.s;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*)
{
    static void* module;
    return &module;
}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*)
{
    st().kernel[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}

hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int)
{
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t)
{
    *n = 4;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    *p = nullptr;
    return hipErrorUnknown;
}

hipError_t hipMalloc(void** p, size_t n)
{
    if (called("hipMalloc")) return hipErrorOutOfMemory;
    std::lock_guard<std::recursive_mutex> l(st().mu);
    *p = malloc(n);
    st().dev[(char*)*p] = n;
    st().dev_bytes += n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    called("hipFree");
    std::lock_guard<std::recursive_mutex> l(st().mu);
    auto it = st().dev.find((char*)p);
    if (it == st().dev.end()) {
        bad("hipFree of an unknown block");
        return hipErrorInvalidValue;
    }
    st().dev_bytes -= it->second;
    st().dev.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    if (called("hipHostMalloc")) return hipErrorOutOfMemory;
    std::lock_guard<std::recursive_mutex> l(st().mu);
    *p = malloc(n);
    st().host[(char*)*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    called("hipHostFree");
    std::lock_guard<std::recursive_mutex> l(st().mu);
    if (!st().host.erase((char*)p)) bad("hipHostFree of an unknown block");
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k)
{
    if (called("hipMemcpy")) return hipErrorUnknown;
    {
        std::lock_guard<std::recursive_mutex> l(st().mu);
        if (!inside(st().dev, k == hipMemcpyHostToDevice ? d : s, n)) {
            bad("copy outside device memory");
            return hipErrorInvalidValue;
        }
    }
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t)
{
    if (called("hipMemcpyAsync")) return hipErrorUnknown;
    if (std::lock_guard<std::recursive_mutex> l(st().mu);
        k == hipMemcpyHostToDevice && !inside(st().host, s, n))
        bad("asynchronous upload of memory that is not pinned");
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemset(void* d, int v, size_t n)
{
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    std::lock_guard<std::recursive_mutex> l(st().mu);
    a->type = inside(st().host, p, 1)  ? hipMemoryTypeHost
              : inside(st().dev, p, 1) ? hipMemoryTypeDevice
                                       : hipMemoryTypeUnregistered;
    return hipSuccess;
}

hipError_t hipStreamCreate(hipStream_t* s)
{
    *s = (hipStream_t)malloc(8);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s)
{
    free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    std::this_thread::sleep_for(std::chrono::milliseconds(st().sync_ms));
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e)
{
    *e = (hipEvent_t)malloc(8);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    // a schedule's time falls with each call, so the last one timed is kept
    *ms = 1.0f + 1000.0f / (float)++st().count["hipEventElapsedTime"];
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
    st().capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
    st().capturing = false;
    *g = (hipGraph_t)malloc(8);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    called("hipGraphInstantiate");
    *x = (hipGraphExec_t)malloc(8);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x)
{
    free(x);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g)
{
    free(g);
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t)
{
    std::lock_guard<std::recursive_mutex> l(st().mu);
    st().count["hipLaunchKernel"]++;
    if (grid.x == 0 || grid.y == 0 || grid.z == 0 || grid.y > 65535 || grid.z > 65535) {
        bad("grid out of the hardware's range");
        return hipErrorInvalidValue;
    }
    const std::string& name = st().kernel[f];
    if (name.find("coherence_band_batch_kernel") != std::string::npos)
        check_band_batch(args, grid.x);
    if (name.find("esd_final_kernel") != std::string::npos ||
        name.find("geocoreg_final_kernel") != std::string::npos)
        if (void* out = *(void**)args[2]; !inside(st().dev, out, 48) && !inside(st().host, out, 48))
            bad("sums written to memory that is not there");
    return hipSuccess;
}

}  // extern "C"
