// A stand-in for the HIP runtime calls of libdvmh_amd.so and of converted
// programs, for tests of host decisions on a machine without a GPU: device
// memory is reserved address space that nothing touches, launches and copies
// do nothing but are written down, a completion word is reached as soon as the
// stream is asked.  Load it (RTLD_GLOBAL) before the runtime.  Test
// infrastructure only: no result computed through it means anything.
#include <dlfcn.h>
#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include <hip/hip_runtime_api.h>

namespace {

struct Launch {
    std::string name;
    unsigned grid, block;
};
std::vector<Launch> launches;   // the first KEPT of them
constexpr size_t KEPT = 4096;
long launched = 0;
std::map<char *, size_t> blocks, pinned;
size_t capacity = (size_t)288 << 30, used = 0;
long syncs = 0, asked = 0, refused = 0, graphs = 0;
bool capturing = false;
dim3 configGrid, configBlock;

// every word the device would have set
void complete() {
    for (auto &b : pinned)
        if (b.second >= 1024 && b.second < 4096) *(volatile unsigned long long *)b.first = 1ULL << 62;
}

}  // namespace

extern "C" {

void fake_capacity(long bytes) { capacity = (size_t)bytes; }
long fake_used() { return (long)used; }
long fake_refused() { return refused; }
long fake_asked() { return asked; }   // hipMalloc calls
long fake_syncs() { return syncs; }
long fake_graphs() { return graphs; }
// p lies in memory the device has handed out and not taken back
int fake_live(const void *p) {
    auto it = blocks.upper_bound((char *)p);
    if (it == blocks.begin()) return 0;
    --it;
    return (char *)p < it->first + it->second;
}
void fake_clear() { launches.clear(); launched = 0; }
long fake_launches() { return launched; }
const char *fake_launch_name(long i) { return launches[(size_t)i].name.c_str(); }
long fake_launch_grid(long i) { return launches[(size_t)i].grid; }
long fake_launch_block(long i) { return launches[(size_t)i].block; }

hipError_t hipMalloc(void **p, size_t bytes) {
    asked++;
    if (used + bytes > capacity) {
        refused++;
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    void *m = mmap(nullptr, bytes, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return hipErrorOutOfMemory;
    blocks[(char *)m] = bytes;
    used += bytes;
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    auto it = blocks.find((char *)p);
    if (it == blocks.end()) {
        fprintf(stderr, "fake_hip: hipFree of %p, which is not allocated\n", p);
        abort();
    }
    munmap(p, it->second);
    used -= it->second;
    blocks.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    *p = calloc(1, bytes);
    pinned[(char *)*p] = bytes;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    pinned.erase((char *)p);
    free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    p->maxThreadsPerBlock = 1024;
    p->maxThreadsDim[0] = p->maxThreadsDim[1] = p->maxThreadsDim[2] = 1024;
    p->sharedMemPerBlock = 65536;
    p->regsPerMultiprocessor = 131072;
    snprintf(p->name, sizeof(p->name), "fake");
    snprintf(p->gcnArchName, sizeof(p->gcnArchName), "gfx950");
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) { memset(a, 0, sizeof(*a)); a->numRegs = 64; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static char *word = nullptr;
    if (!word && hipMalloc((void **)&word, 4096) != hipSuccess) return hipErrorOutOfMemory;
    *p = word;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *free_, size_t *total) { *free_ = capacity - used; *total = capacity; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceSynchronize() { complete(); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    static char handles[64];
    static int n = 0;
    *s = (hipStream_t)&handles[n++];
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { syncs++; complete(); return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { complete(); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { complete(); return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { capturing = true; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { capturing = false; *g = (hipGraph_t)malloc(1); return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { *e = (hipGraphExec_t)malloc(1); graphs++; return hipSuccess; }
hipError_t hipGraphGetNodes(hipGraph_t, hipGraphNode_t *, size_t *n) { *n = 1000; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { launched++; launches.push_back({"graph", 1, 1}); return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { free(g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { free(e); graphs--; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
    configGrid = grid;
    configBlock = block;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    *grid = configGrid;
    *block = configBlock;
    *lds = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **, size_t, hipStream_t) {
    if (launched++ >= (long)KEPT) return hipSuccess;
    Dl_info info;
    const char *name = dladdr(f, &info) && info.dli_sname ? info.dli_sname : "?";
    if ((unsigned long)grid.x * block.x >= 1UL << 32) name = "too large";
    launches.push_back({name, grid.x * grid.y * grid.z, block.x * block.y * block.z});
    return hipSuccess;
}

}  // extern "C"
