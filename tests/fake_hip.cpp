// A stand-in for the HIP runtime, for tests of the library's host code without a GPU: device memory is
// host memory filled with zeros, a launch only notes the kernel's name, and an allocation can be made to
// fail.  Loaded into the global scope before libefe_gpu.so, whose references it then serves.
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const void*, std::string> kernels;
std::string launches;
long allocations = 0, failing = -1;
int last = 0;
constexpr int kOutOfMemory = 2;
int memory(void** p, size_t n) {
    if (allocations++ == failing) return last = kOutOfMemory;
    *p = calloc(n ? n : 1, 1);
    return *p ? 0 : (last = kOutOfMemory);
}
struct Dim {
    uint32_t x, y, z;
};
Dim cfgGrid, cfgBlock;
size_t cfgShared;
void* cfgStream;
}  // namespace

extern "C" {
// the tests' side: the k-th allocation from now on fails (-1: none); names of the kernels launched since
void fake_fail(long k) {
    allocations = 0;
    failing = k;
}
long fake_allocations() { return allocations; }
const char* fake_launches() {
    static std::string out;
    out.swap(launches);
    launches.clear();
    return out.c_str();
}

void** __hipRegisterFatBinary(const void*) { return (void**)malloc(8); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
    kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim g, Dim b, size_t sh, void* st) {
    cfgGrid = g, cfgBlock = b, cfgShared = sh, cfgStream = st;
    return 0;
}
int __hipPopCallConfiguration(Dim* g, Dim* b, size_t* sh, void** st) {
    *g = cfgGrid, *b = cfgBlock, *sh = cfgShared, *st = cfgStream;
    return 0;
}
int hipLaunchKernel(const void* f, Dim, Dim, void**, size_t, void*) {
    launches += kernels[f] + "\n";
    return 0;
}
int hipMalloc(void** p, size_t n) { return memory(p, n); }
int hipHostMalloc(void** p, size_t n, unsigned) { return memory(p, n); }
int hipFree(void* p) { return free(p), 0; }
int hipHostFree(void* p) { return free(p), 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { return memcpy(d, s, n), 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { return memcpy(d, s, n), 0; }
int hipMemsetAsync(void* d, int v, size_t n, void*) { return memset(d, v, n), 0; }
int hipGetLastError() {
    const int e = last;
    last = 0;
    return e;
}
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : e ? "error" : "no error"; }
int hipGetDevice(int* d) { return *d = 0; }
int hipGetSymbolAddress(void** p, const void*) { return *p = nullptr, 0; }
int hipDeviceSynchronize() { return 0; }
int hipEventCreate(void** e) { return *e = malloc(1), 0; }
int hipEventCreateWithFlags(void** e, unsigned) { return *e = malloc(1), 0; }
int hipEventDestroy(void* e) { return free(e), 0; }
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 0.0f, 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipGraphDestroy(void* g) { return free(g), 0; }
int hipGraphExecDestroy(void* g) { return free(g), 0; }
int hipGraphInstantiate(void** e, void*, void**, char*, size_t) { return *e = malloc(1), 0; }
int hipGraphLaunch(void*, void*) { return 0; }
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) { return *g = malloc(1), 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { return *s = malloc(1), 0; }
int hipStreamDestroy(void* s) { return free(s), 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
}
