// A stand-in for the HIP runtime that runs nothing, so that the library's host side can
// be watched without a GPU: device memory is host memory, copies happen at once, kernels
// are noted and not run. It counts what a call leaves behind: asynchronous copies of host
// memory that no synchronisation has followed, and bytes allocated. Allocations and
// asynchronous copies can be made to fail.
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
enum { kSuccess = 0, kInvalid = 1, kOutOfMemory = 2 };
enum { kHostToDevice = 1, kDeviceToHost = 2 };
struct Dim3 { uint32_t x, y, z; };

std::map<void*, size_t> allocations;
size_t allocated = 0, peak = 0;
int pending = 0;                                    // host copies enqueued since the last synchronisation
long malloc_countdown = -1, copy_countdown = -1;    // 0: the next one fails; negative: none
std::map<const void*, std::string> kernels;
struct Launch { std::string name; Dim3 grid, block; };
std::vector<Launch> launches;
struct Config { Dim3 grid, block; size_t shared; void* stream; };
std::vector<Config> configs;

bool fails(long& countdown) { return countdown >= 0 && countdown-- == 0; }
void drop(void* p) {
    auto it = allocations.find(p);
    if (it == allocations.end()) return;
    allocated -= it->second;
    allocations.erase(it);
    std::free(p);
}
}  // namespace

extern "C" {

// ---- for the tests
int rec_pending() { return pending; }
size_t rec_allocated() { return allocated; }
size_t rec_peak() { return peak; }
void rec_reset_peak() { peak = allocated; }
void rec_fail_malloc(long n) { malloc_countdown = n; }
void rec_fail_copy(long n) { copy_countdown = n; }
void rec_clear_launches() { launches.clear(); }
int rec_launches() { return (int)launches.size(); }
const char* rec_launch(int i, uint32_t* grid) {
    grid[0] = launches[(size_t)i].grid.x;
    grid[1] = launches[(size_t)i].grid.y;
    grid[2] = launches[(size_t)i].grid.z;
    return launches[(size_t)i].name.c_str();
}

// ---- the runtime
int hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (fails(malloc_countdown)) return kOutOfMemory;
    *p = std::calloc(1, n ? n : 1);
    if (!*p) return kOutOfMemory;
    allocations[*p] = n;
    allocated += n;
    if (allocated > peak) peak = allocated;
    return kSuccess;
}
int hipFree(void* p) {   // waits for the device
    pending = 0;
    drop(p);
    return kSuccess;
}
int hipMemcpy(void* dst, const void* src, size_t n, int) { std::memmove(dst, src, n); return kSuccess; }
int hipMemcpyAsync(void* dst, const void* src, size_t n, int kind, void*) {
    if (fails(copy_countdown)) return kInvalid;
    std::memmove(dst, src, n);
    if (kind == kHostToDevice || kind == kDeviceToHost) ++pending;
    return kSuccess;
}
int hipMemsetAsync(void* p, int v, size_t n, void*) { std::memset(p, v, n); return kSuccess; }
int hipStreamSynchronize(void*) { pending = 0; return kSuccess; }
int hipEventSynchronize(void*) { pending = 0; return kSuccess; }
int hipStreamCreateWithFlags(void** s, unsigned) { *s = std::malloc(1); return kSuccess; }
int hipStreamDestroy(void* s) { std::free(s); return kSuccess; }
int hipStreamWaitEvent(void*, void*, unsigned) { return kSuccess; }
int hipEventCreate(void** e) { *e = std::malloc(1); return kSuccess; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = std::malloc(1); return kSuccess; }
int hipEventDestroy(void* e) { std::free(e); return kSuccess; }
int hipEventRecord(void*, void*) { return kSuccess; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0.0f; return kSuccess; }
int hipGetDevice(int* d) { *d = 0; return kSuccess; }
int hipSetDevice(int) { return kSuccess; }
int hipGetDeviceCount(int* n) { *n = 1; return kSuccess; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return kSuccess; }   // asked for the compute units only
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return kSuccess; }
int hipGetSymbolAddress(void** p, const void* symbol) { *p = const_cast<void*>(symbol); return kSuccess; }
int hipGetLastError() { return kSuccess; }
const char* hipGetErrorString(int) { return "a recorded error"; }
int hipLaunchKernel(const void* f, Dim3 grid, Dim3 block, void**, size_t, void*) {
    launches.push_back({kernels.count(f) ? kernels[f] : "?", grid, block});
    return kSuccess;
}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void* stream) {
    configs.push_back({grid, block, shared, stream});
    return kSuccess;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* shared, void** stream) {
    const Config c = configs.back();
    configs.pop_back();
    *grid = c.grid; *block = c.block; *shared = c.shared; *stream = c.stream;
    return kSuccess;
}
void** __hipRegisterFatBinary(const void*) { return reinterpret_cast<void**>(&allocations); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

}  // extern "C"
