// A host stand-in for the part of the HIP runtime that libnmi.so calls, for tests of its host code
// without a GPU: loaded with global symbol scope before the library.  Kernel launches are noted and do
// nothing; device memory is address space that nobody touches.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

struct dim3 {
    uint32_t x, y, z;
};
struct Config {
    dim3 grid, block;
    size_t shmem;
    void* stream;
};
constexpr int kSuccess = 0, kOutOfMemory = 2, kCaptureUnsupported = 900;

std::map<const void*, std::string>& names() {
    static std::map<const void*, std::string> m;
    return m;
}
std::string g_log;
Config g_config{};
int g_last = kSuccess;
uintptr_t g_next = uintptr_t{1} << 40;
size_t g_limit = SIZE_MAX;
int g_mallocs = 0, g_capturing = 0;

}  // namespace

extern "C" {

// --- the tests' side
const char* stub_take_log() {                  // launches since the last call: "name x y z block\n"
    static std::string out;
    out.swap(g_log);
    g_log.clear();
    return out.c_str();
}
void stub_malloc_limit(size_t bytes) { g_limit = bytes; }   // hipMalloc of more fails
int stub_mallocs() { return g_mallocs; }
void stub_capturing(int on) { g_capturing = on; }           // every stream; hipMalloc then fails

// --- the runtime's side
void** __hipRegisterFatBinary(const void*) {
    static void* handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, void* stream) {
    g_config = Config{grid, block, shmem, stream};
    return kSuccess;
}
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, void** stream) {
    *grid = g_config.grid;
    *block = g_config.block;
    *shmem = g_config.shmem;
    *stream = g_config.stream;
    return kSuccess;
}
int hipLaunchKernel(const void* host, dim3 grid, dim3 block, void**, size_t, void*) {
    char dims[96];
    std::snprintf(dims, sizeof(dims), " %u %u %u %u\n", grid.x, grid.y, grid.z, block.x);
    g_log += names()[host] + dims;
    return kSuccess;
}
int hipMalloc(void** p, size_t bytes) {
    *p = nullptr;
    if (g_capturing) return g_last = kCaptureUnsupported;
    if (bytes > g_limit) return g_last = kOutOfMemory;
    ++g_mallocs;
    *p = reinterpret_cast<void*>(g_next);
    g_next += (bytes + 0xffff) & ~size_t{0xffff};
    return kSuccess;
}
int hipFree(void*) { return kSuccess; }
int hipHostMalloc(void** p, size_t bytes, unsigned) {
    *p = std::malloc(bytes);
    return kSuccess;
}
int hipGetLastError() {                        // reports once, as the runtime does
    const int e = g_last;
    g_last = kSuccess;
    return e;
}
const char* hipGetErrorString(int) { return "error"; }
int hipGetDevice(int* dev) {
    *dev = 0;
    return kSuccess;
}
int hipDeviceGetAttribute(int* value, int, int) {
    *value = 256;                              // the only attribute asked for: compute units
    return kSuccess;
}
int hipStreamIsCapturing(void*, int* status) {
    *status = g_capturing;                     // 0: none, 1: active
    return kSuccess;
}
int hipDeviceSynchronize() { return kSuccess; }
int hipFuncSetAttribute(const void*, int, int) { return kSuccess; }
int hipGetSymbolAddress(void** p, const void*) {
    *p = reinterpret_cast<void*>(uintptr_t{1} << 39);
    return kSuccess;
}
int hipMemcpy(void*, const void*, size_t, int) { return kSuccess; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 1;
    return kSuccess;
}

}  // extern "C"
