// A stand-in for the HIP runtime, for programs without a GPU (LD_PRELOAD): "device" memory is host memory, copies happen at
// once, kernels do not run.  Each launch adds a line to the file that HIP_STUB_LOG names:
//     <kernel> <grid x> <grid y> <grid z> <dynamic LDS bytes>
// and with HIP_STUB_COPIES set each copy on a stream
//     copy <bytes> 1 1 0
// A kernel whose name holds HIP_STUB_FULL is said to fit 8 workgroups to a CU, any other one 4.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Dim3 {
    unsigned x, y, z;
};
struct Config {
    Dim3 grid, block;
    size_t shared;
    void *stream;
};
std::vector<Config> configs;
std::map<const void *, std::string> names;

int allocate(void **p, size_t bytes) { return (*p = calloc(1, bytes ? bytes : 1)) ? 0 : 2; }
}  // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *) {
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) { names[host] = name; }
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void *stream) { return configs.push_back({grid, block, shared, stream}), 0; }
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shared, void **stream) {
    const Config c = configs.back();
    configs.pop_back();
    *grid = c.grid, *block = c.block, *shared = c.shared, *stream = c.stream;
    return 0;
}
int hipLaunchKernel(const void *host, Dim3 grid, Dim3, void **, size_t shared, void *) {
    if (FILE *f = getenv("HIP_STUB_LOG") ? fopen(getenv("HIP_STUB_LOG"), "a") : nullptr) {
        fprintf(f, "%s %u %u %u %zu\n", names[host].c_str(), grid.x, grid.y, grid.z, shared);
        fclose(f);
    }
    return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *host, int, size_t) {
    const char *full = getenv("HIP_STUB_FULL");
    *n = full && names[host].find(full) != std::string::npos ? 8 : 4;
    return 0;
}
int hipMalloc(void **p, size_t bytes) { return allocate(p, bytes); }
int hipFree(void *p) { return free(p), 0; }
int hipHostMalloc(void **p, size_t bytes, unsigned) { return allocate(p, bytes); }
int hipHostFree(void *p) { return free(p), 0; }
int hipMemcpy(void *dst, const void *src, size_t bytes, int) { return memmove(dst, src, bytes), 0; }
int hipMemcpyAsync(void *dst, const void *src, size_t bytes, int, void *) {
    if (getenv("HIP_STUB_COPIES"))
        if (FILE *f = getenv("HIP_STUB_LOG") ? fopen(getenv("HIP_STUB_LOG"), "a") : nullptr) {
            fprintf(f, "copy %zu 1 1 0\n", bytes);
            fclose(f);
        }
    return memmove(dst, src, bytes), 0;
}
int hipMemset(void *p, int value, size_t bytes) { return memset(p, value, bytes), 0; }
int hipMemsetAsync(void *p, int value, size_t bytes, void *) { return memset(p, value, bytes), 0; }
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipGetDevice(int *d) { return *d = 0; }
int hipSetDevice(int) { return 0; }
int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipGetDevicePropertiesR0600(void *prop, int) {
    strcpy((char *)prop, "stand-in");
    strcpy((char *)prop + 1160, "gfx950");  // gcnArchName of hipDeviceProp_tR0600, whose layout the versioned name fixes
    return 0;
}
const char *hipGetErrorString(int) { return "error of the stand-in"; }
int hipGetLastError() { return 0; }
int hipGetSymbolAddress(void **p, const void *) {
    static void *scratch = nullptr;
    if (!scratch) allocate(&scratch, 32u << 20);
    *p = scratch;
    return 0;
}
int hipStreamSynchronize(void *) { return 0; }
}
