// A HIP runtime without a GPU for tests of the library's host code: device memory is host memory, copies
// copy, streams and events are nothing, graphs are not supported, and a kernel launch is noted by the
// kernel's name and does nothing.  What the host code makes of results that never arrive can be seen this
// way, and what it launches.
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#define API extern "C" __attribute__((visibility("default")))
typedef int Err;   // hipError_t
enum { kOk = 0, kNoLds = 1, kUnsupported = 801 };

namespace {
struct Dim {
    unsigned x, y, z;
};
std::map<const void *, std::string> &names() {
    static std::map<const void *, std::string> m;
    return m;
}
std::string &launched() {
    static std::string s;
    return s;
}
int refuse_lds = 0;
Dim cfg_grid, cfg_block;
size_t cfg_lds;
void *cfg_stream;
}  // namespace

// the test's side
API const char *fake_launched() { return launched().c_str(); }
API void fake_clear() { launched().clear(); }
API void fake_refuse_lds(int on) { refuse_lds = on; }

// what compiled host code calls
API void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
API void __hipUnregisterFatBinary(void **) {}
API void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                               int *) {
    names()[host] = name;
}
API void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
API Err __hipPushCallConfiguration(Dim grid, Dim block, size_t lds, void *stream) {
    cfg_grid = grid;
    cfg_block = block;
    cfg_lds = lds;
    cfg_stream = stream;
    return kOk;
}
API Err __hipPopCallConfiguration(Dim *grid, Dim *block, size_t *lds, void **stream) {
    *grid = cfg_grid;
    *block = cfg_block;
    *lds = cfg_lds;
    *stream = cfg_stream;
    return kOk;
}
API Err hipLaunchKernel(const void *f, Dim grid, Dim block, void **args, size_t, void *) {
    const std::string &name = names()[f];
    launched() += name + " " + std::to_string(grid.x) + " " + std::to_string(block.x * block.y * block.z);
    if (name.find("ColGeo") != std::string::npos)   // a march of columns.h: its first argument
        for (int q = 0; q < 5; q++) launched() += " " + std::to_string(((const int *)args[0])[q]);
    launched() += "\n";
    return kOk;
}
API Err hipFuncSetAttribute(const void *, int, int) { return refuse_lds ? kNoLds : kOk; }
API Err hipGetLastError() { return kOk; }
API const char *hipGetErrorString(Err) { return "fake"; }
API Err hipGetDevice(int *d) {
    *d = 0;
    return kOk;
}
API Err hipDeviceGetAttribute(int *v, int, int) {
    *v = 160 * 1024;   // asked for the LDS of a workgroup only
    return kOk;
}
API Err hipMalloc(void **p, size_t n) {
    *p = calloc(1, n);
    return kOk;
}
API Err hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
API Err hipFree(void *p) {
    free(p);
    return kOk;
}
API Err hipHostFree(void *p) { return hipFree(p); }
API Err hipMemcpy(void *d, const void *s, size_t n, int) {
    memcpy(d, s, n);
    return kOk;
}
API Err hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *) { return hipMemcpy(d, s, n, k); }
API Err hipMemsetAsync(void *d, int v, size_t n, void *) {
    memset(d, v, n);
    return kOk;
}
API Err hipGetSymbolAddress(void **p, const void *) {
    static char buf[1 << 20];
    *p = buf;
    return kOk;
}
API Err hipStreamCreateWithFlags(void **s, unsigned) {
    *s = nullptr;
    return kOk;
}
API Err hipStreamDestroy(void *) { return kOk; }
API Err hipStreamSynchronize(void *) { return kOk; }
API Err hipStreamIsCapturing(void *, int *c) {
    *c = 0;
    return kOk;
}
API Err hipStreamBeginCapture(void *, int) { return kUnsupported; }
API Err hipStreamEndCapture(void *, void **) { return kUnsupported; }
API Err hipGraphInstantiate(void **, void *, void **, char *, size_t) { return kUnsupported; }
API Err hipGraphLaunch(void *, void *) { return kUnsupported; }
API Err hipGraphDestroy(void *) { return kOk; }
API Err hipGraphExecDestroy(void *) { return kOk; }
API Err hipEventCreate(void **e) {
    *e = nullptr;
    return kOk;
}
API Err hipEventCreateWithFlags(void **e, unsigned) { return hipEventCreate(e); }
API Err hipEventDestroy(void *) { return kOk; }
API Err hipEventRecord(void *, void *) { return kOk; }
API Err hipEventRecordWithFlags(void *, void *, unsigned) { return kOk; }
API Err hipEventSynchronize(void *) { return kOk; }
API Err hipEventElapsedTime(float *ms, void *, void *) {
    *ms = 0.0f;
    return kOk;
}
