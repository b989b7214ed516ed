// A HIP runtime of host memory, for tests of the library's host code where
// there is no GPU: device memory is counted and limited host memory, copies are
// memcpy, and a launch is only noted by name: no kernel runs, except that
// those which report to the host leave their launch's number, so that nothing
// waits for it.  Loaded with RTLD_GLOBAL before the library, its functions take
// the runtime's place.
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<void *, size_t> g_blocks;
std::map<const void *, std::string> g_names;
std::string g_log;
size_t g_live = 0, g_limit = (size_t)1 << 40;
void (*g_hook)(const char *, void **) = nullptr;
struct Dim {
    unsigned x, y, z;
};
struct Call {
    Dim grid, block;
    size_t lds;
    void *stream;
} g_call;
constexpr int kNoMemory = 2;
int g_last = 0;  // the last error, until it is asked for
}  // namespace

extern "C" {
// ---- for the tests
size_t hostrt_live() { return g_live; }
void hostrt_limit(size_t bytes) { g_limit = bytes; }
// called with the name and the arguments' addresses of every launch
void hostrt_hook(void (*f)(const char *, void **)) { g_hook = f; }
// the kernels launched since the last call, one a line: mangled name and grid
const char *hostrt_launches()
{
    static std::string out;
    out.swap(g_log);
    g_log.clear();
    return out.c_str();
}

// ---- memory
int hipMalloc(void **p, size_t n)
{
    *p = nullptr;
    if (g_live + n > g_limit) return g_last = kNoMemory;
    if (posix_memalign(p, 4096, n ? n : 1)) return kNoMemory;
    memset(*p, 0, n);
    g_blocks[*p] = n;
    g_live += n;
    return 0;
}
int hipFree(void *p)
{
    const auto it = g_blocks.find(p);
    if (it == g_blocks.end()) return p ? 1 : 0;
    g_live -= it->second;
    g_blocks.erase(it);
    free(p);
    return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned) { return (*p = calloc(n ? n : 1, 1)) ? 0 : kNoMemory; }
int hipHostFree(void *p)
{
    free(p);
    return 0;
}
int hipMemGetInfo(size_t *room, size_t *total)
{
    *room = g_limit > g_live ? g_limit - g_live : 0;
    *total = g_limit;
    return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int)
{
    memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *) { return hipMemcpy(d, s, n, kind); }
int hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int kind)
{
    for (size_t i = 0; i < h; i++) hipMemcpy((char *)d + i * dp, (const char *)s + i * sp, w, kind);
    return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, void *)
{
    memset(d, v, n);
    return 0;
}
int hipGetSymbolAddress(void **p, const void *)
{
    static void *mem = calloc(1, (size_t)1 << 20);
    *p = mem;
    return 0;
}

// ---- device, stream, events, errors
int hipGetDeviceCount(int *n)
{
    *n = 1;
    return 0;
}
int hipGetDevice(int *d)
{
    *d = 0;
    return 0;
}
int hipGetDevicePropertiesR0600(void *, int) { return 0; }
int hipStreamCreateWithFlags(void **s, unsigned)
{
    *s = malloc(1);
    return 0;
}
int hipStreamSynchronize(void *) { return 0; }
int hipEventCreate(void **e)
{
    *e = malloc(1);
    return 0;
}
int hipEventRecord(void *, void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *)
{
    *ms = 0.0f;
    return 0;
}
int hipGetLastError()
{
    const int e = g_last;
    g_last = 0;
    return e;
}
const char *hipGetErrorString(int e) { return e == kNoMemory ? "out of memory" : "error"; }

// ---- launches
void **__hipRegisterFatBinary(const void *)
{
    static void *handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *)
{
    g_names[f] = name;
}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t lds, void *stream)
{
    g_call = {grid, block, lds, stream};
    return 0;
}
int __hipPopCallConfiguration(Dim *grid, Dim *block, size_t *lds, void **stream)
{
    *grid = g_call.grid;
    *block = g_call.block;
    *lds = g_call.lds;
    *stream = g_call.stream;
    return 0;
}
int hipLaunchKernel(const void *f, Dim grid, Dim, void **args, size_t, void *)
{
    const std::string &name = g_names[f];
    g_log += name + " " + std::to_string(grid.x) + " " + std::to_string(grid.y) + "\n";
    if (g_hook) g_hook(name.c_str(), args);
    // arguments (..., numbers, number) of the two kernels that report
    const int at = name.find("k_reduce_rows_host") != std::string::npos ? 3
                   : name.find("k_sum_chunks") != std::string::npos     ? 6
                                                                        : -1;
    if (at >= 0)
        for (unsigned i = 0; i < grid.x; i++)
            (*(unsigned long long **)args[at])[i] = *(unsigned long long *)args[at + 1];
    return 0;
}
}
