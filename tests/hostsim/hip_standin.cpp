// A stand-in for the HIP runtime, for tests of the library's host side where
// there is no GPU: it has the runtime's soname, so a process that loads it
// first gives it to libthesis_stencil.so.  Device memory is host memory,
// kernels do not run.  Every call goes to one hook,
//   int hook(event, handle, size, args)
// whose result is the call's error code (for "capturing": the stream's
// capture status).  A launch's event is its kernel's name, its handle the
// stream, its size the number of workgroups, args the kernel's arguments.
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

extern "C" {
typedef int (*Hook)(const char *event, void *handle, size_t size, void **args);
static Hook g_hook;
void standin_hook(Hook h) { g_hook = h; }
static int call(const char *event, void *handle = nullptr, size_t size = 0, void **args = nullptr)
{
    return g_hook ? g_hook(event, handle, size, args) : 0;
}

struct dim3_ { unsigned x, y, z; };
struct Config { dim3_ grid, block; size_t lds; void *stream; };
static thread_local Config t_config;
static std::mutex g_mutex;
static std::map<const void *, std::string> &names()
{
    static std::map<const void *, std::string> m;
    return m;
}

void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    std::lock_guard<std::mutex> lock(g_mutex);
    names()[host] = name;
}
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t lds, void *s) { t_config = {g, b, lds, s}; return 0; }
int __hipPopCallConfiguration(dim3_ *g, dim3_ *b, size_t *lds, void **s)
{
    *g = t_config.grid; *b = t_config.block; *lds = t_config.lds; *s = t_config.stream;
    return 0;
}
static int launch(const char *kind, const void *fn, dim3_ g, void **args, void *s)
{
    std::string name;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        name = kind + names()[fn];
    }
    return call(name.c_str(), s, (size_t)g.x * g.y * g.z, args);
}
int hipLaunchKernel(const void *fn, dim3_ g, dim3_, void **args, size_t, void *s) { return launch("", fn, g, args, s); }
int hipLaunchCooperativeKernel(const void *fn, dim3_ g, dim3_, void **args, unsigned, void *s)
{
    return launch("coop ", fn, g, args, s);
}

static int memory(const char *event, void **p, size_t n)
{
    const int e = call(event, nullptr, n);
    *p = e ? nullptr : calloc(1, n);
    return e;
}
int hipMalloc(void **p, size_t n) { return memory("malloc", p, n); }
int hipHostMalloc(void **p, size_t n, unsigned) { return memory("malloc host", p, n); }
int hipFree(void *p) { return call("free", p); }  // kept, so that addresses stay distinct
int hipHostFree(void *p) { return call("free host", p); }
int hipGetSymbolAddress(void **p, const void *) { static char scratch[32 << 20]; *p = scratch; return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *st) { memcpy(d, s, n); return call("copy", st, n); }
int hipMemsetAsync(void *, int, size_t n, void *st) { return call("memset", st, n); }

int hipGetDevice(int *d) { *d = 0; return 0; }
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipDeviceGetAttribute(int *v, int, int) { *v = 256; return 0; }  // CUs; every other limit asked for is above it
int hipGetDevicePropertiesR0600(void *, int) { return 1; }
int hipDeviceSynchronize() { return 0; }
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return 0; }
const char *hipGetErrorString(int) { return "stand-in error"; }
int hipGetLastError() { return 0; }

int hipStreamCreate(void **s) { *s = malloc(1); return 0; }
int hipStreamDestroy(void *) { return 0; }
int hipStreamSynchronize(void *s) { return call("sync", s); }
int hipStreamIsCapturing(void *s, int *status) { *status = call("capturing", s); return 0; }
int hipThreadExchangeStreamCaptureMode(int *mode)
{
    static thread_local int current = 0;  // global
    const int old = current;
    current = *mode;
    *mode = old;
    return call("mode", nullptr, (size_t)current);
}
int hipEventCreate(void **e) { *e = malloc(1); return 0; }
int hipEventDestroy(void *) { return 0; }
int hipEventRecord(void *, void *s) { return call("record", s); }
int hipEventSynchronize(void *) { return call("event sync"); }
int hipEventElapsedTime(float *ms, void *, void *) { *ms = 1; return 0; }
int hipStreamBeginCapture(void *, int) { return 1; }
int hipStreamEndCapture(void *, void **) { return 1; }
int hipGraphInstantiate(void **, void *, void **, char *, size_t) { return 1; }
int hipGraphLaunch(void *, void *) { return 1; }
int hipGraphDestroy(void *) { return 0; }
int hipGraphExecDestroy(void *) { return 0; }
}
