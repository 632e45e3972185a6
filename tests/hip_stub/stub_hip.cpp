// Stand-in for the HIP runtime calls that libvsfeel_bm3d.so makes: memory is
// host memory, kernels are not run but logged, streams and events are tokens.
// Loaded before the library (RTLD_GLOBAL), it shows what the host code
// allocates, launches and captures on a machine without a GPU.

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

struct Dim3 {
    uint32_t x, y, z;
};
struct Exec {
    std::string log;  // the captured sequence
};

std::map<const void *, std::string> kernels;  // host stub -> name
std::map<void *, size_t> blocks;
size_t live = 0, limit = SIZE_MAX;
std::string events;        // what has been logged since stub_take_log
std::string captured;
bool capturing = false;
Dim3 grid, block;
size_t shmem;
void *stream;
char token[1];

void log(const std::string &s) { (capturing ? captured : events) += s + "\n"; }
void *handle() { return std::malloc(1); }

}  // namespace

extern "C" {

// ------------------------------------------------- the tests' side
void stub_limit(size_t bytes) { limit = bytes; }
size_t stub_live() { return live; }
// the log so far, which starts anew
const char *stub_take_log()
{
    static std::string out;
    out.swap(events);
    events.clear();
    return out.c_str();
}

// ------------------------------------------------- the library's side
void **__hipRegisterFatBinary(const void *)
{
    static void *bin = token;
    return &bin;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *)
{
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t s, void *q)
{
    grid = g;
    block = b;
    shmem = s;
    stream = q;
    return 0;
}
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *s, void **q)
{
    *g = grid;
    *b = block;
    *s = shmem;
    *q = stream;
    return 0;
}
int hipLaunchKernel(const void *f, Dim3, Dim3, void **, size_t, void *)
{
    log("kernel " + kernels[f]);
    return 0;
}

int hipMalloc(void **p, size_t n)
{
    *p = nullptr;
    if (n > limit || live > limit - n) {
        return 2;  // hipErrorOutOfMemory
    }
    *p = std::malloc(n ? n : 1);
    blocks[*p] = n;
    live += n;
    return 0;
}
int hipFree(void *p)
{
    const auto it = blocks.find(p);
    if (it != blocks.end()) {
        live -= it->second;
        blocks.erase(it);
        std::free(p);
    }
    return 0;
}
int hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = std::malloc(n ? n : 1);
    return 0;
}
int hipHostFree(void *p)
{
    std::free(p);
    return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int)
{
    std::memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *)
{
    std::memcpy(d, s, n);
    return 0;
}

int hipGetDeviceCount(int *n)
{
    *n = 1;
    return 0;
}
int hipSetDevice(int) { return 0; }
int hipGetLastError() { return 0; }
const char *hipGetErrorString(int) { return "stub error"; }
int hipGetSymbolAddress(void **p, const void *s)
{
    *p = const_cast<void *>(s);
    return 0;
}

int hipStreamCreateWithFlags(void **s, unsigned)
{
    *s = handle();
    return 0;
}
int hipStreamDestroy(void *s)
{
    std::free(s);
    return 0;
}
int hipStreamSynchronize(void *) { return 0; }
int hipStreamWaitEvent(void *, void *, unsigned) { return 0; }
int hipEventCreate(void **e)
{
    *e = handle();
    return 0;
}
int hipEventCreateWithFlags(void **e, unsigned)
{
    *e = handle();
    return 0;
}
int hipEventDestroy(void *e)
{
    std::free(e);
    return 0;
}
int hipEventRecord(void *, void *) { return 0; }
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *)
{
    *ms = 0.0f;
    return 0;
}

int hipStreamBeginCapture(void *, int)
{
    log("capture");
    captured.clear();
    capturing = true;
    return 0;
}
int hipStreamEndCapture(void *, void **g)
{
    capturing = false;
    *g = new Exec{captured};
    return 0;
}
int hipGraphInstantiate(void **x, void *g, void *, char *, size_t)
{
    *x = new Exec(*static_cast<Exec *>(g));
    return 0;
}
int hipGraphExecUpdate(void *x, void *g, void *, int *result)
{
    *static_cast<Exec *>(x) = *static_cast<Exec *>(g);
    *result = 0;
    return 0;
}
int hipGraphLaunch(void *x, void *)
{
    log("replay");
    events += static_cast<Exec *>(x)->log;
    return 0;
}
int hipGraphDestroy(void *g)
{
    delete static_cast<Exec *>(g);
    return 0;
}
int hipGraphExecDestroy(void *x)
{
    delete static_cast<Exec *>(x);
    return 0;
}

}  // extern "C"
