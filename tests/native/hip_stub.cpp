// The HIP runtime calls of libgalx.so on the host, for tests of its host code without a GPU: device memory is host memory
// (each allocation filled with the indices of its doubles), kernels do nothing, and a copy runs no sooner than a call that
// waits for it.  stub_fail makes one call fail, stub_busy lets the queued work take a while.
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <string>
#include <unistd.h>

namespace {
struct Dim3 { unsigned x, y, z; };
struct Copy { void* dst; const void* src; size_t n; };
std::deque<Copy> queued;             // copies nobody has waited for
long issued = 0, finished = 0;       // copies so far: all, and those that ran
std::map<void*, long> recorded;      // event: the copies issued before it
std::map<std::string, long> calls;   // calls so far of each entry point
std::map<std::string, long> fail_at; // the call that fails
int last_error = 0;
unsigned busy_us = 0;
struct { Dim3 g, b; size_t s; void* st; } config;

int called(const char* name)
{
    auto f = fail_at.find(name);
    const bool bad = f != fail_at.end() && ++calls[name] == f->second;
    if (f == fail_at.end()) ++calls[name];
    if (bad) last_error = 2;
    return bad ? 2 : 0;
}

void run_until(long upto)
{
    if (busy_us) usleep(busy_us);
    busy_us = 0;
    for (; finished < upto; finished++) {
        std::memcpy(queued.front().dst, queued.front().src, queued.front().n);
        queued.pop_front();
    }
}
}  // namespace

extern "C" {
// the test's side
void stub_fail(const char* name, long nth) { fail_at[name] = nth ? calls[name] + nth : 0; }
void stub_busy(unsigned us) { busy_us = us; }
long stub_calls(const char* name) { return calls[name]; }
long stub_pending(void) { return issued - finished; }

// the library's side
int hipGetDeviceCount(int* n) { *n = 1; return called("hipGetDeviceCount"); }
int hipSetDevice(int) { return called("hipSetDevice"); }
int hipDeviceSynchronize(void) { run_until(issued); return called("hipDeviceSynchronize"); }
int hipGetLastError(void) { int e = last_error; last_error = 0; return e; }
const char* hipGetErrorString(int e) { return e ? "stub error" : "no error"; }
int hipMalloc(void** p, size_t n)
{
    if (int e = called("hipMalloc")) return e;
    double* d = static_cast<double*>(std::malloc(n + sizeof(double)));
    for (size_t i = 0; i < n / sizeof(double); i++) d[i] = double(i);
    *p = d;
    return 0;
}
int hipFree(void* p) { std::free(p); return called("hipFree"); }
int hipHostMalloc(void** p, size_t n, unsigned)
{
    if (int e = called("hipHostMalloc")) return e;
    *p = std::calloc(n, 1);
    return 0;
}
int hipHostFree(void* p) { run_until(issued); std::free(p); return called("hipHostFree"); }
int hipMemcpyAsync(void* dst, const void* src, size_t n, int, void*)
{
    if (int e = called("hipMemcpyAsync")) return e;
    queued.push_back({dst, src, n});
    issued++;
    return 0;
}
int hipMemcpy(void* dst, const void* src, size_t n, int)
{
    run_until(issued);
    std::memcpy(dst, src, n);
    return called("hipMemcpy");
}
int hipMemset(void* p, int v, size_t n) { std::memset(p, v, n); return called("hipMemset"); }
int hipMemsetAsync(void* p, int v, size_t n, void*) { std::memset(p, v, n); return called("hipMemsetAsync"); }
int hipStreamCreateWithFlags(void** s, unsigned) { *s = std::malloc(1); return called("hipStreamCreateWithFlags"); }
int hipStreamDestroy(void* s) { std::free(s); return called("hipStreamDestroy"); }
int hipStreamSynchronize(void*) { run_until(issued); return called("hipStreamSynchronize"); }
int hipEventCreateWithFlags(void** e, unsigned) { *e = std::malloc(1); return called("hipEventCreateWithFlags"); }
int hipEventCreate(void** e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void* e) { std::free(e); return called("hipEventDestroy"); }
int hipEventRecord(void* e, void*) { recorded[e] = issued; return called("hipEventRecord"); }
int hipEventSynchronize(void* e)
{
    if (int r = called("hipEventSynchronize")) return r;
    run_until(recorded[e]);
    return 0;
}
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 0.f; return called("hipEventElapsedTime"); }
int hipPointerGetAttributes(void*, const void*) { called("hipPointerGetAttributes"); return 1; }
int hipGetSymbolAddress(void**, const void*) { return 1; }
int hipLaunchKernel(const void*, Dim3, Dim3, void**, size_t, void*) { return called("hipLaunchKernel"); }
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t s, void* st) { config = {g, b, s, st}; return 0; }
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* s, void** st)
{
    *g = config.g;
    *b = config.b;
    *s = config.s;
    *st = config.st;
    return 0;
}
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}
