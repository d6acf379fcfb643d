// A HIP runtime for tests of the library's host code on machines without a GPU:
// preloaded into a child process, it takes the place of the runtime's functions
// that libswept1d calls.  Device memory is host memory, copies are done when they
// are called, streams and events are nothing.  Kernels do nothing, but for the
// network step, which adds 1 to every value of its input, so that a test can
// follow a state; a device check finds the word it set unchanged, which passes.
//
// A test makes calls fail through the functions at the end.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <string>
#include <sys/syscall.h>
#include <unistd.h>

namespace {
struct Dim { uint32_t x, y, z; };
std::map<const void*, std::string> names;
std::map<const char*, size_t> sizes;
std::set<std::string> launched;
thread_local struct { Dim grid, block; size_t shared; void* stream; } config;
char dummy[64];
const void *copy_src, *copy_dst;  // of the last asynchronous copy
long uploads;    // copies from the host to the device
long unordered;  // work on the null stream that its call does not wait for
long populated;  // bytes that madvise was asked to make present
long launches, launch_limit = -1, mallocs, malloc_limit = -1, copies, copy_limit = -1;
thread_local long last_error;
size_t new_limit = ~(size_t)0, watch;
void *watched[8], *freed[8];  // live and freed blocks of `watch` bytes (freed ones are kept)
std::recursive_mutex guard;  // of all the above
typedef std::lock_guard<std::recursive_mutex> Lock;
int fail(long& count, long limit)
{
    Lock lock(guard);
    ++count;
    if (limit < 0 || count <= limit) return 0;
    last_error = 2;
    return 2;  // hipErrorOutOfMemory
}
size_t size_of(const void* p)
{
    Lock lock(guard);
    auto it = sizes.find((const char*)p);
    return it == sizes.end() ? 0 : it->second;
}
}  // namespace

void* operator new(size_t n)
{
    if (n > new_limit) throw std::bad_alloc();
    void* p = malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    if (watch && n == watch)
        for (void*& w : watched)
            if (!w) {
                w = p;
                break;
            }
    return p;
}
void operator delete(void* p) noexcept
{
    if (watch && p)
        for (int i = 0; i < 8; ++i)
            if (watched[i] == p && !freed[i]) {
                freed[i] = memset(p, 0x5a, watch);
                return;
            }
    free(p);
}
void operator delete(void* p, size_t) noexcept { operator delete(p); }

extern "C" {

void** __hipRegisterFatBinary(const void*) { return (void**)dummy; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t shared, void* stream)
{
    config = {grid, block, shared, stream};
    return 0;
}
int __hipPopCallConfiguration(Dim* grid, Dim* block, size_t* shared, void** stream)
{
    *grid = config.grid;
    *block = config.block;
    *shared = config.shared;
    *stream = config.stream;
    return 0;
}
int hipLaunchKernel(const void* f, Dim, Dim, void** args, size_t, void*)
{
    Lock lock(guard);
    const std::string& name = names[f];
    launched.insert(name);
    const bool network = name.find("k_net_fwdId") != std::string::npos;
    if (network && fail(launches, launch_limit)) return 2;
    if (network) {  // (in, 1/in_scale, parameters, weights, du, out, ..)
        const double* in = *(const double**)args[0];
        double* out = *(double**)args[5];
        const size_t bytes = std::min(size_of(in), size_of(out));
        if (!in || !out || !bytes) abort();
        for (size_t i = 0; i < bytes / sizeof(double); ++i) out[i] = in[i] + 1;
    }
    return 0;
}
int hipMalloc(void** p, size_t n)
{
    *p = nullptr;
    if (fail(mallocs, malloc_limit)) return 2;
    if (!(*p = calloc(n ? n : 1, 1))) return 2;
    Lock lock(guard);
    sizes[(const char*)*p] = n;
    return 0;
}
int hipFree(void* p)
{
    Lock lock(guard);
    sizes.erase((const char*)p);
    free(p);
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned)
{
    if (!(*p = calloc(n, 1))) return 2;
    Lock lock(guard);
    sizes[(const char*)*p] = n;
    return 0;
}
int hipHostFree(void* p) { return hipFree(p); }
int hipPointerGetAttributes(int* type, const void* p)  // the first member is the type of memory
{
    Lock lock(guard);
    auto it = sizes.upper_bound((const char*)p);
    *type = it != sizes.begin() && (--it, (const char*)p < it->first + it->second);
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int kind)
{
    uploads += kind == 1;
    unordered += kind == 1 || kind == 3;
    memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*)
{
    uploads += kind == 1;
    if (fail(copies, copy_limit)) return 2;
    copy_src = s;
    copy_dst = d;
    memcpy(d, s, n);
    return 0;
}
int hipMemset(void* p, int v, size_t n)
{
    ++unordered;
    memset(p, v, n);
    return 0;
}
int hipMemsetAsync(void* p, int v, size_t n, void*)
{
    memset(p, v, n);
    return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned)
{
    *s = dummy;
    return 0;
}
int hipStreamDestroy(void*) { return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipStreamIsCapturing(void*, int* status)
{
    *status = 0;
    return 0;
}
int hipEventCreate(void** e)
{
    *e = dummy;
    return 0;
}
int hipEventCreateWithFlags(void** e, unsigned)
{
    *e = dummy;
    return 0;
}
int hipEventDestroy(void*) { return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*)
{
    *ms = 1;
    return 0;
}
int hipGetDevice(int* d)
{
    *d = 0;
    return 0;
}
int hipDeviceGetAttribute(int* v, int, int)
{
    *v = 256;
    return 0;
}
int hipGetLastError()
{
    const long e = last_error;
    last_error = 0;
    return (int)e;
}
const char* hipGetErrorString(int) { return "stub"; }

// From now on: the network step, device allocation or asynchronous copy after
// `more` further ones fails (negative: none does); operator new fails above `most`
// bytes.
void stub_fail_launch(long more) { launches = 0, launch_limit = more; }
void stub_fail_malloc(long more) { mallocs = 0, malloc_limit = more; }
void stub_fail_copy(long more) { copies = 0, copy_limit = more; }
void stub_fail_new(size_t most) { new_limit = most; }
int madvise(void* p, size_t n, int advice)
{
    if (advice == 23) populated += n;  // MADV_POPULATE_WRITE
    return (int)syscall(SYS_madvise, p, n, advice);
}
long stub_uploads() { return uploads; }
long stub_unordered() { return unordered; }
long stub_mallocs() { return mallocs; }  // since the last stub_fail_malloc
long stub_populated() { return populated; }
// The names of the library's kernels, and of those launched since the last call, a
// line each.
const char* stub_kernels()
{
    static std::string lines;
    lines.clear();
    for (const auto& k : names) lines += k.second + "\n";
    return lines.c_str();
}
const char* stub_launched()
{
    static std::string lines;
    lines.clear();
    for (const std::string& k : launched) lines += k + "\n";
    launched.clear();
    return lines.c_str();
}
const void* stub_copy_src() { return copy_src; }
const void* stub_copy_dst() { return copy_dst; }
// Blocks of `size` bytes from operator new are kept when they are deleted; the
// number of those that were, and how many of them have been written to since.
void stub_watch_new(size_t size) { watch = size; }
int stub_freed() { return (int)(std::end(freed) - std::count(freed, std::end(freed), nullptr) - freed); }
int stub_freed_written()
{
    int n = 0;
    for (void* p : freed)
        for (size_t i = 0; p && i < watch; ++i)
            if (((unsigned char*)p)[i] != 0x5a) {
                ++n;
                break;
            }
    return n;
}
}
