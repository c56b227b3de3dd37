// HIP runtime entry points of librxmesh_amd.so for tests without a GPU, put in
// front of the real ones with LD_PRELOAD: device memory is host memory (zeroed),
// kernels are not run, and what the library asks of the runtime -- launches by
// name and stream, waits, allocations -- is recorded. So the order of the
// library's host calls can be checked, and a failed allocation or a capturing
// stream be had on demand. Results of kernels are all zeros here.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct dim3
{
    uint32_t x, y, z;
};
enum { kOk = 0, kInvalid = 1, kNoMemory = 2, kCaptureUnsupported = 900, kUnknown = 999 };
struct Rec
{
    std::map<const void*, std::string> names;  // host handle -> kernel
    std::map<void*, size_t>            live;
    std::vector<std::string>           log;
    int  fail_in = 0, wait_fail_in = 0;  // > 0: that allocation / wait from now fails
    bool capturing = false;
    int  last_error = kOk;  // sticky until hipGetLastError reads it
    dim3 grid{}, block{};
    size_t lds = 0;
    void*  stream = nullptr;
} r;
std::string at(void* stream) { return " @" + std::to_string(reinterpret_cast<uintptr_t>(stream)); }
int fail(int e)
{
    r.last_error = e;
    return e;
}
}  // namespace

extern "C" {
void   rec_fail_malloc(int n) { r.fail_in = n; }
void   rec_fail_wait(int n) { r.wait_fail_in = n; }
void   rec_capturing(int on) { r.capturing = on != 0; }
size_t rec_live_count() { return r.live.size(); }
size_t rec_live_bytes()
{
    size_t n = 0;
    for (auto& q : r.live) n += q.second;
    return n;
}
// the log since the last call, one entry a line
const char* rec_log()
{
    static std::string s;
    s.clear();
    for (auto& l : r.log) s += l + "\n";
    r.log.clear();
    return s.c_str();
}

void** __hipRegisterFatBinary(const void*)
{
    static void* h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    r.names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
int  __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void* s)
{
    r.grid = g, r.block = b, r.lds = lds, r.stream = s;
    return kOk;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, void** s)
{
    *g = r.grid, *b = r.block, *lds = r.lds, *s = r.stream;
    return kOk;
}
int hipLaunchKernel(const void* host, dim3, dim3, void**, size_t, void* s)
{
    r.log.push_back("launch " + r.names[host] + at(s));
    return kOk;
}
int hipFuncSetAttribute(const void*, int, int) { return kOk; }
int hipGetLastError()
{
    const int e  = r.last_error;
    r.last_error = kOk;
    return e;
}
int hipGetDevice(int* d)
{
    *d = 0;
    return kOk;
}
int hipDeviceGetAttribute(int* v, int, int)
{
    *v = 256;
    return kOk;
}
int hipMalloc(void** p, size_t n)
{
    if (r.capturing) return r.log.push_back("illegal malloc"), fail(kCaptureUnsupported);
    if (r.fail_in > 0 && --r.fail_in == 0) return fail(kNoMemory);
    *p         = std::calloc(n ? n : 1, 1);
    r.live[*p] = n;
    return kOk;
}
int hipFree(void* p)
{
    if (!p) return kOk;
    if (!r.live.erase(p)) return fail(kInvalid);
    std::free(p);
    return kOk;
}
int hipMemcpy(void* d, const void* s, size_t n, int)
{
    if (r.capturing) return r.log.push_back("illegal copy"), fail(kCaptureUnsupported);
    std::memcpy(d, s, n);
    return kOk;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void* stream)
{
    if (r.capturing) return r.log.push_back("illegal copy"), fail(kCaptureUnsupported);
    std::memcpy(d, s, n);
    r.log.push_back("copy" + at(stream));
    return kOk;
}
int hipStreamSynchronize(void* s)
{
    if (r.capturing) return r.log.push_back("illegal wait"), fail(kCaptureUnsupported);
    if (r.wait_fail_in > 0 && --r.wait_fail_in == 0) return fail(kUnknown);
    r.log.push_back("wait" + at(s));
    return kOk;
}
int hipStreamIsCapturing(void*, int* status)
{
    *status = r.capturing ? 1 : 0;
    return kOk;
}
}
