// A HIP runtime that computes nothing, for tests of the library's host logic without a GPU: loaded with
// its symbols global before libvmx.so, it serves the HIP calls that the library makes.  Device memory is
// address space of the process (mapped when touched) up to a capacity, copies stay within one allocation and
// those to and from the host are made at once, kernels do nothing, and every call that a test may ask about is written to a log.  A test
// sets the capacity and makes a launch or a copy fail.
#include <stddef.h>
#include <stdint.h>
#include <string.h>
#include <sys/mman.h>

#include <map>
#include <mutex>
#include <string>

namespace {
enum { kSuccess = 0, kOutOfMemory = 2, kInvalidValue = 1, kUnknown = 999 };
struct Dim3 { uint32_t x, y, z; };
struct Call { Dim3 grid, block; size_t shared; void* stream; };
std::recursive_mutex mu;
std::map<const void*, std::string> kernels;       // host stub -> mangled device name
std::map<void*, size_t> blocks;
size_t capacity = (size_t)288 << 30, used = 0, peak = 0;
std::string text, fail_kernel;
int fail_launch_in = 0, fail_copy_in = 0, last = kSuccess, serial = 0;
std::map<std::string, int> watched;               // kernel name -> argument whose first word is logged
Call pushed;
bool logging = false;
using Lock = std::lock_guard<std::recursive_mutex>;
void note(const std::string& s) { if (logging) { text += s; text += '\n'; } }
std::string num(size_t v) { return std::to_string(v); }
int done(int e) { if (e != kSuccess) last = e; return e; }
int take(void** p, size_t n) {
    Lock l(mu);
    note("malloc " + num(n));
    if (used + n > capacity) return done(kOutOfMemory);
    void* m = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return done(kOutOfMemory);
    blocks[m] = n ? n : 1;
    used += n;
    if (used > peak) peak = used;
    *p = m;
    return kSuccess;
}
int give(void* p) {
    Lock l(mu);
    auto it = blocks.find(p);
    if (it == blocks.end()) return done(kInvalidValue);
    note("free " + num(it->second));
    munmap(p, it->second);
    used -= it->second;
    blocks.erase(it);
    return kSuccess;
}
bool within_one_block(const void* p, size_t n) {
    auto it = blocks.upper_bound(const_cast<void*>(p));
    if (it == blocks.begin()) return false;
    --it;
    return (const char*)p + n <= (const char*)it->first + it->second;
}
int copy(void* d, const void* s, size_t n, int kind) {
    Lock l(mu);
    note("copy " + num(kind) + " " + num(n));
    if ((kind != 2 && !within_one_block(d, n)) || (kind != 1 && !within_one_block(s, n))) return done(kInvalidValue);
    if (fail_copy_in > 0 && --fail_copy_in == 0) return done(kUnknown);
    if (kind != 3) memcpy(d, s, n);               // 1: to the device, 2: to the host; 3: within it, not made
    return kSuccess;
}
int handle(void** h) { Lock l(mu); *h = (void*)(intptr_t)++serial; return kSuccess; }
}  // namespace

extern "C" {
// ---- the test's side
void fake_log(int on) { Lock l(mu); logging = on != 0; text.clear(); }
const char* fake_text() { return text.c_str(); }
void fake_capacity(size_t bytes) { capacity = bytes; }
size_t fake_used() { return used; }
size_t fake_peak() { const size_t p = peak; peak = used; return p; }
// the nth launch from now of a kernel whose name holds `part` fails, once
void fake_fail_launch(const char* part, int nth) { Lock l(mu); fail_kernel = part; fail_launch_in = nth; }
void fake_fail_copy(int nth) { Lock l(mu); fail_copy_in = nth; }
void fake_watch(const char* part, int argument) { Lock l(mu); watched[part] = argument; }

// ---- the library's side
int hipGetDeviceCount(int* n) { *n = 1; return kSuccess; }
int hipGetDevice(int* d) { *d = 0; return kSuccess; }
int hipSetDevice(int) { return kSuccess; }
int hipDeviceSynchronize() { return kSuccess; }
const char* hipGetErrorString(int) { return "made to fail"; }
int hipGetLastError() { Lock l(mu); const int e = last; last = kSuccess; return e; }
int hipMalloc(void** p, size_t n) { return take(p, n); }
int hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n); }
int hipFree(void* p) { return give(p); }
int hipHostFree(void* p) { return give(p); }
int hipMemcpy(void* d, const void* s, size_t n, int kind) { return copy(d, s, n, kind); }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void*) { return copy(d, s, n, kind); }
int hipMemset(void* d, int v, size_t n) { memset(d, v, n); return kSuccess; }
int hipGetSymbolAddress(void** p, const void*) { return take(p, (size_t)4 << 20); }
int hipStreamCreateWithFlags(void** s, unsigned) { return handle(s); }
int hipStreamDestroy(void*) { return kSuccess; }
int hipStreamSynchronize(void*) { Lock l(mu); note("wait stream"); return kSuccess; }
int hipEventCreate(void** e) { return handle(e); }
int hipEventCreateWithFlags(void** e, unsigned) { return handle(e); }
int hipEventDestroy(void*) { return kSuccess; }
int hipEventRecord(void* e, void*) { Lock l(mu); note("record " + num((size_t)(intptr_t)e)); return kSuccess; }
int hipEventSynchronize(void* e) { Lock l(mu); note("wait " + num((size_t)(intptr_t)e)); return kSuccess; }
int hipEventElapsedTime(float* ms, void*, void*) { *ms = 1.0f; return kSuccess; }
int hipStreamBeginCapture(void*, int) { Lock l(mu); note("capture"); return kSuccess; }
int hipStreamEndCapture(void*, void** g) { return handle(g); }
int hipGraphInstantiate(void** e, void*, void**, char*, size_t) { return handle(e); }
int hipGraphLaunch(void*, void*) { Lock l(mu); note("replay"); return kSuccess; }
int hipGraphDestroy(void*) { return kSuccess; }
int hipGraphExecDestroy(void*) { return kSuccess; }
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels[f] = name;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t shared, void* stream) {
    pushed = Call{g, b, shared, stream};
    return kSuccess;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* shared, void** stream) {
    *g = pushed.grid; *b = pushed.block; *shared = pushed.shared; *stream = pushed.stream;
    return kSuccess;
}
int hipLaunchKernel(const void* f, Dim3 g, Dim3 b, void** args, size_t shared, void*) {
    Lock l(mu);
    const std::string& name = kernels[f];
    std::string line = "launch " + name + " " + num(g.x) + " " + num(g.y) + " " + num(g.z) + " " + num(b.x) + " " + num(shared);
    for (const auto& w : watched)
        if (name.find(w.first) != std::string::npos) line += " " + std::to_string(*(const int*)args[w.second]);
    note(line);
    if (fail_launch_in > 0 && name.find(fail_kernel) != std::string::npos && --fail_launch_in == 0) return done(kUnknown);
    return kSuccess;
}
}
