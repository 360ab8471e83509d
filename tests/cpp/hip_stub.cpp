// The HIP runtime calls libmf3d_hip.so makes, without a GPU: memory is an address
// and a size, kernels are recorded by name and not run, downloads deliver bytes of 1
// (a state that has stopped). Loaded before the library, so that its host code --
// what it allocates, which kernels it chooses, what it does when a call fails -- can
// be checked on a CPU.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
struct Dim {
    unsigned x, y, z;
};
struct Config {
    Dim grid, block;
    size_t shmem;
    void* stream;
};
std::recursive_mutex mu;
std::map<const void*, std::string> names;
std::map<uintptr_t, size_t> live;
std::vector<std::string> log_;
std::vector<Config> configs;
uintptr_t next_addr = uintptr_t(1) << 44;
size_t in_use = 0, limit = SIZE_MAX;
std::string fail_next;  // one call or kernel whose name holds this text
int last_error = 0;
constexpr int kOutOfMemory = 2, kUnknown = 999;

int fails(const std::string& what) {
    if (fail_next.empty() || what.find(fail_next) == std::string::npos) return 0;
    fail_next.clear();
    return last_error = kUnknown;
}
int note(const char* what) {
    std::lock_guard<std::recursive_mutex> l(mu);
    log_.push_back(what);
    return fails(what);
}
void* handle() { return std::malloc(8); }
}  // namespace

extern "C" {
// ---- the test's side
void stub_limit(size_t bytes) { limit = bytes; }
size_t stub_in_use() { return in_use; }
void stub_fail(const char* text) { fail_next = text; }
int stub_log_size() { return (int)log_.size(); }
const char* stub_log(int i) { return log_[i].c_str(); }
void stub_clear() { log_.clear(); }

// ---- the runtime's side
void** __hipRegisterFatBinary(const void*) { return (void**)handle(); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* fn, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*) {
    std::lock_guard<std::recursive_mutex> l(mu);
    names[fn] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t shmem, void* stream) {
    std::lock_guard<std::recursive_mutex> l(mu);
    configs.push_back(Config{grid, block, shmem, stream});
    return 0;
}
int __hipPopCallConfiguration(Dim* grid, Dim* block, size_t* shmem, void** stream) {
    std::lock_guard<std::recursive_mutex> l(mu);
    const Config c = configs.back();
    configs.pop_back();
    *grid = c.grid, *block = c.block, *shmem = c.shmem, *stream = c.stream;
    return 0;
}
int hipLaunchKernel(const void* fn, Dim, Dim, void**, size_t, void*) {
    std::lock_guard<std::recursive_mutex> l(mu);
    return note(names[fn].c_str());
}
int hipMalloc(void** p, size_t n) {
    std::lock_guard<std::recursive_mutex> l(mu);
    if (int e = note("hipMalloc")) return e;
    if (n > limit || in_use > limit - n) return last_error = kOutOfMemory;
    *p = (void*)next_addr;
    live[next_addr] = n;
    in_use += n;
    next_addr += (n + 4095) / 4096 * 4096 + 4096;
    return 0;
}
int hipFree(void* p) {
    std::lock_guard<std::recursive_mutex> l(mu);
    auto it = live.find((uintptr_t)p);
    if (!p) return 0;
    if (it == live.end()) return last_error = kUnknown;
    in_use -= it->second;
    live.erase(it);
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::calloc(1, n);
    return 0;
}
int hipHostFree(void* p) {
    std::free(p);
    return 0;
}
int hipMemset(void*, int, size_t) { return note("hipMemset"); }
static void deliver(void* dst, size_t n, int kind) {
    if (kind == 2) std::memset(dst, 1, n);  // device to host
}
int hipMemcpy(void* dst, const void*, size_t n, int kind) {
    deliver(dst, n, kind);
    return note("hipMemcpy");
}
int hipMemcpyAsync(void* dst, const void*, size_t n, int kind, void*) {
    deliver(dst, n, kind);
    return note("hipMemcpyAsync");
}
int hipDeviceSynchronize() { return note("hipDeviceSynchronize"); }
int hipStreamSynchronize(void*) { return note("hipStreamSynchronize"); }
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { return *s = handle(), 0; }
int hipStreamDestroy(void*) { return 0; }
int hipStreamBeginCapture(void*, int) { return note("hipStreamBeginCapture"); }
int hipStreamEndCapture(void*, void** g) { return *g = handle(), 0; }
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) { return *x = handle(), 0; }
int hipGraphLaunch(void*, void*) { return note("hipGraphLaunch"); }
int hipGraphExecDestroy(void*) { return 0; }
int hipGraphDestroy(void*) { return 0; }
int hipEventCreate(void** e) { return *e = handle(), 0; }
int hipEventCreateWithFlags(void** e, unsigned) { return *e = handle(), 0; }
int hipEventDestroy(void*) { return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* ms, void*, void*) { return *ms = 0.0f, 0; }
int hipGetDevice(int* d) { return *d = 0, 0; }
int hipGetSymbolAddress(void** p, const void*) { return *p = (void*)next_addr, 0; }
int hipGetLastError() {
    const int e = last_error;
    last_error = 0;
    return e;
}
const char* hipGetErrorString(int) { return "stub error"; }
}
