// A stand-in for the HIP runtime, preloaded by tests of the host code where
// there is no GPU: device memory is the host's (zeroed), copies copy, kernels
// are counted by name and not run, and an allocation or a launch fails when it is
// asked to.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
struct dim3_t {
    uint32_t x, y, z;
};
std::map<const void *, std::string> &names() {
    static std::map<const void *, std::string> m;
    return m;
}
std::map<std::string, long> &launches() {
    static std::map<std::string, long> m;
    return m;
}
std::map<void *, size_t> &blocks() {
    static std::map<void *, size_t> m;
    return m;
}
std::string watched, failing;
int watchedArg = -1, lastError = 0;
long failLaunchAt = -1;
long nulls = 0, failAt = -1, live = 0;
int handle;   // what every stream, event and graph is
constexpr int kOk = 0, kOutOfMemory = 2;

int allocate(void **p, size_t n) {
    *p = nullptr;
    if (failAt >= 0 && failAt-- == 0) return kOutOfMemory;
    *p = std::calloc(n ? n : 1, 1);
    if (!*p) return kOutOfMemory;
    blocks()[*p] = n;
    live += (long)n;
    return kOk;
}
int release(void *p) {
    const auto it = blocks().find(p);
    if (it == blocks().end()) return kOk;
    live -= (long)it->second;
    blocks().erase(it);
    std::free(p);
    return kOk;
}
int copy(void *d, const void *s, size_t n) {
    if (n && (!d || !s)) return 1;   // hipErrorInvalidValue
    std::memmove(d, s, n);
    return kOk;
}
}  // namespace

extern "C" {

// the tests' side: the k-th allocation from now on fails (0: the next, below 0: none)
void fake_hip_fail_at(long k) { failAt = k; }
long fake_hip_pending_failure() { return failAt; }
long fake_hip_live_bytes() { return live; }
// launches of the kernels whose name contains part
long fake_hip_launches(const char *part) {
    long n = 0;
    for (const auto &l : launches())
        if (l.first.find(part) != std::string::npos) n += l.second;
    return n;
}
// counts the launches of such a kernel whose argument (a pointer) is null
void fake_hip_watch(const char *part, int arg) {
    watched = part;
    watchedArg = arg;
    nulls = 0;
}
long fake_hip_nulls() { return nulls; }
// the k-th launch from now on of such a kernel fails
void fake_hip_fail_launch(const char *part, long k) {
    failing = part;
    failLaunchAt = k;
}

void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    names()[fn] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
int __hipPushCallConfiguration(dim3_t, dim3_t, size_t, void *) { return kOk; }
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *s, void **st) {
    *g = *b = dim3_t{1, 1, 1};
    *s = 0;
    *st = nullptr;
    return kOk;
}
int hipLaunchKernel(const void *fn, dim3_t, dim3_t, void **args, size_t, void *) {
    const std::string &name = names()[fn];
    if (failLaunchAt >= 0 && name.find(failing) != std::string::npos && failLaunchAt-- == 0) return lastError = 719;
    ++launches()[name];
    if (watchedArg >= 0 && name.find(watched) != std::string::npos && !*static_cast<void **>(args[watchedArg])) ++nulls;
    return kOk;
}
int hipMalloc(void **p, size_t n) { return allocate(p, n); }
int hipHostMalloc(void **p, size_t n, unsigned) { return allocate(p, n); }
int hipFree(void *p) { return release(p); }
int hipHostFree(void *p) { return release(p); }
int hipMemcpy(void *d, const void *s, size_t n, int) { return copy(d, s, n); }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) { return copy(d, s, n); }
int hipGetDeviceCount(int *n) {
    *n = 1;
    return kOk;
}
int hipSetDevice(int) { return kOk; }
int hipDeviceSynchronize() { return kOk; }
int hipGetLastError() {
    const int e = lastError;
    lastError = kOk;
    return e;
}
const char *hipGetErrorString(int) { return "an error of the stand-in"; }
int hipGetSymbolAddress(void **p, const void *) {
    static void *area = std::calloc(1 << 20, 1);
    *p = area;
    return kOk;
}
int hipStreamCreateWithFlags(void **s, unsigned) {
    *s = &handle;
    return kOk;
}
int hipStreamDestroy(void *) { return kOk; }
int hipStreamSynchronize(void *) { return kOk; }
int hipStreamWaitEvent(void *, void *, unsigned) { return kOk; }
int hipStreamBeginCapture(void *, int) { return kOk; }
int hipStreamEndCapture(void *, void **g) {
    *g = &handle;
    return kOk;
}
int hipEventCreate(void **e) {
    *e = &handle;
    return kOk;
}
int hipEventCreateWithFlags(void **e, unsigned) {
    *e = &handle;
    return kOk;
}
int hipEventDestroy(void *) { return kOk; }
int hipEventRecord(void *, void *) { return kOk; }
int hipEventSynchronize(void *) { return kOk; }
int hipEventElapsedTime(float *ms, void *, void *) {
    *ms = 0;
    return kOk;
}
int hipGraphDestroy(void *) { return kOk; }
int hipGraphExecDestroy(void *) { return kOk; }
int hipGraphInstantiate(void **e, void *, void *, char *, size_t) {
    *e = &handle;
    return kOk;
}
int hipGraphLaunch(void *, void *) { return kOk; }
int hipGraphUpload(void *, void *) { return kOk; }
int hipLaunchHostFunc(void *, void (*fn)(void *), void *user) {
    fn(user);
    return kOk;
}
}
