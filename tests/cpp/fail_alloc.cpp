// hipMalloc and hipHostMalloc in front of the HIP runtime's, for tests of a full device
// and of missing page-locked memory: loaded with global symbols before libqmb, which then
// calls these. A call whose size lies in the chosen range fails once `skip` such calls
// have succeeded, `times` times; every other call goes through.
#include <dlfcn.h>

#include <cstddef>

namespace {
struct Rule {
    size_t lo = 1, hi = 0;  // no size
    int skip = 0, error = 0, times = 0, failed = 0;
    bool hit(size_t bytes) {
        if (bytes < lo || bytes > hi || failed == times) return false;
        if (skip > 0) {
            --skip;
            return false;
        }
        ++failed;
        return true;
    }
} device_rule, host_rule;

void *runtime(const char *name) {
    static void *lib = dlopen("libamdhip64.so.7", RTLD_LAZY);
    return dlsym(lib, name);
}
constexpr int kOutOfMemory = 2;          // hipErrorOutOfMemory
constexpr size_t kTooMuch = (size_t)1 << 45;  // more than any device has
}  // namespace

extern "C" {

// Out of memory (error = 2) is the runtime's own answer to a request that no device can
// hold, so that its last error is set as in earnest; other errors are returned as given.
int hipMalloc(void **p, size_t bytes) {
    static auto real = reinterpret_cast<int (*)(void **, size_t)>(runtime("hipMalloc"));
    if (!device_rule.hit(bytes)) return real(p, bytes);
    return device_rule.error == kOutOfMemory ? real(p, kTooMuch) : device_rule.error;
}

int hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    static auto real = reinterpret_cast<int (*)(void **, size_t, unsigned)>(runtime("hipHostMalloc"));
    if (!host_rule.hit(bytes)) return real(p, bytes, flags);
    return host_rule.error;
}

void fail_device(size_t lo, size_t hi, int skip, int error, int times) {
    device_rule = Rule{lo, hi, skip, error, times, 0};
}
void fail_host(size_t lo, size_t hi, int skip, int error, int times) { host_rule = Rule{lo, hi, skip, error, times, 0}; }
int failed_device() { return device_rule.failed; }
int failed_host() { return host_rule.failed; }
}
