// A hipMalloc that counts its calls and lets chosen ones find no device memory.  Loaded with
// global symbols before the library under test, so that the library's calls bind to it; a
// call that is to fail asks the real one for more than any device has, so the runtime's own
// error state is what a full device leaves.
#include <dlfcn.h>

#include <cstddef>

namespace {
using Malloc = int (*)(void**, std::size_t);
long calls = 0, failFrom = -1, failCount = 0;

Malloc real() {
    static const Malloc fn = [] {
        void* lib = dlopen("libamdhip64.so", RTLD_NOW);
        return lib ? reinterpret_cast<Malloc>(dlsym(lib, "hipMalloc")) : nullptr;
    }();
    return fn;
}
}  // namespace

extern "C" {

// Calls number `from`, ..., `from + count - 1` from now on fail.
void oom_arm(long from, long count) {
    calls = 0;
    failFrom = from;
    failCount = count;
}

long oom_calls() { return calls; }

int hipMalloc(void** p, std::size_t bytes) {
    const long i = calls++;
    if (!real()) return 1;
    return real()(p, i >= failFrom && i < failFrom + failCount ? std::size_t(1) << 60 : bytes);
}
}
