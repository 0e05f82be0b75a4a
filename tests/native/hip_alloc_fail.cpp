// Stands between libmlmq.so and the HIP runtime's allocations (loaded first,
// with RTLD_GLOBAL): lets chosen ones fail as they do where memory runs out,
// by asking the runtime for more than any device has.
#include <dlfcn.h>

#include <cstddef>
#include <map>
#include <mutex>

namespace {

constexpr size_t kTooMuch = (size_t)1 << 60;
std::mutex mu;
std::map<void *, size_t> live;
size_t live_bytes = 0;
int before_failure = -1;   // allocations that still succeed (-1: no failure due)
int failures = 0;

template <typename F>
F real(const char *name) {
    static void *lib = [] {
        void *h = dlopen("libamdhip64.so.7", RTLD_NOW);
        return h ? h : dlopen("/opt/rocm/lib/libamdhip64.so", RTLD_NOW);
    }();
    return reinterpret_cast<F>(dlsym(lib, name));
}

bool due() {
    if (before_failure < 0 || before_failure-- > 0) return false;
    ++failures;
    return true;
}

}  // namespace

extern "C" {

// The next allocation after `successes` more fails (-1: none).
void alloc_fail_after(int successes) {
    std::lock_guard<std::mutex> lk(mu);
    before_failure = successes;
    failures = 0;
}
int alloc_failures(void) { return failures; }
size_t alloc_live(void) { return live_bytes; }   // device bytes

int hipMalloc(void **p, size_t bytes) {
    std::lock_guard<std::mutex> lk(mu);
    const auto f = real<int (*)(void **, size_t)>("hipMalloc");
    if (due()) return f(p, kTooMuch);
    const int e = f(p, bytes);
    if (e == 0) {
        live[*p] = bytes;
        live_bytes += bytes;
    }
    return e;
}

int hipFree(void *p) {
    std::lock_guard<std::mutex> lk(mu);
    const auto it = live.find(p);
    if (it != live.end()) {
        live_bytes -= it->second;
        live.erase(it);
    }
    return real<int (*)(void *)>("hipFree")(p);
}

int hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    std::lock_guard<std::mutex> lk(mu);
    return real<int (*)(void **, size_t, unsigned)>("hipHostMalloc")(p, due() ? kTooMuch : bytes, flags);
}

}  // extern "C"
