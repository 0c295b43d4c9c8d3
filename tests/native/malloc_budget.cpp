// hipMalloc and hipFree with a budget, loaded into a process of its own before
// the library so that its calls resolve here (tests/memory_check.py): device
// memory that runs out without any running out.
#include <dlfcn.h>

#include <cstddef>
#include <map>
#include <mutex>
#include <vector>

namespace {
std::mutex mutex;
std::map<void*, size_t> sizes;
std::vector<size_t> asked;
size_t used = 0, limit = ~(size_t)0;

template <typename F>
F real(const char* name) {
    static void* hip = dlopen("libamdhip64.so.7", RTLD_LAZY);
    return reinterpret_cast<F>(dlsym(hip, name));
}
}  // namespace

extern "C" {

int hipMalloc(void** p, size_t n) {
    static auto* f = real<int (*)(void**, size_t)>("hipMalloc");
    std::lock_guard<std::mutex> l(mutex);
    asked.push_back(n);
    if (n > limit || used > limit - n) return 2;  // hipErrorOutOfMemory
    const int e = f(p, n);
    if (e == 0) {
        sizes[*p] = n;
        used += n;
    }
    return e;
}

int hipFree(void* p) {
    static auto* f = real<int (*)(void*)>("hipFree");
    std::lock_guard<std::mutex> l(mutex);
    const auto it = sizes.find(p);
    if (it != sizes.end()) {
        used -= it->second;
        sizes.erase(it);
    }
    return f(p);
}

// Room for `bytes` beside what is allocated now.
void budget_room(size_t bytes) {
    std::lock_guard<std::mutex> l(mutex);
    limit = used + bytes;
}
void budget_off() {
    std::lock_guard<std::mutex> l(mutex);
    limit = ~(size_t)0;
}
size_t budget_used() { return used; }
// Sizes asked for since the last call; returns how many there were.
size_t budget_asked(size_t* out, size_t capacity) {
    std::lock_guard<std::mutex> l(mutex);
    const size_t n = asked.size();
    for (size_t i = 0; i < n && i < capacity; i++) out[i] = asked[i];
    asked.clear();
    return n;
}
}
