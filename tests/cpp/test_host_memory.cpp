// Pinned host memory and threads of the host call (get_offset): none for plans that make
// no call or one, then one block for all plans that call in turn, as large as the largest
// batch needs, and all of it given back with the last plan; results do not depend on it.
// Counts the library's hipHostMalloc and hipHostFree by standing in front of the runtime's.
#include <dirent.h>
#include <dlfcn.h>
#include <emida_amd.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <vector>

static std::mutex g_mu;
static std::map<void*, size_t> g_pinned;
static size_t g_live = 0, g_most = 0, g_calls = 0;

extern "C" int hipHostMalloc(void** p, size_t n, unsigned flags) {
    static auto real = (int (*)(void**, size_t, unsigned))dlsym(RTLD_NEXT, "hipHostMalloc");
    const int rc = real(p, n, flags);
    std::lock_guard<std::mutex> lock(g_mu);
    if (rc == 0) {
        g_pinned[*p] = n;
        g_live += n;
        if (g_live > g_most) g_most = g_live;
        ++g_calls;
    }
    return rc;
}
extern "C" int hipHostFree(void* p) {
    static auto real = (int (*)(void*))dlsym(RTLD_NEXT, "hipHostFree");
    {
        std::lock_guard<std::mutex> lock(g_mu);
        auto it = g_pinned.find(p);
        if (it != g_pinned.end()) {
            g_live -= it->second;
            g_pinned.erase(it);
        }
    }
    return real(p);
}

static int g_failures = 0;
#define CHECK(cond)                                                            \
    do {                                                                       \
        if (!(cond)) {                                                         \
            std::fprintf(stderr, "FAILED line %d: %s (live %zu, most %zu, calls %zu)\n", __LINE__, #cond, g_live, \
                         g_most, g_calls);                                     \
            ++g_failures;                                                      \
        }                                                                      \
    } while (0)

static void ok(int rc, const char* what) {
    if (rc != EMIDA_OK) {
        std::fprintf(stderr, "%s: error %d: %s\n", what, rc, emida_last_error());
        std::exit(2);
    }
}

static size_t threads() {
    size_t n = 0;
    DIR* d = opendir("/proc/self/task");
    while (d && readdir(d)) ++n;
    if (d) closedir(d);
    return n;
}

struct plan {
    emida_offset* h = nullptr;
    uint32_t w;
    std::vector<uint16_t> ref, pic;
    explicit plan(uint32_t side) : w(side), ref((size_t)side * side), pic(ref.size()) {
        for (uint32_t y = 0; y < w; ++y)
            for (uint32_t x = 0; x < w; ++x)
                for (int k = 0; k < 2; ++k) {
                    const double u = x - 1.3 * k, v = y + 0.6 * k;
                    (k ? pic : ref)[(size_t)y * w + x] = (uint16_t)(
                        30000 + 9000 * std::sin(0.31 * u + 0.15 * v) + 7000 * std::cos(0.17 * u - 0.43 * v));
                }
        const emida_size2 begins[2] = {{3, 5}, {w - 40, w - 40}};
        ok(emida_offset_create(&h, EMIDA_F32, EMIDA_U16, {w, w}, begins, 2, {32, 32}, {63, 63}, 1,
                               EMIDA_CROSS_POLICY_FFT, 3, 1),
           "create");
        ok(emida_offset_allocate_memory(h, ref.data()), "allocate");
    }
    ~plan() { emida_offset_destroy(h); }
    std::vector<double> call() {
        std::vector<double> r(2 * 8);
        ok(emida_offset_get_offset(h, pic.data(), r.data(), r.data() + 4), "get_offset");
        return r;
    }
};

int main() {
    const size_t small = (512 << 10) + (256 << 10), large = (size_t)2 * 1100 * 1100 + (512 << 10);
    std::vector<double> first, again;
    { plan warm(64); first = warm.call(); }  // the runtime's own threads and memory
    for (double v : first) CHECK(std::isfinite(v));
    CHECK(g_live == 0 && g_calls == 0);
    const size_t before = threads();
    {
        plan a(500), b(500), c(1100);
        CHECK(g_calls == 0 && threads() == before);
        first = a.call();
        CHECK(g_calls == 0 && threads() == before);
        for (int i = 0; i < 3; ++i) {
            again = a.call();
            CHECK(again == first);
        }
        CHECK(g_calls == 1 && g_live <= small);
        CHECK(b.call() == first && b.call() == first);  // the same pixels
        CHECK(g_calls == 1);
        const auto l = c.call();
        CHECK(g_calls == 2 && g_live <= small + large);
        CHECK(c.call() == l && a.call() == first);
        CHECK(g_calls == 2);
    }
    CHECK(g_live == 0);
    for (int i = 0; i < 3; ++i) {  // one plan after the other, a call each
        plan p(500);
        CHECK(p.call() == first);
    }
    CHECK(g_calls == 2 && g_live == 0);
    if (g_failures) return 1;
    std::printf("host memory: ok\n");
    return 0;
}
