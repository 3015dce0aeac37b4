// jmm_read_samples_noalloc with rows wider than the read: counts the C++
// allocations of 64 KB or more that are made during the call.
#include "jmm_engine.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

static bool g_count = false;
static int g_large = 0;

static void *take(size_t n)
{
    if (g_count && n >= 65536) ++g_large;
    return std::malloc(n ? n : 1);
}

void *operator new(size_t n) { return take(n); }
void *operator new[](size_t n) { return take(n); }
void *operator new(size_t n, const std::nothrow_t &) noexcept { return take(n); }
void *operator new[](size_t n, const std::nothrow_t &) noexcept { return take(n); }
void operator delete(void *p) noexcept { std::free(p); }
void operator delete[](void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
void operator delete[](void *p, size_t) noexcept { std::free(p); }

int main()
{
    const int n = 2000, sweeps = 100, room = 150;
    std::vector<jmm_chain_spec> specs(n);
    for (int c = 0; c < n; ++c) {
        jmm_chain_spec &s = specs[c];
        std::memset(&s, 0, sizeof s);
        s.boundary = JMM_PERIODIC;
        s.nbn = -1;
        s.N = 2;
        s.T = 1.0;
        s.L0 = 20.0;
        s.max_step = 0.5;
        s.cutoff = 3.0;
        s.pot_p[0] = s.pot_p[1] = 1.0;
        s.seed = 3;
        s.chain_id = (uint32_t)c;
    }
    jmm_engine_opts o;
    std::memset(&o, 0, sizeof o);
    o.form = JMM_FORM_BATCHED_FP32;
    o.sample_capacity = sweeps;
    jmm_engine *e = nullptr;
    std::vector<jmm_sample> out((size_t)n * room);
    uint32_t got = 0;
    int rc = jmm_create(specs.data(), n, &o, &e);
    if (!rc) rc = jmm_run_sweeps(e, sweeps);
    if (!rc) rc = jmm_synchronize(e);
    if (!rc) {
        g_count = true;
        rc = jmm_read_samples_noalloc(e, out.data(), room, &got);
        g_count = false;
    }
    std::printf("rc %d sweeps %u large allocations %d\n", rc, got, g_large);
    if (rc) std::printf("%s\n", jmm_last_error());
    jmm_destroy(e);
    return rc || got != (uint32_t)sweeps || g_large ? 1 : 0;
}
