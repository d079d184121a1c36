// Parareal solves with a bound on the library's device memory: hipMalloc of this executable, which
// the library calls in the runtime's place, refuses what would exceed it.  Arguments: n, slices,
// coarse kind, path (0 fused, 1 staged).  A solve without a bound, then one whose bound is the
// fields that the solve needs (four slice arrays, three slices, the staged path's five), without
// any for a work field.  Prints "equal" when both give the same bits.
#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "stencilparareal.h"

static size_t g_limit = ~(size_t)0, g_held = 0;
static std::map<void*, size_t> g_sizes;

extern "C" int hipMalloc(void** p, size_t bytes)
{
    using Fn = int (*)(void**, size_t);
    static const Fn real = (Fn)dlsym(RTLD_NEXT, "hipMalloc");
    if (g_held + bytes > g_limit) return 2;  // hipErrorOutOfMemory
    const int r = real(p, bytes);
    if (r == 0) g_held += g_sizes[*p] = bytes;
    return r;
}

extern "C" int hipFree(void* p)
{
    using Fn = int (*)(void*);
    static const Fn real = (Fn)dlsym(RTLD_NEXT, "hipFree");
    const auto it = g_sizes.find(p);
    if (it != g_sizes.end()) {
        g_held -= it->second;
        g_sizes.erase(it);
    }
    return real(p);
}

#define CHECK(call)                                                            \
    do {                                                                       \
        if ((call) != SP_OK) {                                                 \
            std::printf("%s: %s\n", #call, sp_last_error());                   \
            std::exit(1);                                                      \
        }                                                                      \
    } while (0)

int main(int argc, char** argv)
{
    if (argc != 5) return 2;
    const int n = std::atoi(argv[1]), slices = std::atoi(argv[2]), kind = std::atoi(argv[3]), path = std::atoi(argv[4]);
    const size_t field = (size_t)n * n * n * 8;
    sp_ctx* ctx = nullptr;
    CHECK(sp_ctx_create(0, &ctx));
    sp_layout l;
    CHECK(sp_layout_compact(n, n, n, SP_F64, &l));
    void *u = nullptr, *q = nullptr;
    CHECK(sp_malloc(ctx, (long long)field, &u));
    CHECK(sp_malloc(ctx, (long long)field, &q));
    const double at[] = {0.4, 0.7}, sigma[] = {0.1, 0.15}, amp[] = {1.0, 0.5};
    CHECK(sp_fill_gaussians(ctx, &l, u, 2, at, at, at, sigma, amp));

    std::vector<double> out[2];
    for (int bounded = 0; bounded < 2; ++bounded) {
        sp_prop* p = nullptr;
        CHECK(sp_prop_create(ctx, n, n, n, 1. / n, 0.01, 0., 1., -0.5, 0.25, &p));
        CHECK(sp_prop_set_path(p, path));
        sp_parareal_cfg c{};
        c.slices = slices;
        c.kmax = 2;
        c.steps_fine = 4 * slices;
        c.steps_coarse = 2 * slices;
        c.end_time = c.steps_coarse * 1e-4;
        c.coarse_kind = kind;
        c.coarse_dtype = SP_F64;
        c.coarse_substeps = 1;
        if (bounded) g_limit = g_held + (4 * slices + 3 + (path == SP_PATH_STAGED ? 5 : 0)) * field + (1u << 20);
        sp_parareal* pr = nullptr;
        CHECK(sp_parareal_create(p, &c, &pr));
        CHECK(sp_parareal_run(pr, &l, u, &l, q, nullptr));
        out[bounded].resize(field / 8);
        CHECK(sp_memcpy_d2h(ctx, out[bounded].data(), q, (long long)field));
        CHECK(sp_parareal_destroy(pr));
        CHECK(sp_prop_destroy(p));
    }
    const bool equal = std::memcmp(out[0].data(), out[1].data(), field) == 0;
    std::puts(equal && std::isfinite(out[0][0]) ? "equal" : "different");
    return 0;
}
