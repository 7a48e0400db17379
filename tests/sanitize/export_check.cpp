// Exported tables where the host has neither page-locked memory nor 2 MB of ordinary memory for the pieces they are
// copied in: gdp_plan_fetch says so, writes no cost, and the same plan is fetched once there is memory again.
// The operator new of this program is the one the library's containers use.  Run by tests/test_hip_export.py.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "../../include/galvatron_dp_hip.h"

static size_t largest = (size_t)-1;   // larger requests are refused

void *operator new(size_t n)
{
    void *p = n > largest ? nullptr : malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

#define CHECK(x) do { if (!(x)) { printf("line %d: %s (%s)\n", __LINE__, #x, gdp_last_error()); return 1; } } while (0)

int main()
{
    setenv("GALVATRON_DP_PINNED_LIMIT_MB", "1", 1);
    const int L = 3, S = 5, V = 700;
    std::vector<int32_t> mem((size_t)L * S), res(L), mark((size_t)L * V * S, -7);
    std::vector<double> intra((size_t)L * S), inter((size_t)L * S * S, 0.25), f((size_t)V * S, 0.0);
    for (int i = 0; i < L * S; ++i) mem[(size_t)i] = 1 + i * 7, intra[(size_t)i] = 1.0 + i % 4;
    const int64_t other_mem = 0;
    const double other_time = 0.0;
    double total = 0.0;
    int32_t left = 0;
    gdp_problem p = {L, V, S, mem.data(), intra.data(), inter.data(), nullptr, L, 1, &other_mem, &other_time, GDP_EXPORT_F | GDP_EXPORT_MARK, f.data()};
    gdp_result r = {&total, &left, res.data(), f.data(), mark.data()};
    const gdp_problem *pp = &p;
    gdp_result *rr = &r;
    gdp_plan *plan = nullptr;
    CHECK(gdp_plan_create(1, &pp, &plan) == GDP_OK);
    CHECK(gdp_plan_run(plan, 0, nullptr) == GDP_OK);
    largest = 1 << 20;
    CHECK(gdp_plan_fetch(plan, &rr) == GDP_E_NOMEM);
    for (double x : f) CHECK(x == 0.0);
    largest = (size_t)-1;
    CHECK(gdp_plan_fetch(plan, &rr) == GDP_OK);
    CHECK(f[(size_t)(V - 1) * S] > 0.0 && mark[(size_t)(V - 1) * S] >= 0 && left >= 0);
    gdp_plan_destroy(plan);
    printf("fetched\n");
    return 0;
}
