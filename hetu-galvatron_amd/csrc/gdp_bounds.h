// Lower bounds that take strategies out of an instance before its DP runs (kernels: gdp_bounds.hip; the host side
// that builds the smaller instance: reduce_batch in gdp_api.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <stdint.h>

constexpr int GDP_BOUND_MAX_S = 128;      // strategies (an argmin is a byte, a matrix at most 16 elements per thread)
constexpr int GDP_BOUND_MAX_L = 512;      // layers (running sums of four paths in LDS)
constexpr int GDP_BOUND_MAX_LS = 40960;   // layers x strategies: the argmin table of a pass lives in LDS
constexpr int GDP_BOUND_MAX_LAM = 64;     // multipliers
constexpr int GDP_BOUND_MAX_KEY = 8;
constexpr int GDP_BOUND_THREADS = 1024;    // at most, per pass; at least GDP_BOUND_MAX_L
constexpr int GDP_BOUND_PARTS = 32;       // at most this many threads share a target strategy
constexpr int GDP_BOUND_LOW = 3;          // paths above the budget that are spliced with the one below it

struct GdpBoundInst {
    const int32_t *mem;      // [L][S]
    const double *intra;     // [L][S]
    const double *inter;     // [T][S][S]
    const double *inter_t;   // [T][S][S], every matrix transposed
    const int32_t *index;    // [L] layer -> matrix
    const double *lam;       // [NL] ascending, lam[0] = 0
    const int64_t *budget;   // [K] start row of every key; negative: the key has no solution
    double *P, *Q;           // [NL][L][S] cheapest way from the first layer up to (l, s), and from there to the last
    double *path_time;       // [NL] of the cheapest path under multiplier i: its time,
    int64_t *path_mem;       //      its memory
    uint8_t *path;           // [NL][L] and its strategies
    double *ub;              // [K] time of the best path found that fits the budget; +inf: none found
    uint8_t *keep;           // [L][S] 1: (l, s) may lie on a best path of some key
    double magnitude;        // sum over the layers of the largest finite |intra| and |inter|
    int32_t L, V, S, K;
};

// Elements of a transition matrix per thread that instances of S strategies need with that many threads per pass (1, 2,
// 4, 8 or 16; 0: more than that many threads take).
__attribute__((visibility("hidden"))) int gdp_bound_elements(int S, int threads);
// Transposes the matrices, runs the passes of all multipliers, finds the upper bounds and marks what stays.
// pairs: {instance, matrix} of every matrix that is to be transposed.
__attribute__((visibility("hidden")))
hipError_t gdp_launch_bounds(const GdpBoundInst *inst, int n, int n_lam, int max_LS, int max_S, int max_K,
                             int elements, int threads, const int2 *pairs, int n_pairs, hipStream_t stream);
