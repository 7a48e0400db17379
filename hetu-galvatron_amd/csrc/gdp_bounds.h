// Lower bounds that take strategies out of an instance before its DP runs (kernels: gdp_bounds.hip; the host side
// that builds the smaller instance: reduce_batch in gdp_api.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include "../../include/galvatron_dp_hip.h"

constexpr int GDP_BOUND_MAX_S = 128;      // strategies
constexpr int GDP_BOUND_MAX_L = 512;      // layers
constexpr int GDP_BOUND_MAX_LS = 40960;   // layers x strategies
constexpr int GDP_BOUND_MAX_LAM = 128;    // multipliers
constexpr int GDP_BOUND_MAX_KEY = 8;
constexpr int GDP_BOUND_WINDOW = 8;       // multipliers around a key's best one that its upper bound comes from
constexpr double GDP_BOUND_FAR = 1e200;   // for +inf: 512 of them and the costs of a path (below 1e100) have room above
constexpr int GDP_BOUND_MEM = 1 << 30;    // memory sums saturate here, above every budget; two of them fit 32 bits

constexpr int GDP_FRONTIER_KEPT = 8192;   // strategies that stay, over all layers of an instance
constexpr int GDP_FRONTIER_LABELS = 1024; // room in memory for so many labels, and transitions, per layer on average
constexpr int GDP_KEY_LABELS = 512;       // ... so many labels of a key with a workgroup of its own
constexpr int GDP_KEY_LABELS_MAX_L = 128; // its layers
constexpr double GDP_KEY_LABELS_MOST = 0.8;   // share of the strategies that no other one dominates

// What bounds::launch_labels finds for an instance; the strategies lie in GdpBoundInst.res.
struct GdpFrontierOut {
    double total[GDP_BOUND_MAX_KEY];      // +inf: the key has no solution
    double executed[GDP_BOUND_MAX_KEY];   // candidates looked at
    int32_t remaining[GDP_BOUND_MAX_KEY];
    int32_t status[GDP_BOUND_MAX_KEY];    // 0: solved; otherwise nothing else of the key is valid; 1: no path was found for it
};

// From w bins on, strategy s (counted among those of its layer that stay) can be reached at cost c.
struct GdpFrontierLabel {
    double c;
    int32_t w, s;
};

// A matrix on its way to the passes, and what they read of it.
struct GdpBoundMatrix {
    const double *src;       // [S][S], device memory or page-locked host memory
    double *fwd, *bwd;       // the same with GDP_BOUND_FAR for +inf, and transposed
    int32_t S, pad;
};

struct GdpBoundInst {
    const int32_t *mem;      // [L][S]
    const double *intra;     // [L][S]
    double *inter_f;         // [T][S][S], GDP_BOUND_FAR for +inf
    double *inter_t;         // [T][S][S], the same with every matrix transposed
    const int32_t *index;    // [L] layer -> matrix
    const double *lam;       // [NL] ascending, lam[0] = 0
    const int64_t *budget;   // [K] start row of every key; negative: the key has no solution
    double *P, *Q;           // [NL][L][S] cheapest way from the first layer up to (l, s), and from there to the last
    uint32_t *P_mem, *Q_mem; // [NL][L][S] memory of those ways
    double *end;             // [NL] cheapest way through all layers
    unsigned long long *ub;  // [K] time of the best path found that fits the budget, ordered as an unsigned number; ~0: none found
    int32_t *best;           // [K] the multiplier whose bound is the best
    uint8_t *keep;           // [L][S] bit k: (l, s) may lie on a best path of key k
    unsigned long long *marks;   // [K][L][2] the same by key, strategies 0 to 63 and from 64 on; 16-byte aligned
    const double *other_time;// [K]
    // of the frontier: the labels of all layers, the transitions between and the costs of what stays, the results; of keys with a
    // workgroup of their own one after the other
    GdpFrontierLabel *hist;
    int32_t *hist_mem;
    double *hist_turns, *hist_intra;
    GdpFrontierOut *out;     // this and `res`: device memory, or page-locked host memory
    int32_t *res;            // [K][L]
    double magnitude;        // sum over the layers of the largest finite |intra| and |inter|
    double limit;            // ns that the layers ahead of the DP over what stays may take, by its own account
    int32_t L, V, S, K, T, n_hist, n_hist_turns, n_lam;
};

// Nothing in here allocates: gdp_solve_static uses it too.
namespace bounds {
// Whether an instance has the form, its costs apart (reducible in gdp_api.hip).
__attribute__((visibility("hidden"))) bool has_form(const gdp_problem *q);
// What the environment says of bounds: false with GALVATRON_DP_REDUCE=0 and with GALVATRON_DP_SKIP=0 (every cell is asked for);
// *forced: with GALVATRON_DP_REDUCE=1 (every instance that has the form takes them).
__attribute__((visibility("hidden"))) bool allowed(bool *forced);
// Share of the strategies of a layer, and on average of 4 layers, that are cheaper in time than every one that needs no more memory.
__attribute__((visibility("hidden"))) double undominated(const gdp_problem *q, int layer);
__attribute__((visibility("hidden"))) double undominated(const gdp_problem *q);
// How many multipliers an instance takes whose keys have a workgroup each, given the share of its undominated strategies.
__attribute__((visibility("hidden"))) int key_multipliers(const gdp_problem *q, double undominated);
// The multipliers of an instance: 0 and a geometric series around (range of times) / (range of memory costs).
__attribute__((visibility("hidden"))) void multipliers(const gdp_problem *q, int n_lam, double *lam);
// What is laid out before a set of launches: head_bytes (a multiple of 16) are copied from `head`, if there is one, page-locked host memory,
// to head_to, and the matrices are laid out.
struct Inputs {
    const GdpBoundMatrix *matrices;
    int n_matrices;
    const void *head;
    void *head_to;
    size_t head_bytes;
};
__attribute__((visibility("hidden"))) hipError_t lay_out(const Inputs &in, int max_S, hipStream_t stream);
// Runs the passes of all multipliers, finds the upper bounds and marks what stays.
// max_rows: layers times (strategies / 64, rounded up).  held: most layers have the matrix of the one before.
__attribute__((visibility("hidden")))
hipError_t launch(const GdpBoundInst *inst, int n, int n_lam, int max_LS, int max_rows, int max_S, int max_K, bool held,
                  hipStream_t stream);
// The DP over what stays, after it: a workgroup per instance (gdp_frontier.hip), or per key of each (gdp_key_labels.hip; up to
// GDP_KEY_LABELS_MAX_L layers).
__attribute__((visibility("hidden"))) hipError_t launch_labels(const GdpBoundInst *inst, int n, int max_K, hipStream_t stream);
__attribute__((visibility("hidden"))) hipError_t launch_key_labels(const GdpBoundInst *inst, int n, int max_K, hipStream_t stream);
// Of all keys of an instance: 0 solved, 1 no path was found for one, otherwise given up; candidates looked at.
inline int status_of(const GdpFrontierOut &o, int K)
{
    int status = 0;
    for (int k = 0; k < K; ++k)
        if (o.status[k] == 1) return 1;
        else if (o.status[k] != 0) status = o.status[k];
    return status;
}
inline double executed_of(const GdpFrontierOut &o, int K)
{
    double sum = 0;
    for (int k = 0; k < K; ++k) sum += o.executed[k];
    return sum;
}
// What stays of q, given the marks ([L][S]), as arrays of R strategies a layer: kept[L][R] is the strategy of q, or -1 for
// padding, which costs +inf; memory costs less cut[l] (may be null).  matrix(l): that of layer l of q.  R: the most that
// stay of a layer, at least; at least one stays of every layer.  inter [L][R][R] and intra hold zeros and +inf before.
template <class Matrix>
void fill_kept(const gdp_problem *q, const uint8_t *keep, int R, Matrix matrix, const int32_t *cut, int32_t *kept_of, int32_t *mem, double *intra,
               double *inter)
{
    const int L = q->L, S = q->S;
    int before = 0;
    for (int l = 0; l < L; ++l) {
        int32_t *kept = kept_of + (size_t)l * R;
        int n = 0;
        for (int s = 0; s < S; ++s)
            if (keep[(size_t)l * S + s]) kept[n++] = s;
        for (int j = n; j < R; ++j) kept[j] = -1;
        const double *M = matrix(l);
        double *to = inter + (size_t)l * R * R;
        for (int j = 0; j < R; ++j) {
            const int s = kept[j < n ? j : n - 1];
            mem[(size_t)l * R + j] = q->mem[(size_t)l * S + s] - (cut ? cut[l] : 0);
            if (j >= n) continue;
            intra[(size_t)l * R + j] = q->intra[(size_t)l * S + s];
            if (l == 0) {   // the zeros before the first layer are reached from every strategy: its cheapest transition
                double c = INFINITY;
                for (int sp = 0; sp < S; ++sp) {
                    const double x = 0.0 + M[(size_t)sp * S + s];
                    c = x < c ? x : c;
                }
                for (int i = 0; i < R; ++i) to[(size_t)i * R + j] = c;
            } else {
                for (int i = 0; i < before; ++i) to[(size_t)i * R + j] = M[(size_t)kept_of[(size_t)(l - 1) * R + i] * S + s];
            }
        }
        before = n;
    }
}
}  // namespace bounds

#ifdef __HIPCC__
// A double from an unsigned number of the same order.
__device__ __forceinline__ double gdp_unordered(unsigned long long o)
{
    return __longlong_as_double((long long)(o >> 63 ? o & ~(1ull << 63) : ~o));
}

// Rounding of P and Q under multiplier lam: sums of at most 2 L + 2 terms whose magnitudes add up to no more than
// magnitude + lam * (L + 1) * V, each rounded, and cut to make room for an index, by no more than 2^-45 of it.
__device__ __forceinline__ double gdp_bound_margin(int L, int V, double magnitude, double lam)
{
    return 4.0 * (double)(L + 4) * 0x1p-45 * (magnitude + lam * ((double)(L + 1) * (double)V));
}
#endif
