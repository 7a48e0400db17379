// Lower bounds per (layer, strategy), so that the DP runs over the strategies that can matter only.
//
// For a multiplier lam >= 0 per bin of memory the budget can be priced instead of counted: with costs
// intra + lam * mem the cheapest path through the layers is a plain min-plus product of L vectors and matrices,
// S*S operations per layer instead of V*S*S.  P[l][s] is the cheapest way from the first layer to (l, s), both ends
// included, Q[l][s] the cheapest way on from there; every path that uses (l, s) and fits the budget B takes at least
//     P[l][s] + Q[l][s] - lam * B
// of time.  Any path that fits gives an upper bound U on the optimum.  Where the lower bound exceeds U (by more than
// the rounding of both) no optimal path of that budget uses (l, s), and no path that ties with one does: the DP
// without (l, s) has the same value in every cell of an optimal path -- a cheaper way into such a cell through
// (l, s) would be a path below U -- and values elsewhere can only be larger, so that no candidate ties that did not
// tie before.  The optimum, its strategies (ties to the lowest index: the order of what stays is kept) and what is
// left of the budget are those of the whole instance, bit for bit.
//
// The bounds are loose by what the last layers before the budget waste, a fraction of one layer, while most
// strategies lose more than that against the best ones: of 64 strategies 1 to 7 per layer stay, 2 on average (L = 80, random
// costs), of 40 of a layer that is repeated 28 times and trades memory for time 20.
#include "gdp_bounds.h"

#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>

namespace {

static_assert(GDP_BOUND_MAX_S == 128, "two blocks of 64 targets; a strategy in the low 7 bits of a candidate");

// The inputs as the passes read them, which takes more than its name says.  First workgroups of 16 KB of `head` each, which go where they are read from then on; then a
// 16-row band of a matrix each, as it is and transposed, +inf replaced by GDP_BOUND_FAR; LDS turns the band around so that both
// sides are read and written along rows.
// Both may lie in page-locked host memory: what the copy engine would bring in a copy of its own, and the first kernel would wait for
// through a signal between the two (20 us and more of a call), comes over the bus where it is needed.
typedef unsigned uint4v __attribute__((ext_vector_type(4)));
constexpr int HEAD = 1024;   // times 16 bytes
__global__ __launch_bounds__(256) void gdp_bound_transpose_kernel(const GdpBoundMatrix *matrices, int bands, const uint4v *head, uint4v *head_to, int n_head)
{
    __shared__ double tile[16][GDP_BOUND_MAX_S + 1];
    const int head_blocks = (n_head + HEAD - 1) / HEAD, b = (int)blockIdx.x - head_blocks;
    if (b < 0) {
        const int first = (int)blockIdx.x * HEAD + (int)threadIdx.x;
        uint4v x[HEAD / 256];
#pragma unroll
        for (int i = 0; i < HEAD / 256; ++i) x[i] = head[min(first + 256 * i, n_head - 1)];
#pragma unroll
        for (int i = 0; i < HEAD / 256; ++i)
            if (first + 256 * i < n_head) head_to[first + 256 * i] = x[i];
        return;
    }
    const GdpBoundMatrix M = matrices[b / bands];
    const int S = M.S, r0 = b % bands * 16;
    if (r0 >= S) return;
    const int rows = S - r0 < 16 ? S - r0 : 16, all = rows * S;
    const double *const src = M.src + (size_t)r0 * S;
    double x[16 * GDP_BOUND_MAX_S / 256];
#pragma unroll
    for (int i = 0; i < 16 * GDP_BOUND_MAX_S / 256; ++i)   // all of them on their way at once
        if (i * 256 < all) x[i] = src[min((int)threadIdx.x + 256 * i, all - 1)];
#pragma unroll
    for (int i = 0; i < 16 * GDP_BOUND_MAX_S / 256; ++i) {
        const int e = (int)threadIdx.x + 256 * i;
        if (e >= all) continue;
        const double y = fmin(x[i], GDP_BOUND_FAR);
        tile[e / S][e % S] = y;
        M.fwd[(size_t)r0 * S + e] = y;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < all; e += 256) {
        const int c = e / rows, r = e % rows;
        M.bwd[(size_t)c * S + r0 + r] = tile[r][c];
    }
}

// Global memory, said so: the compiler takes a pointer that comes from memory for one that may point anywhere, and waits
// for everything under way around what it may point at.
typedef const __attribute__((address_space(1))) double *gdouble;
typedef const __attribute__((address_space(1))) int32_t *gint;
typedef __attribute__((address_space(1))) double *gout;
typedef __attribute__((address_space(1))) uint32_t *guint;
typedef const __attribute__((address_space(1))) uint32_t *guint_in;
typedef __attribute__((address_space(1))) unsigned long long *gulong;

__device__ __forceinline__ double min_f64(double a, double b)
{
    double r;   // the bare instruction: no operand is a NaN
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

typedef unsigned uint2v __attribute__((ext_vector_type(2)));
typedef int int2v __attribute__((ext_vector_type(2)));   // the words of a double, without the shifts of __hiloint2double

// Minimum over the lanes l, l ^ 16, l ^ 32 and l ^ 48, in all four.  (A swap of two copies of x leaves the even rows, or
// the lower half, twice in one and the others twice in the other.)
__device__ __forceinline__ double min_of_rows(double x)
{
    const uint2v w = __builtin_bit_cast(uint2v, x);
    const uint2v lo = __builtin_amdgcn_permlane16_swap(w.x, w.x, false, false), hi = __builtin_amdgcn_permlane16_swap(w.y, w.y, false, false);
    const uint2v a = {lo.x, hi.x}, b = {lo.y, hi.y};
    x = min_f64(__builtin_bit_cast(double, a), __builtin_bit_cast(double, b));
    const uint2v v = __builtin_bit_cast(uint2v, x);
    const uint2v lo2 = __builtin_amdgcn_permlane32_swap(v.x, v.x, false, false), hi2 = __builtin_amdgcn_permlane32_swap(v.y, v.y, false, false);
    const uint2v c = {lo2.x, hi2.x}, d = {lo2.y, hi2.y};
    return min_f64(__builtin_bit_cast(double, c), __builtin_bit_cast(double, d));
}

constexpr int INDEX = GDP_BOUND_MAX_S - 1;   // low bits of a candidate that hold its source strategy
constexpr int TARGETS = 16;                  // target strategies of a wave: 16 lanes read a line of 128 bytes
constexpr int PARTS = 64 / TARGETS;          // lanes that share one of them

// x with `index`, a constant, in its low bits; high: ~INDEX, in a register (v_and_or_b32 takes no other constant).
__device__ __forceinline__ double with_index(double x, int index, int high)
{
    int2v w = __builtin_bit_cast(int2v, x);
    w.x = (w.x & high) | index;
    return __builtin_bit_cast(double, w);
}

// An array as the buffer instructions see it: an address is a register of the lane plus one of the wave, no arithmetic.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *p, size_t bytes)
{
    const uintptr_t a = (uintptr_t)p;   // the same in all lanes, said so
    const uintptr_t u = (uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32 |
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)a);
    return __builtin_amdgcn_make_buffer_rsrc((void *)u, 0, __builtin_amdgcn_readfirstlane((int)(uint32_t)bytes), 0x27000);
}

__device__ __forceinline__ double load_double(__amdgpu_buffer_rsrc_t b, int lane_bytes, int wave_bytes)
{
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b, lane_bytes, wave_bytes, 0));
}

// One pass over the layers of one instance under one multiplier: forwards (P) or backwards (Q), and the memory of the
// paths behind them.  grid (2 * multipliers, instances); a wave has 16 target strategies and 4 lanes for each, a lane up to
// E of the source strategies.  A step is E candidates per lane, two exchanges between the 4 lanes and one barrier, behind
// which every wave reads all sources back from LDS.  A candidate carries its source in its low bits, so that the
// minimum is the argmin as well, and what the path behind it needs of memory is one look into LDS beside the chain.
// The serial chain of L steps is what takes the time, and in it the instructions that a SIMD issues: 4 waves of 16 sources
// per lane, not 16 of 4, whose reductions and addresses cost as much again each; matrices are AHEAD steps ahead in registers.
// What it reads is bound by how many lines a load touches: 4 lanes of a target side by side, a line for every 4 lanes, took
// 151 us where 16 targets side by side take 69.  Against a step of two barriers, 1024 threads and a select per candidate for
// the argmin: L = 80, S = 64 131 -> 69 us, L = 48, S = 88 102 -> 77, 256 instances of S = 44 635 -> 400.
// HELD: for instances whose layers mostly have the matrix of the layer before.  It stays in registers, and is waited for
// where it changes: what a compute unit reads, 16 bytes a clock, is what bounds the pass otherwise.
// L = 48, S = 88 77 -> 39 us, 256 instances of S = 44 400 -> 140; where every layer has a matrix of its own (L = 80, S = 64,
// 70 us) there is nothing to hold.
template <int E, int AHEAD, bool HELD>
__global__ __launch_bounds__(64 * GDP_BOUND_MAX_S / TARGETS) void gdp_bound_pass_kernel(const GdpBoundInst *inst)
{
    static_assert(E % 2 == 0 && AHEAD % 2 == 0 && E * PARTS <= GDP_BOUND_MAX_S, "");
    constexpr int STRIDE = E + 2;   // of the sources of a part: 16 bytes at a time from 4 different places in the banks
    __shared__ __align__(16) double X[2][PARTS * STRIDE];
    __shared__ uint32_t need[2][GDP_BOUND_MAX_S];    // memory of the path behind each source
    __shared__ int32_t mat[GDP_BOUND_MAX_L];
    const GdpBoundInst &I = inst[blockIdx.y];
    const int L = I.L, S = I.S, V = I.V, t = (int)threadIdx.x, li = (int)blockIdx.x >> 1;
    const bool back = blockIdx.x & 1u;
    const double lam = ((gdouble)(uintptr_t)I.lam)[li];
    const int p = (t & 63) / TARGETS, target = (t >> 6) * TARGETS + t % TARGETS, s = min(target, S - 1);
    for (int l = t; l < L; l += (int)blockDim.x) mat[l] = ((gint)(uintptr_t)I.index)[l];
    for (int e = t; e < PARTS * STRIDE; e += (int)blockDim.x) X[0][e] = X[1][e] = GDP_BOUND_FAR * 0x1p40;   // sources beyond S
    if (blockIdx.x == 0 && t < I.K) ((gulong)(uintptr_t)I.ub)[t] = ~0ull;
    const size_t LS = (size_t)L * S;
    const __amdgpu_buffer_rsrc_t tables = buffer_of(back ? I.inter_t : I.inter_f, (size_t)I.T * S * S * 8),
                                 intra = buffer_of(I.intra, LS * 8), mem = buffer_of(I.mem, LS * 4),
                                 out = buffer_of((back ? I.Q : I.P) + li * LS, LS * 8),
                                 out_mem = buffer_of((back ? I.Q_mem : I.P_mem) + li * LS, LS * 4);
    const bool mine = p == 0 && target < S;
    const int place = target / E * STRIDE + target % E;   // of this target among the sources of the next step
    int at[E];                                            // of the elements of a matrix, in bytes
#pragma unroll
    for (int j = 0; j < E; ++j) at[j] = (min(p * E + j, S - 1) * S + s) * 8;

    // What a step needs from memory: its part of the matrix and the costs of the layer whose strategies it reaches.
    struct Inputs {
        double m[HELD ? 1 : E], intra;
        int32_t mem;
    };
    double m[HELD ? E : 1];
    int held = -1;
    // step i: the matrix of layer first + i * step, into the strategies of layer to + i * step
    const int first = back ? L - 1 : 0, to = back ? L - 2 : 0, step = back ? -1 : 1, steps = back ? L - 1 : L;
    auto fetch_costs = [&](int l, Inputs &in) {
        in.mem = __builtin_amdgcn_raw_buffer_load_b32(mem, s * 4, l * S * 4, 0);
        in.intra = load_double(intra, s * 8, l * S * 8);
    };
    auto matrix_of = [&](int i) { return mat[first + min(i, steps - 1) * step]; };
    auto fetch_matrix = [&](int matrix, double *into) {
#pragma unroll
        for (int j = 0; j < E; ++j) into[j] = load_double(tables, at[j], matrix * S * S * 8);
    };
    auto fetch = [&](int i, int matrix, Inputs &in) {
        if constexpr (!HELD) fetch_matrix(__builtin_amdgcn_readfirstlane(matrix), in.m);
        fetch_costs(to + i * step, in);
    };
    auto cost = [&](const Inputs &in) {
        return in.mem < V && in.intra < GDP_BOUND_FAR ? in.intra + lam * (double)in.mem : GDP_BOUND_FAR;
    };
    auto more = [](uint32_t m, int32_t by) { return min(m + (uint32_t)by, (uint32_t)GDP_BOUND_MEM); };   // by: <= GDP_BOUND_MEM
    // What a step found, to be written while the next one computes: the layer, costs, the memory behind them, on its way
    // from LDS, and what the strategy itself needs.
    struct Found {
        int layer;
        double x;
        uint32_t m;
        int32_t by;
    } found = {0, 0.0, 0, 0};
    auto write = [&](int i) {   // what step i - 1 found
        const uint32_t m2 = more(found.m, found.by);
        const int row = __builtin_amdgcn_readfirstlane(found.layer) * S;
        if (mine) {
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, found.x), out, s * 8, row * 8, 0);
            __builtin_amdgcn_raw_buffer_store_b32(back ? found.m : m2, out_mem, s * 4, row * 4, 0);
            need[i & 1][target] = m2;
        }
    };
    __syncthreads();
    if (back) {
        Inputs last;
        fetch_costs(L - 1, last);
        found.layer = L - 1;
        found.by = min(last.mem, GDP_BOUND_MEM);
        if (mine) X[0][place] = cost(last);
    } else if (mine) {   // (what the first step writes of layer 0 is overwritten by the second)
        X[0][place] = 0.0;
    }
    constexpr int LOOK = HELD ? 0 : AHEAD;   // steps from one that looks a matrix up to the one that uses it
    int next_matrix = matrix_of(LOOK);
    int high = ~INDEX;
    asm volatile("" : "+v"(high));   // in a register
    const int part = p * E;
    auto pass = [&](int i, Inputs &in) {
        write(i);
        if constexpr (HELD) {
            const int matrix = __builtin_amdgcn_readfirstlane(next_matrix);
            if (matrix != held) fetch_matrix(matrix, m);
            held = matrix;
        }
        const double *const M = HELD ? m : in.m;
        __syncthreads();   // the other half of X and `need` is still being read until the next one
        const double *from = X[i & 1] + p * STRIDE;
        double best[2];
#pragma unroll
        for (int j = 0; j < E; j += 2) {
            const double a = with_index(from[j] + M[j], j, high), b = with_index(from[j + 1] + M[j + 1], j + 1, high);
            best[0] = j ? min_f64(best[0], a) : a;
            best[1] = j ? min_f64(best[1], b) : b;
        }
        const double c = cost(in);
        int32_t by = min(in.mem, GDP_BOUND_MEM);
        asm volatile("" : "+v"(by));   // here, and not as a copy at the top of the loop that waits for every load
        fetch(min(i + AHEAD, steps - 1), next_matrix, in);   // the last ones once more: no branch
        next_matrix = matrix_of(i + LOOK + 1);
        int2v w = __builtin_bit_cast(int2v, min_f64(best[0], best[1]));
        w.x += part;
        double x = __builtin_bit_cast(double, w);
        x = min_of_rows(x);
        const double z = x + c;
        if (mine) X[(i + 1) & 1][place] = z;
        const uint32_t m = need[i & 1][__builtin_bit_cast(int2v, x).x & INDEX];
        const bool real = i < steps;
        found.x = !real ? found.x : back ? x : z;
        found.m = real ? m : found.m;
        found.by = real ? by : found.by;
        found.layer = real ? to + i * step : found.layer;
    };
    Inputs in[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
        fetch(min(a, steps - 1), matrix_of(a), in[a]);
        __builtin_amdgcn_sched_barrier(0);   // in this order: the first step waits for the first of them only
    }
    // Whole turns of AHEAD steps: a way out in between would make the registers of every turn wait for all loads.  Steps
    // beyond the last find nothing new.
    int i = 0;
    for (; i < steps; i += AHEAD)
#pragma unroll
        for (int a = 0; a < AHEAD; ++a) pass(i + a, in[a]);
    write(i);
    if (back) return;
    // the cheapest end
    __syncthreads();
    if (mine) X[0][target] = found.x;
    __syncthreads();
    if (t >= 64) return;
    double least = X[0][min(t, S - 1)];
    least = min_f64(least, X[0][min(t + 64, S - 1)]);
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) least = min_f64(least, __shfl_xor(least, w));
    if (t == 0) ((gout)(uintptr_t)I.end)[li] = least;
}

// Doubles as unsigned numbers of the same order, for atomicMin.
__device__ __forceinline__ unsigned long long ordered(double x)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    return b >> 63 ? ~b : b | 1ull << 63;
}

__device__ __forceinline__ double of_lane(double x, int lane)
{
    const int2v w = __builtin_bit_cast(int2v, x);
    const int2v r = {__builtin_amdgcn_readlane(w.x, lane), __builtin_amdgcn_readlane(w.y, lane)};
    return __builtin_bit_cast(double, r);
}

// Minimum over a wave, in all lanes.
template <int CTRL, int ROWS>
__device__ __forceinline__ double lower_of_moved(double x)
{
    const int2v w = __builtin_bit_cast(int2v, x);   // a lane without a source keeps its own
    const int2v m = {__builtin_amdgcn_update_dpp(w.x, w.x, CTRL, ROWS, 0xf, false), __builtin_amdgcn_update_dpp(w.y, w.y, CTRL, ROWS, 0xf, false)};
    return min_f64(x, __builtin_bit_cast(double, m));
}
__device__ __forceinline__ double lowest_of(double x)
{
    x = lower_of_moved<0x111, 0xf>(x);   // row_shr:1, 2, 4, 8
    x = lower_of_moved<0x112, 0xf>(x);
    x = lower_of_moved<0x114, 0xf>(x);
    x = lower_of_moved<0x118, 0xf>(x);
    x = lower_of_moved<0x142, 0xa>(x);   // row_bcast:15, 31
    x = lower_of_moved<0x143, 0xc>(x);
    return of_lane(x, 63);
}

// Upper bound of one key: the best path that fits among all that go the cheapest way to some (l, s) under one multiplier
// and the cheapest way on under another, both of the GDP_BOUND_WINDOW around the one whose bound is the best.  Where all
// layers are alike every layer changes its strategy at the same multiplier, and only such a splice comes near the
// budget.  grid (256-element groups of the largest table, keys, instances); a (l, s) per thread.
// Against splices of 4 whole paths the bound leaves half to a fifth of the labels (L = 80, S = 64 68 -> 43 per layer, 30 layers
// of two kinds that trade memory for time 738 -> 261) in the same 6 us.
__global__ __launch_bounds__(256) void gdp_bound_upper_kernel(const GdpBoundInst *inst, int n_lam)
{
    constexpr int W = GDP_BOUND_WINDOW;
    __shared__ double red[4];
    const GdpBoundInst &I = inst[blockIdx.z];
    const int key = (int)blockIdx.y, t = (int)threadIdx.x, lane = t & 63, LS = I.L * I.S;
    if (key >= I.K || (int)blockIdx.x * 256 >= LS) return;   // the whole workgroup
    const gdouble P = (gdouble)(uintptr_t)I.P, Q = (gdouble)(uintptr_t)I.Q, lams = (gdouble)(uintptr_t)I.lam, ends = (gdouble)(uintptr_t)I.end;
    const guint_in P_mem = (guint_in)(uintptr_t)I.P_mem, Q_mem = (guint_in)(uintptr_t)I.Q_mem;
    const int64_t B = ((const __attribute__((address_space(1))) int64_t *)(uintptr_t)I.budget)[key];
    // the best multiplier, every wave for itself
    double d = -INFINITY;
    int at_d = 0;
    for (int at = lane; at < n_lam; at += 64) {
        const double e = ends[at] - lams[at] * (double)B;
        if (e > d) {
            d = e;
            at_d = at;
        }
    }
    if (B < 0) return;   // the whole workgroup
    const double most = -lowest_of(-d);
    int best_at = n_lam;
    for (unsigned long long with = __builtin_amdgcn_ballot_w64(d == most); with; with &= with - 1)
        best_at = min(best_at, __builtin_amdgcn_readlane(at_d, __builtin_ctzll(with)));
    const int first = max(0, min(best_at - W / 2, n_lam - W));
    if (blockIdx.x == 0 && t == 0) I.best[key] = best_at;
    const int e = min((int)blockIdx.x * 256 + t, LS - 1);
    double p[W], q[W], lam[W];
    uint32_t pm[W], qm[W];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const size_t at = (size_t)(first + i) * LS + e;
        p[i] = P[at];
        q[i] = Q[at];
        pm[i] = P_mem[at];
        qm[i] = Q_mem[at];
        lam[i] = lams[first + i];
    }
    double best = INFINITY;
#pragma unroll
    for (int i = 0; i < W; ++i) {
        p[i] -= lam[i] * (double)pm[i];
        q[i] -= lam[i] * (double)qm[i];
    }
#pragma unroll
    for (int i = 0; i < W; ++i)
#pragma unroll
        for (int j = 0; j < W; ++j)
            if ((int64_t)(pm[i] + qm[j]) <= B) best = fmin(best, p[i] + q[j]);
    best = lowest_of(best);
    if (lane == 0) red[t >> 6] = best;
    __syncthreads();
    if (t != 0) return;
    best = fmin(fmin(red[0], red[1]), fmin(red[2], red[3]));
    if (best < GDP_BOUND_FAR / 2) atomicMin(I.ub + key, ordered(best + gdp_bound_margin(I.L, I.V, I.magnitude, lam[W - 1])));
}

// What stays: (l, s) is out when for every key some multiplier's bound lies above that key's upper bound.  The
// margin covers the rounding of the bound; that of the upper bound is part of it, and that of the DP's own sums is less
// than either.
// grid (ROWS times 64 strategies of a layer, instances), PARTS waves for each with 8 multipliers at a time.  What takes
// the time is the round trips of the loads: with 8 waves all 64 multipliers of an element are asked for at once (L = 80,
// S = 64 26.8 -> 6.3 us, L = 48, S = 88 25.0 -> 5.7 us).  A batch that fills the device with one wave per 64 elements
// hides them by itself and would only start more waves, and what it does wait for is the start of its workgroups, so that one has
// 4 layers (256 instances of S = 44 44 us with a layer each, 32 with 4).
template <int PARTS, int ROWS>
__global__ __launch_bounds__(64 * PARTS * ROWS) void gdp_bound_keep_kernel(const GdpBoundInst *inst, int n_lam)
{
    static_assert(PARTS == 1 || ROWS == 1, "waves that meet at the barrier all get there");
    __shared__ unsigned left[PARTS][64];
    const GdpBoundInst &I = inst[blockIdx.y];
    const int L = I.L, S = I.S, LS = L * S, K = I.K, lane = (int)threadIdx.x & 63, part = PARTS == 1 ? 0 : (int)threadIdx.x >> 6;
    const int halves = (S + 63) / 64, row = (int)blockIdx.x * ROWS + (ROWS == 1 ? 0 : (int)threadIdx.x >> 6), l = row / halves, half = row - l * halves,
              s = 64 * half + lane;
    if (l >= L) return;   // the whole workgroup, or a wave that meets no other
    const int at = l * S + min(s, S - 1);
    // the keys: a lane each asks for what is known of it, all at once
    const int own = min(lane, K - 1);
    const int64_t own_budget = ((const __attribute__((address_space(1))) int64_t *)(uintptr_t)I.budget)[own];
    const unsigned long long own_ub = ((const __attribute__((address_space(1))) unsigned long long *)(uintptr_t)I.ub)[own];
    const int V = I.V;
    const double magnitude = I.magnitude;
    const gdouble P = (gdouble)(uintptr_t)I.P, Q = (gdouble)(uintptr_t)I.Q, lams = (gdouble)(uintptr_t)I.lam;
    const gulong marks = (gulong)(uintptr_t)I.marks;   // (here: behind a store the compiler would fetch it again)
    __attribute__((address_space(1))) uint8_t *const keep = (__attribute__((address_space(1))) uint8_t *)(uintptr_t)I.keep;
    unsigned alive = (1u << K) - 1;
    double ub[GDP_BOUND_MAX_KEY], budget[GDP_BOUND_MAX_KEY];
    for (int i0 = 8 * part; i0 < n_lam; i0 += 8 * PARTS) {
        double p[8], q[8], lam[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {   // beyond the last: the last once more
            const size_t row = (size_t)min(i0 + i, n_lam - 1) * LS + at;
            p[i] = P[row];
            q[i] = Q[row];
            lam[i] = lams[min(i0 + i, n_lam - 1)];
        }
        if (i0 == 8 * part) {
            const double as_double = (double)own_budget, bound = own_budget >= 0 ? gdp_unordered(own_ub) : -INFINITY;   // (no solution: nothing stays)
#pragma unroll
            for (int k = 0; k < GDP_BOUND_MAX_KEY; ++k) {
                budget[k] = of_lane(as_double, k);
                ub[k] = of_lane(bound, k);
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const double r = p[i] + q[i];
            const double margin = gdp_bound_margin(L, V, magnitude, lam[i]);
#pragma unroll
            for (int k = 0; k < GDP_BOUND_MAX_KEY; ++k)
                if (k < K && r - lam[i] * budget[k] > ub[k] + margin) alive &= ~(1u << k);
        }
    }
    if constexpr (PARTS > 1) {
        left[part][lane] = alive;
        __syncthreads();
        if (part != 0) return;
#pragma unroll
        for (int w = 1; w < PARTS; ++w) alive &= left[w][lane];
    }
    if (s < S) keep[at] = (uint8_t)alive;
    else alive = 0;
    for (int k = 0; k < K; ++k) {
        const unsigned long long these = __builtin_amdgcn_ballot_w64(alive >> k & 1);
        const gulong mark = marks + 2 * ((size_t)k * L + l);
        if (lane == 0) mark[half] = these;
        if (lane == 0 && halves == 1) mark[1] = 0;
    }
}

}  // namespace

bool bounds::has_form(const gdp_problem *q)
{
    constexpr uint32_t whole = GDP_EXPORT_F | GDP_EXPORT_MARK | GDP_COMPUTE_ALL | GDP_KEEP_MARKS | GDP_LAUNCH_FUSED | GDP_LAUNCH_PER_LAYER;
    return !(q->flags & whole) && q->L >= 2 && q->L <= GDP_BOUND_MAX_L && q->S >= 2 && q->S <= GDP_BOUND_MAX_S &&
           q->n_key >= 1 && q->n_key <= GDP_BOUND_MAX_KEY && q->L * q->S <= GDP_BOUND_MAX_LS;
}

bool bounds::allowed(bool *forced)
{
    const char *env = getenv("GALVATRON_DP_REDUCE"), *skip = getenv("GALVATRON_DP_SKIP");
    *forced = env && *env && atoi(env) != 0;
    return !(env && *env && !*forced) && !(skip && *skip && atoi(skip) == 0);
}

double bounds::undominated(const gdp_problem *q, int layer)
{
    const int32_t *const mem = q->mem + (size_t)layer * q->S;
    const double *const time = q->intra + (size_t)layer * q->S;
    int16_t order[GDP_MAX_S];
    for (int s = 0; s < q->S; ++s) order[s] = (int16_t)s;
    std::sort(order, order + q->S, [&](int a, int b) { return mem[a] != mem[b] ? mem[a] < mem[b] : time[a] < time[b]; });   // allocates nothing
    double least = INFINITY;
    int stay = 0;
    for (int i = 0; i < q->S && mem[order[i]] < q->V; ++i) {
        stay += time[order[i]] < least;
        least = fmin(least, time[order[i]]);
    }
    return (double)stay / q->S;
}

double bounds::undominated(const gdp_problem *q)
{
    const int m = q->L < 4 ? q->L : 4;
    const size_t S = (size_t)q->S;
    double share = 0, last = 0;
    for (int k = 0, before = -1; k < m; ++k) {
        const int l = (int)((int64_t)q->L * (2 * k + 1) / (2 * m));
        if (before < 0 || memcmp(q->mem + l * S, q->mem + before * S, sizeof(int32_t) * S) != 0 || memcmp(q->intra + l * S, q->intra + before * S, sizeof(double) * S) != 0)
            last = undominated(q, l);
        share += last;
        before = l;
    }
    return share / m;
}

// Twice as many leave fewer labels where those are many, which the undominated strategies of all layers tell best, and take 3 us longer (a
// wave of passes on every compute unit instead of every second).  110 calls of random inputs, us with 64 / 128: up to 250 of these strategies 64 is as fast or up to
// 4 us faster; above 183 / 172, 190 / 153, 228 / 140, 235 / 219, 351 / 269, 1263 / 424.  256 are slower in nearly all.
int bounds::key_multipliers(const gdp_problem *q, double undominated)
{
    constexpr double MANY = 250;
    return undominated * q->S * q->L <= MANY ? 64 : GDP_BOUND_MAX_LAM;
}

void bounds::multipliers(const gdp_problem *q, int n_lam, double *lam)
{
    double t0 = INFINITY, t1 = -INFINITY, m0 = INFINITY, m1 = 0;
    for (size_t k = 0; k < (size_t)q->L * q->S; ++k) {
        if (q->mem[k] >= q->V || !(q->intra[k] < INFINITY)) continue;
        t0 = fmin(t0, q->intra[k]);
        t1 = fmax(t1, q->intra[k]);
        m0 = fmin(m0, (double)q->mem[k]);
        m1 = fmax(m1, (double)q->mem[k]);
    }
    const double range = t1 > t0 ? t1 - t0 : 1.0, base = range / fmax(1.0, m1 - m0);
    lam[0] = 0.0;
    for (int i = 1; i < n_lam; ++i) lam[i] = base * exp2(-6.0 + 12.0 * (i - 1) / (n_lam - 2));
}

hipError_t bounds::lay_out(const Inputs &in, int max_S, hipStream_t stream)
{
    const int bands = (max_S + 15) / 16, n_head = in.head ? (int)(in.head_bytes / 16) : 0;
    if (n_head == 0 && in.n_matrices == 0) return hipSuccess;
    gdp_bound_transpose_kernel<<<(unsigned)((n_head + HEAD - 1) / HEAD + in.n_matrices * bands), 256, 0, stream>>>(
        in.matrices, bands, static_cast<const uint4v *>(in.head), static_cast<uint4v *>(in.head_to), n_head);
    return hipGetLastError();
}

hipError_t bounds::launch(const GdpBoundInst *inst, int n, int n_lam, int max_LS, int max_rows, int max_S, int max_K, bool held, hipStream_t stream)
{
    const dim3 grid(2u * (unsigned)n_lam, (unsigned)n);
    const unsigned threads = 64u * (unsigned)((max_S + TARGETS - 1) / TARGETS);
#define GDP_PASS(E, AHEAD) \
    if (max_S <= PARTS * E && held) gdp_bound_pass_kernel<E, 4, true><<<grid, threads, 0, stream>>>(inst); \
    else if (max_S <= PARTS * E) gdp_bound_pass_kernel<E, AHEAD, false><<<grid, threads, 0, stream>>>(inst)
    GDP_PASS(4, 4);
    else GDP_PASS(6, 4);
    else GDP_PASS(8, 4);
    else GDP_PASS(10, 4);
    else GDP_PASS(12, 4);
    else GDP_PASS(16, 4);
    else GDP_PASS(22, 2);
    else GDP_PASS(32, 2);
#undef GDP_PASS
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    gdp_bound_upper_kernel<<<dim3((unsigned)((max_LS + 255) / 256), (unsigned)max_K, (unsigned)n), 256, 0, stream>>>(inst, n_lam);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    if ((int64_t)max_rows * n <= 1024)   // 8 waves of each are on the device at a time
        gdp_bound_keep_kernel<8, 1><<<dim3((unsigned)max_rows, (unsigned)n), 512, 0, stream>>>(inst, n_lam);
    else
        gdp_bound_keep_kernel<1, 4><<<dim3((unsigned)(max_rows + 3) / 4, (unsigned)n), 256, 0, stream>>>(inst, n_lam);
    return hipGetLastError();
}
