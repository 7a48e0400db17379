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

namespace {

static_assert(GDP_BOUND_MAX_S <= 128, "the cheapest end of a path: two strategies per lane");
static_assert(GDP_BOUND_MAX_LAM <= 64 && GDP_BOUND_LOW + 1 == 4, "the upper bounds: a multiplier per lane, a path per wave");

__device__ __forceinline__ double lagrangian(int32_t mem, double intra, double lam, int V)
{
    return mem < V && intra < INFINITY ? intra + lam * (double)mem : (double)INFINITY;
}

// inter_t: grid (pairs, 16-row bands of the largest matrix), 256 threads; LDS turns the band around so that both
// sides are read and written along rows.
__global__ __launch_bounds__(256) void gdp_bound_transpose_kernel(const GdpBoundInst *inst, const int2 *pairs)
{
    __shared__ double tile[16][GDP_BOUND_MAX_S + 1];
    const int2 w = pairs[blockIdx.x];
    const GdpBoundInst &I = inst[w.x];
    const int S = I.S, r0 = (int)blockIdx.y * 16;
    if (r0 >= S) return;
    const int rows = S - r0 < 16 ? S - r0 : 16;
    const double *src = I.inter + (size_t)w.y * S * S;
    double *dst = const_cast<double *>(I.inter_t) + (size_t)w.y * S * S;
    for (int e = threadIdx.x; e < rows * S; e += 256) tile[e / S][e % S] = src[(size_t)r0 * S + e];
    __syncthreads();
    for (int e = threadIdx.x; e < rows * S; e += 256) {
        const int c = e / rows, r = e % rows;
        dst[(size_t)c * S + r0 + r] = tile[r][c];
    }
}

// One pass over the layers of one instance under one multiplier: forwards (P, the path and its cost) or backwards
// (Q).  grid (2 * multipliers, instances): the serial chain of L steps is what takes the time, so everything that
// does not depend on it runs side by side -- multipliers and directions in workgroups of their own, a step's S*S
// candidates on up to 1024 threads (thread = target strategy + S * part, its sources part, part + G, ...: loads run
// along the rows), and the matrices of the next two steps are on their way to registers meanwhile.  A step is then two
// barriers and the reduction over the parts: L = 80, S = 64 207 -> 132 us, L = 48, S = 88 147 -> 102 us and L = 32,
// S = 44 79 -> 50 us against loads one step ahead behind comparisons.
template <int E, int NT>
__global__ __launch_bounds__(NT, NT == GDP_BOUND_THREADS ? 4 : 8) void gdp_bound_pass_kernel(const GdpBoundInst *inst)
{
    extern __shared__ uint8_t arg_of[];   // [L][S], forwards only
    __shared__ double X[GDP_BOUND_MAX_S], part_v[GDP_BOUND_THREADS];
    __shared__ uint8_t part_i[GDP_BOUND_THREADS];
    __shared__ int32_t mat[GDP_BOUND_MAX_L];
    __shared__ uint8_t path[GDP_BOUND_MAX_L];
    const GdpBoundInst &I = inst[blockIdx.y];
    const int L = I.L, S = I.S, V = I.V, t = (int)threadIdx.x, li = (int)blockIdx.x >> 1;
    const bool back = blockIdx.x & 1u;
    const double lam = I.lam[li];
    const int G = min(NT / S, GDP_BOUND_PARTS), s = t % S, g = min(t / S, G - 1), c_at = min(t, S - 1);
    const size_t SS = (size_t)S * S;
    for (int l = t; l < L; l += NT) mat[l] = I.index[l];
    if (t < S) X[t] = 0.0;
    __syncthreads();
    // Global memory, said so: the compiler takes a pointer that comes from memory for one that may point anywhere.
    typedef const __attribute__((address_space(1))) double *gdouble;
    typedef const __attribute__((address_space(1))) int32_t *gint;
    typedef __attribute__((address_space(1))) double *gout;
    const gdouble tables = (gdouble)(uintptr_t)(back ? I.inter_t : I.inter), intra = (gdouble)(uintptr_t)I.intra;
    const gint mem = (gint)(uintptr_t)I.mem;
    const gout out = (gout)(uintptr_t)((back ? I.Q : I.P) + (size_t)li * L * S);

    // What a step needs from memory: its part of the matrix and the layer's costs of strategy t.  Sources beyond the last
    // are the last once more, so that nothing here depends on a comparison and the loads of a step leave together.
    struct Inputs {
        double m[E], intra;
        int32_t mem;
    };
    auto from = [&](int k) { return min(g + k * G, S - 1); };
    constexpr int AHEAD = E <= 8 ? 2 : 1;   // steps: two sets of 16 elements do not fit the registers of 1024 threads
    auto fetch = [&](int l, Inputs &in) {
        const gdouble M = tables + (size_t)__builtin_amdgcn_readfirstlane(mat[l]) * SS;
#pragma unroll
        for (int k = 0; k < E; ++k) in.m[k] = M[from(k) * S + s];
        in.mem = mem[l * S + c_at];
        in.intra = intra[l * S + c_at];
    };
    const int first = back ? L - 1 : 0, step = back ? -1 : 1;
    // Step i; its registers are filled again for step i + AHEAD as soon as they have been read.
    auto pass = [&](int i, Inputs &in) {
        const int l = first + i * step;
        const double c = lagrangian(in.mem, in.intra, lam, V);
        if (back) {
            // X is Q[l]; what lies before layer l sees the cost of (l, s) on top of it
            if (t < S) {
                out[(size_t)l * S + t] = X[t];
                X[t] += c;
            }
            if (l == 0) return;
            __syncthreads();
        }
        double best = INFINITY;
        int arg = 0;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const double v = X[from(k)] + in.m[k];
            arg = v < best ? from(k) : arg;
            best = v < best ? v : best;
        }
        if (i + AHEAD < L) fetch(l + AHEAD * step, in);
        if (t < G * S) {
            part_v[t] = best;
            part_i[t] = (uint8_t)arg;
        }
        __syncthreads();
        if (t < S) {   // thread t is part 0 of target t
#pragma unroll 8
            for (int p = 1; p < G; ++p) {   // no branch: the reads of all parts are in flight together
                const double v = part_v[p * S + t];
                const int a = part_i[p * S + t];
                arg = v < best ? a : arg;
                best = v < best ? v : best;
            }
            if (back) {
                X[t] = best;
            } else {
                X[t] = best + c;
                out[(size_t)l * S + t] = X[t];
                arg_of[l * S + t] = (uint8_t)arg;
            }
        }
        __syncthreads();
    };
    Inputs in[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a)
        if (a < L) fetch(first + a * step, in[a]);
    for (int i = 0; i < L; i += AHEAD)
#pragma unroll
        for (int a = 0; a < AHEAD; ++a)
            if (i + a < L) pass(i + a, in[a]);
    if (back) return;
    if (t < 64) {   // the cheapest end: two strategies per lane at most, then across the wave
        int b = t < S ? t : 0;
        double least = X[b];
        if (t + 64 < S && X[t + 64] < least) {
            b = t + 64;
            least = X[b];
        }
#pragma unroll
        for (int w = 32; w > 0; w >>= 1) {
            const double v = __shfl_xor(least, w);
            const int a = __shfl_xor(b, w);
            if (v < least || (v == least && a < b)) {
                least = v;
                b = a;
            }
        }
        if (t == 0)
            for (int l = L - 1; l >= 0; --l) {
                path[l] = (uint8_t)b;
                b = arg_of[l * S + b];
            }
    }
    __syncthreads();
    // what the path costs: one layer per thread (L <= 512), summed in LDS
    double time = 0.0, memory = 0.0;
    if (t < L) {
        const int b = path[t], a = arg_of[t * S + b];
        I.path[(size_t)li * L + t] = (uint8_t)b;
        const int32_t m = mem[t * S + b];
        time = tables[(size_t)mat[t] * SS + (size_t)a * S + b] + (m < V ? intra[t * S + b] : (double)INFINITY);
        memory = (double)m;   // whole numbers below 2^41: exact
    }
    part_v[t] = time;
    __syncthreads();
    for (int w = NT / 2; w > 0; w >>= 1) {
        if (t < w) part_v[t] += part_v[t + w];
        __syncthreads();
    }
    if (t == 0) I.path_time[li] = part_v[0];
    __syncthreads();
    part_v[t] = memory;
    __syncthreads();
    for (int w = NT / 2; w > 0; w >>= 1) {
        if (t < w) part_v[t] += part_v[t + w];
        __syncthreads();
    }
    if (t == 0) I.path_mem[li] = (int64_t)part_v[0];
}

// Upper bound of one key: the best of the multipliers' paths that fit, and of the paths that follow one of the
// last paths that do not fit up to some layer and the first one that does from there on (or the other way round) --
// where all layers are alike every layer changes its strategy at the same multiplier, and only such a
// splice comes near the budget.  grid (keys, instances), 256 threads; a candidate per thread from running sums.  Choosing
// the paths and summing them up are a wave's work instead of one thread's walk through memory (L = 80, S = 64 11.5 ->
// 7.0 us, 256 instances of S = 44 8.4 -> 6.9 us).
__global__ __launch_bounds__(256) void gdp_bound_upper_kernel(const GdpBoundInst *inst, int n_lam)
{
    __shared__ double pt[GDP_BOUND_LOW + 1][GDP_BOUND_MAX_L + 1], pm[GDP_BOUND_LOW + 1][GDP_BOUND_MAX_L + 1];
    __shared__ uint8_t st[GDP_BOUND_LOW + 1][GDP_BOUND_MAX_L];
    __shared__ double red[256];
    __shared__ int which[GDP_BOUND_LOW + 1];
    const GdpBoundInst &I = inst[blockIdx.y];
    const int key = (int)blockIdx.x, t = (int)threadIdx.x, L = I.L, S = I.S;
    if (key >= I.K) return;
    const int64_t B = I.budget[key];
    const size_t SS = (size_t)S * S;
    double best = INFINITY;
    if (t < 64) {   // a multiplier per lane: which paths fit, and which there are, are two ballots
        const double time = t < n_lam ? I.path_time[t] : (double)INFINITY;
        const bool fits = time < INFINITY && I.path_mem[t] <= B;
        if (fits) best = time;
        const unsigned long long fit = __ballot(fits), any = __ballot(time < INFINITY);
        if (t <= GDP_BOUND_LOW) {
            const int first = fit ? __ffsll(fit) - 1 : -1;
            unsigned long long below = first > 0 ? any & ((1ull << first) - 1) : 0;
            for (int q = 1; q < t && below; ++q) below ^= 1ull << (63 - __clzll(below));
            which[t] = t == 0 ? first : below ? 63 - __clzll(below) : -1;
        }
    }
    __syncthreads();
    if (which[0] >= 0 && which[1] >= 0) {   // the same in every thread
        for (int e = t; e < (GDP_BOUND_LOW + 1) * L; e += 256) {
            const int q = e / L, l = e % L;
            if (which[q] < 0) continue;
            const uint8_t *p = I.path + (size_t)which[q] * L;
            const int b = p[l];
            st[q][l] = (uint8_t)b;
            // the first layer comes from whatever strategy is cheapest: P under lam[0] = 0 is that plus its own cost
            const double x = l == 0 ? I.P[b]
                                    : I.inter[(size_t)I.index[l] * SS + (size_t)p[l - 1] * S + b] + I.intra[(size_t)l * S + b];
            pt[q][l + 1] = x;
            pm[q][l + 1] = (double)I.mem[(size_t)l * S + b];
        }
        __syncthreads();
        // running sums: a path per wave, 64 layers at a time (their rounding, in whatever order, is within the margin)
        const int q = t >> 6, lane = t & 63;
        if (which[q] >= 0) {
            double time = 0.0, memory = 0.0;   // of the layers before the 64
            if (lane == 0) pt[q][0] = pm[q][0] = 0.0;
            for (int l0 = 1; l0 <= L; l0 += 64) {
                const int l = l0 + lane;
                double x = l <= L ? pt[q][l] : 0.0, y = l <= L ? pm[q][l] : 0.0;
#pragma unroll
                for (int w = 1; w < 64; w <<= 1) {
                    const double u = __shfl_up(x, w), v = __shfl_up(y, w);
                    if (lane >= w) {
                        x += u;
                        y += v;
                    }
                }
                x += time;
                y += memory;
                if (l <= L) {
                    pt[q][l] = x;
                    pm[q][l] = y;
                }
                time = __shfl(x, 63);
                memory = __shfl(y, 63);
            }
        }
        __syncthreads();
        for (int e = t; e < 2 * GDP_BOUND_LOW * (L - 1); e += 256) {
            const int c = 1 + e % (L - 1), d = e / (L - 1), q = 1 + (d >> 1);
            if (which[q] < 0) continue;
            const int a = d & 1 ? 0 : q, b = d & 1 ? q : 0;   // a up to layer c, then b
            if (pm[a][c] + (pm[b][L] - pm[b][c]) > (double)B) continue;
            const double *M = I.inter + (size_t)I.index[c] * SS;
            const double turn = M[(size_t)st[a][c - 1] * S + st[b][c]], was = M[(size_t)st[b][c - 1] * S + st[b][c]];
            const double x = pt[a][c] + (pt[b][L] - pt[b][c]) + (turn - was);
            if (x < best) best = x;
        }
    }
    red[t] = best;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w && red[t + w] < red[t]) red[t] = red[t + w];
        __syncthreads();
    }
    if (t == 0) I.ub[key] = red[0];
}

// What stays: (l, s) is out when for every key some multiplier's bound lies above that key's upper bound.  The
// margin covers the rounding of the bound, of the upper bound and of the DP's own sums: each is a sum of at most
// 4 L + 4 terms whose magnitudes add up to no more than `magnitude` + lam * (L + 1) * V.
// grid (64-element groups of the largest table, instances), PARTS waves with 8 multipliers at a time each.  What takes
// the time is the round trips of the loads: with 8 waves all 64 multipliers of an element are asked for at once (L = 80,
// S = 64 26.8 -> 6.3 us, L = 48, S = 88 25.0 -> 5.7 us).  A batch that fills the device with one wave per 64 elements
// hides them by itself and would only start more waves (256 instances of S = 44 23.6 us with 1 wave, 40 with 8).
template <int PARTS>
__global__ __launch_bounds__(64 * PARTS) void gdp_bound_keep_kernel(const GdpBoundInst *inst, int n_lam)
{
    __shared__ unsigned left[PARTS][64];
    const GdpBoundInst &I = inst[blockIdx.y];
    const int LS = I.L * I.S, K = I.K, lane = (int)threadIdx.x & 63, part = (int)threadIdx.x >> 6;
    if ((int)blockIdx.x * 64 >= LS) return;   // the whole workgroup
    const int e = (int)blockIdx.x * 64 + lane, at = min(e, LS - 1);
    unsigned alive = 0;
    double ub[GDP_BOUND_MAX_KEY], budget[GDP_BOUND_MAX_KEY];
#pragma unroll
    for (int k = 0; k < GDP_BOUND_MAX_KEY; ++k) {
        ub[k] = INFINITY;
        budget[k] = 0.0;
        if (k < K && I.budget[k] >= 0) {
            alive |= 1u << k;
            ub[k] = I.ub[k];
            budget[k] = (double)I.budget[k];
        }
    }
    typedef const __attribute__((address_space(1))) double *gdouble;
    const gdouble P = (gdouble)(uintptr_t)I.P, Q = (gdouble)(uintptr_t)I.Q, lams = (gdouble)(uintptr_t)I.lam;
    const double reach = (double)(I.L + 1) * (double)I.V, magnitude = I.magnitude;
    const double ulp = 16.0 * (double)(I.L + 4) * 0x1p-53;
    for (int i0 = 8 * part; i0 < n_lam; i0 += 8 * PARTS) {
        double p[8], q[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {   // beyond the last: the last once more
            const size_t row = (size_t)min(i0 + i, n_lam - 1) * LS + at;
            p[i] = P[row];
            q[i] = Q[row];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const double lam = lams[min(i0 + i, n_lam - 1)];
            const double r = p[i] + q[i];
            const double margin = ulp * (magnitude + lam * reach);
#pragma unroll
            for (int k = 0; k < GDP_BOUND_MAX_KEY; ++k)
                if (k < K && r - lam * budget[k] > ub[k] + margin) alive &= ~(1u << k);
        }
    }
    left[part][lane] = alive;
    __syncthreads();
    if (part != 0 || e >= LS) return;
#pragma unroll
    for (int w = 1; w < PARTS; ++w) alive &= left[w][lane];
    I.keep[e] = alive != 0;
}

}  // namespace

int gdp_bound_elements(int S, int threads)
{
    const int G = threads / S < GDP_BOUND_PARTS ? threads / S : GDP_BOUND_PARTS;
    const int most = threads == GDP_BOUND_THREADS ? 16 : 4;   // S <= 128: with 1024 threads G >= 8, so 16 are enough
    for (int e = 1; e <= most; e *= 2)
        if (e * G >= S) return e;
    return 0;
}

hipError_t gdp_launch_bounds(const GdpBoundInst *inst, int n, int n_lam, int max_LS, int max_S, int max_K,
                             int elements, int threads, const int2 *pairs, int n_pairs, hipStream_t stream)
{
    gdp_bound_transpose_kernel<<<dim3((unsigned)n_pairs, (unsigned)((max_S + 15) / 16)), 256, 0, stream>>>(inst, pairs);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 grid(2u * (unsigned)n_lam, (unsigned)n);
    const size_t lds = (size_t)max_LS;
    auto launch = [&](auto kernel) { kernel<<<grid, threads, lds, stream>>>(inst); };
    constexpr int WIDE = GDP_BOUND_THREADS, HALF = GDP_BOUND_THREADS / 2;
    if (threads == WIDE) {
        switch (elements) {
        case 1: launch(gdp_bound_pass_kernel<1, WIDE>); break;
        case 2: launch(gdp_bound_pass_kernel<2, WIDE>); break;
        case 4: launch(gdp_bound_pass_kernel<4, WIDE>); break;
        case 8: launch(gdp_bound_pass_kernel<8, WIDE>); break;
        default: launch(gdp_bound_pass_kernel<16, WIDE>); break;
        }
    } else {
        switch (elements) {
        case 1: launch(gdp_bound_pass_kernel<1, HALF>); break;
        case 2: launch(gdp_bound_pass_kernel<2, HALF>); break;
        default: launch(gdp_bound_pass_kernel<4, HALF>); break;
        }
    }
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    gdp_bound_upper_kernel<<<dim3((unsigned)max_K, (unsigned)n), 256, 0, stream>>>(inst, n_lam);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    const dim3 elements64((unsigned)((max_LS + 63) / 64), (unsigned)n);
    if ((int64_t)elements64.x * n <= 1024)   // 8 waves of each are on the device at a time
        gdp_bound_keep_kernel<8><<<elements64, 512, 0, stream>>>(inst, n_lam);
    else
        gdp_bound_keep_kernel<1><<<elements64, 64, 0, stream>>>(inst, n_lam);
    return hipGetLastError();
}
