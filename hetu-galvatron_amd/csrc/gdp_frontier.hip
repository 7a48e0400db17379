// The DP over what the bounds leave, without the budget axis.
//
// f[l][v][s] changes only at a few budgets v: its steps are labels (w, c) -- from w bins on the cost is c -- and a layer's
// labels follow from those of the layer before: a label (w, c) of strategy s' gives (w + mem[s], (c + inter[s'][s]) +
// intra[s]) for strategy s, of which those stay that are cheaper than every one that needs no more memory.  The same
// additions in the same order as in the dense recurrence: rounding is monotone, so that the minimum over the labels up to
// v is f[l][v][s] bit for bit.  Of these, the ones stay that can be part of a best path: c plus a lower bound on every way
// on that fits the budget does not exceed the upper bound of some key (gdp_bounds.hip).  What is dropped is on no best path
// and ties with none, so the walk back finds in every cell of a best path the candidates that tie for it, lowest strategy
// first, as in the dense table.
//
// Of random costs 1 to 200 labels per layer stay whatever the budget (L = 80, S = 64, V = 131072: 40, against 8.4 million
// cells), of identical layers that trade memory for time up to a few thousand.  An instance is one workgroup: its labels
// and what it needs of the next layer live in LDS, its layers follow each other at the price of two barriers.  An instance
// with more labels than fit says so, and is solved as a smaller instance of the dense recurrence.
#include "gdp_bounds.h"
#include "gdp_label_ops.h"

#include <math.h>

namespace {

constexpr int WORKERS = 8, FETCHERS = 4, THREADS = 64 * (WORKERS + FETCHERS);   // waves
constexpr int LABELS = 1536;    // of a layer
constexpr int KEPT = 64;        // strategies of a layer
constexpr int TURNS = 1024;     // transitions between the strategies of two layers
constexpr int WINDOW = 4;       // multipliers per key that labels are held against (with 64 in place of 4 a tenth fewer stay)
constexpr int LINES = 1152;     // doubles: what a layer's strategies are held against, and their costs
// of the walk back: labels, transitions and strategies of the layers that lie in LDS together
constexpr int BACK_LABELS = 4096, BACK_TURNS = 4800, BACK_KEPT = 1024;
static_assert(BACK_LABELS >= LABELS && BACK_TURNS >= TURNS && BACK_KEPT >= KEPT, "a layer fits");
static_assert(WORKERS >= GDP_BOUND_MAX_KEY, "the walk back: a wave per key");

// Keys are whole numbers below 2^53: a double is compared as fast as 32 bits are.
constexpr double KEY_W = 0x1p17, KEY_S = 0x1p11;
static_assert(KEPT <= 64 && LABELS <= 2048, "6 bits and 11");
constexpr int KEY_PAD = 72;   // 8 lanes look at 8 keys at a time each
constexpr int BUCKETS = 64 * WORKERS;
constexpr int SORTED_FROM = 192;   // labels of a layer; 3 more barriers and 7 reads in a row take as long as looking at that many keys

struct Forward {
    Label label[LABELS];
    __align__(16) double lines[2][LINES], turns[2][TURNS];
    // Of the labels as they are found: w, strategy, number within the strategy in one; +inf behind the last.  Of this layer
    // and the next.
    __align__(16) double key[2][LABELS + KEY_PAD];
    double cost[LABELS];
    // where the labels are many: keys by bucket, labels of a bucket and before it, of 64 buckets
    double sorted[LABELS];
    int32_t bucket[BUCKETS], bucket_at[BUCKETS];
    __align__(16) int32_t buckets_of[WORKERS];
};


struct Backward {
    Label label[BACK_LABELS];
    double turns[BACK_TURNS], intra[BACK_KEPT];
    int32_t mem[BACK_KEPT];
};

struct Shared {
    union {
        Forward f;
        Backward b;
        uint8_t keep[GDP_BOUND_MAX_LS];
    };
    // Per layer: strategies that stay, where their list begins, where the transitions into them begin in memory.  One
    // more at the end for the sums.
    int4 layer[GDP_BOUND_MAX_L + 1];
    double lam[GDP_BOUND_MAX_KEY][WINDOW], shift[GDP_BOUND_MAX_KEY][WINDOW], ub[GDP_BOUND_MAX_KEY];
    int32_t found[3];                    // labels of a layer, of the next one and the one after that
    int32_t labels_at[GDP_BOUND_MAX_L + 1];
    int32_t mat[GDP_BOUND_MAX_L];
    int32_t window[GDP_BOUND_MAX_KEY], budget[GDP_BOUND_MAX_KEY];
    int32_t lost;
    uint8_t kept[GDP_FRONTIER_KEPT];
};
static_assert(sizeof(Shared) <= 160 * 1024, "LDS of a compute unit");

// What a wave has on its way from memory for a later layer: transitions, what labels are held against, costs.
template <int LINE>
struct Ahead {
    static constexpr int T = TURNS / 64, N = LINES / 64;
    double turns[T], lines[N];
};

// grid (instances).  What a layer takes is latency, so the chain of a layer is kept short: 8 waves take the labels of a
// strategy each, 64 at a time, and find their order in the next layer by searches in LDS; 4 others in turn have what the
// next 4 layers need of the matrices on its way and lay it out in LDS, and all meet twice per layer.  KEYS: as many at
// least.
// A dependent instruction takes 9 clocks, a read from LDS 64, a barrier 30, so a layer of few labels is 0.9 us, one of 270
// labels and 8 strategies 9.  Against the smaller instance of the dense recurrence that the host made of what stays (kernels,
// without the host's 0.05 to 0.9 ms between them): L = 80, S = 64 311 -> 216 to 255 us by input, L = 48, S = 88 405 -> 90 to 124,
// 256 instances of S = 44 1690 -> 118, 15 stages of a fit 435 -> 217 to 260.
template <int KEYS>
__global__ __launch_bounds__(THREADS) void gdp_frontier_kernel(const GdpBoundInst *inst)
{
    constexpr int LINE = KEYS * WINDOW + 2;   // of a strategy: lines, intra, memory
    // Keys whose lines, and whose multipliers, are held in registers; the others' are read from LDS.  All where there is room for
    // them: no kernel here may need scratch memory, which the runtime would have to obtain for the launch, and gdp_solve_static
    // promises that nothing is obtained.  (8 keys with all of them held took 252 bytes a lane and longer: L = 80, S = 64 408 -> 377 us;
    // 5 keys with two lines held 12 to 16 bytes, 522 -> 517 us; since each key has a status of its own one held is too many by 12: 80
    // static calls of 5 keys 12.06 ms, 12.00 with it.)
    constexpr int LINES_HELD = KEYS <= 4 ? KEYS : KEYS == 5 ? 0 : 2, KEYS_HELD = KEYS <= 5 ? KEYS : 0;
    extern __shared__ __align__(16) char lds[];
    Shared &sh = *reinterpret_cast<Shared *>(lds);
    const GdpBoundInst &I = inst[blockIdx.x];
    const int L = uniform(I.L), S = uniform(I.S), K = uniform(I.K), LS = L * S;
    const int t = (int)threadIdx.x, lane = t & 63, wave = uniform(t >> 6);
    GdpFrontierOut *const out = I.out;
    auto give_up = [&](int why) {   // by the whole workgroup
        if (t < K) out->status[t] = why;
    };

    // ---- what stays, as lists; the keys ----
    const gbyte keep = GLOBAL(gbyte, I.keep);
    for (int e = t; e < LS; e += THREADS) sh.keep[e] = keep[e];
    for (int l = t; l < L; l += THREADS) sh.mat[l] = GLOBAL(gint, I.index)[l];
    if (t == 0) sh.lost = 0;
    if (t < 3) sh.found[t] = 0;
    __syncthreads();
    if (t < GDP_BOUND_MAX_KEY) {
        const bool there = t < K;
        const int64_t B = there ? GLOBAL(const __attribute__((address_space(1))) int64_t *, I.budget)[t] : -1;
        const unsigned long long o = there ? GLOBAL(const __attribute__((address_space(1))) unsigned long long *, I.ub)[t] : 0;
        sh.budget[t] = (int32_t)B;   // a start row; negative: none
        sh.ub[t] = gdp_unordered(o);
        const int first = B < 0 ? 0 : max(0, min(GLOBAL(gint, I.best)[t] - GDP_BOUND_WINDOW / 2, I.n_lam - GDP_BOUND_WINDOW)) + (GDP_BOUND_WINDOW - WINDOW) / 2;
        sh.window[t] = first;
        for (int i = 0; i < WINDOW; ++i) {
            const double lam = GLOBAL(gdouble, I.lam)[first + i];
            sh.lam[t][i] = lam;
            sh.shift[t][i] = lam * (double)B + gdp_bound_margin(I.L, I.V, I.magnitude, lam);
        }
        if (B >= 0 && o == ~0ull) sh.lost = 1;   // no path was found for it
    }
    __syncthreads();
    if (sh.lost) {
        give_up(1);
        return;
    }
    auto kept_of = [&](int l, unsigned long long &lo, unsigned long long &hi) {
        const bool a = lane < S && sh.keep[l * S + min(lane, S - 1)], b = lane + 64 < S && sh.keep[l * S + min(lane + 64, S - 1)];
        lo = __builtin_amdgcn_ballot_w64(a);
        hi = __builtin_amdgcn_ballot_w64(b);
    };
    for (int l = wave; l < L; l += WORKERS + FETCHERS) {
        unsigned long long lo, hi;
        kept_of(l, lo, hi);
        if (lane == 0) sh.layer[l].x = __popcll(lo) + __popcll(hi);
    }
    __syncthreads();
    if (wave == 0) {   // running sums of the numbers and of the transitions, and whether every layer fits
        int sum = 0, turns = 0, bad = 0, before = 0;
        for (int l0 = 0; l0 < L; l0 += 64) {
            const int l = l0 + lane;
            const int n = l < L ? sh.layer[l].x : 0, up = __shfl_up(n, 1), prev = lane ? up : before;
            int x = n, y = n * prev;   // none into the first layer
            bad |= l < L && (n < 1 || n > KEPT || n * LINE > LINES || y > TURNS);
            before = __shfl(n, 63);
            const int own = y;
#pragma unroll
            for (int w = 1; w < 64; w <<= 1) {
                const int x2 = __shfl_up(x, w), y2 = __shfl_up(y, w);
                if (lane >= w) {
                    x += x2;
                    y += y2;
                }
            }
            if (l < L) sh.layer[l] = make_int4(n, sum + x - n, turns + y - own, 0);
            sum += __shfl(x, 63);
            turns += __shfl(y, 63);
        }
        if (lane == 0) sh.layer[L] = make_int4(0, sum, turns, 0);
        if (__builtin_amdgcn_ballot_w64(bad != 0) != 0 || sum > GDP_FRONTIER_KEPT || turns > I.n_hist_turns) sh.lost = 1;
    }
    __syncthreads();
    if (sh.lost) {
        give_up(2);
        return;
    }
    for (int l = wave; l < L; l += WORKERS + FETCHERS) {
        unsigned long long lo, hi;
        kept_of(l, lo, hi);
        const unsigned long long below = (1ull << lane) - 1;
        const int at = sh.layer[l].y;
        if (lo >> lane & 1) sh.kept[at + __popcll(lo & below)] = (uint8_t)lane;
        if (hi >> lane & 1) sh.kept[at + __popcll(lo) + __popcll(hi & below)] = (uint8_t)(lane + 64);
    }
    __syncthreads();   // the marks themselves are not read any more
    if (t == 0) sh.labels_at[0] = 0;
    for (int e = t; e < 2 * (LABELS + KEY_PAD); e += THREADS) sh.f.key[0][e] = INFINITY;   // both
    for (int e = t; e < BUCKETS; e += THREADS) sh.f.bucket[e] = 0;
    __syncthreads();

    const gdouble inter = GLOBAL(gdouble, I.inter_f), intra = GLOBAL(gdouble, I.intra), Q = GLOBAL(gdouble, I.Q);
    const gint mem = GLOBAL(gint, I.mem);
    const giout hist_mem = GLOBAL(giout, I.hist_mem);
    const gout hist_turns = GLOBAL(gout, I.hist_turns), hist_intra = GLOBAL(gout, I.hist_intra);
    const glabel hist = GLOBAL(glabel, I.hist);
    const int n_hist = uniform(I.n_hist);
    const double limit = uniform(I.limit);
    // What a layer takes, in ns: its barriers, the order of many labels, and a wave's turns of 128 labels for every 8th strategy.
    // An instance whose other layers would take longer than the dense recurrence (`limit`) is left to that one; what its
    // labels have taken by then does not come back either way, so that only what is ahead counts.  Ahead, as from layer 2 on, in the
    // first half: of identical layers that trade memory for time the labels of a layer grow towards L / 2 about as they do
    // at the start, and are half of what that comes to in the mean.  In the second half they become fewer again.
    // (Static calls, 2000 inputs of L = 3 to 80, S = 5 to 44, ms in all: dense 521, by labels where they come through 335; 114 take more than 1.1
    // times what they take dense, mostly by the 80 us of bounds whose labels are left at layer 2 or 3, the worst two 1.6 and 2.1.  An account that counts what has been taken, too, and nothing ahead in the second half gives up as late as in the last layer.
    // Growth in the second half is no better guide: it takes layers of two kinds in turn for growing ones.)
    auto layer_ns = [](int n, int before) {
        return (before > SORTED_FROM ? 3000 : 900) + ((n + WORKERS - 1) / WORKERS) * ((before + 127) / 128) * (600 + 200 * KEYS);
    };
    auto hopeless = [&](int ns, int l, int n, int labels) {
        if (labels <= 64) return false;   // (less than a dense layer takes, and these tests lie in the chain)
        const int ahead = L - 1 - l;
        if ((double)ns * (double)ahead > limit * (double)(l + 1)) return true;
        if (l >= L / 2) return (double)ahead * layer_ns(n, labels / 2) > limit;
        if (l < max(2, L / 16)) return false;
        const int half = (l - 1) / 2, grown = labels - uniform(sh.labels_at[half + 1] - sh.labels_at[half]);
        const int top = labels + max(grown, 0) * (L / 2 - l) / (l - half);
        return top > 2 * LABELS || (double)ns + (double)(L - l) * layer_ns(n, top / 2) > 0.9 * limit;
    };

    if (wave >= WORKERS) {
        // ---- the waves that fetch: wave f what layers f, f + 4, ... need ----
        // e / n for e < 2^20 / n
        auto reciprocal = [](int n) { return ((1u << 20) + (unsigned)n - 1) / (unsigned)n; };
        auto quotient = [](int e, unsigned r) { return (int)((unsigned)e * r >> 20); };
        Ahead<LINE> a;
        auto fetch = [&](int l) {
            const int n = uniform(sh.layer[l].x), at = uniform(sh.layer[l].y);
            if (l > 0) {
                const int before = uniform(sh.layer[l - 1].y), all = n * uniform(sh.layer[l - 1].x);
                const unsigned r = reciprocal(n);
                const gdouble M = inter + (size_t)uniform(sh.mat[l]) * S * S;
#pragma unroll
                for (int i = 0; i < Ahead<LINE>::T; ++i) {
                    if (i * 64 >= all) break;
                    const int e = min(lane + i * 64, all - 1), from = quotient(e, r);
                    a.turns[i] = M[(uint32_t)(sh.kept[before + from] * S + sh.kept[at + e - from * n])];
                }
            }
            constexpr unsigned r = ((1u << 20) + LINE - 1) / LINE;
#pragma unroll
            for (int i = 0; i < Ahead<LINE>::N; ++i) {
                if (i * 64 >= n * LINE) break;
                const int e = min(lane + i * 64, n * LINE - 1), b = quotient(e, r), x = e - b * LINE, s = l * S + sh.kept[at + b];
                const int k = x / WINDOW, j = x % WINDOW;
                if (x < KEYS * WINDOW)
                    a.lines[i] = Q[(uint32_t)((sh.window[k] + j) * LS + s)];   // (nothing here waits for what it loads)
                else if (x == KEYS * WINDOW)
                    a.lines[i] = intra[(uint32_t)s];
                else
                    a.lines[i] = __builtin_bit_cast(double, int2v{mem[(uint32_t)s], 0});
            }
        };
        auto place = [&](int l) {
            const int n = uniform(sh.layer[l].x), at = uniform(sh.layer[l].y), to = l & 1;
            if (l > 0) {
                const int all = n * uniform(sh.layer[l - 1].x), turns_at = uniform(sh.layer[l].z);
#pragma unroll
                for (int i = 0; i < Ahead<LINE>::T; ++i) {
                    if (i * 64 >= all) break;
                    const int e = lane + i * 64;
                    if (e < all) {
                        sh.f.turns[to][e] = a.turns[i];
                        hist_turns[(uint32_t)(turns_at + e)] = a.turns[i];
                    }
                }
            }
            constexpr unsigned r = ((1u << 20) + LINE - 1) / LINE;
#pragma unroll
            for (int i = 0; i < Ahead<LINE>::N; ++i) {
                if (i * 64 >= n * LINE) break;
                const int e = lane + i * 64, b = quotient(e, r), x = e - b * LINE;
                if (e < n * LINE) {
                    sh.f.lines[to][e] = x < KEYS * WINDOW ? a.lines[i] - sh.shift[x / WINDOW][x % WINDOW] : a.lines[i];
                    if (x == KEYS * WINDOW) hist_intra[(uint32_t)(at + b)] = a.lines[i];
                    if (x > KEYS * WINDOW) hist_mem[(uint32_t)(at + b)] = __builtin_bit_cast(int2v, a.lines[i]).x;
                }
            }
        };
        const int f = wave - WORKERS;
        if (f < L) fetch(f);
        if (f == 0) {
            place(0);
            if (FETCHERS < L) fetch(FETCHERS);
        }
        __syncthreads();
        int at = 0, sum = 0;
        int ns = 0;
        for (int l = 0, slot = 0; l < L; ++l, slot = slot == 2 ? 0 : slot + 1) {   // the same barriers, and the same ways out, as the workers'
            const int n = uniform(sh.layer[l].x);
            ns += layer_ns(n, l ? sum : 1);
            if (sum > SORTED_FROM)
                for (int e = t - 64 * WORKERS; e < BUCKETS; e += 64 * FETCHERS) sh.f.bucket[e] = 0;
            for (int e = t - 64 * WORKERS; e < sum; e += 64 * FETCHERS) sh.f.key[(l + 1) & 1][e] = INFINITY;   // of the layer before
            if (l + 1 < L && (l + 1) % FETCHERS == f) place(l + 1);
            __syncthreads();
            sum = uniform(sh.found[slot]);
            if (sum == 0 || sum > LABELS || at + sum > n_hist || hopeless(ns, l, n, sum)) return;
            at += sum;
            if (l % FETCHERS == f && l > 0 && l + FETCHERS < L) fetch(l + FETCHERS);
            if (n > 1 && sum > SORTED_FROM) {
                __syncthreads();
                __syncthreads();
                __syncthreads();
            }
            if (n > 1) __syncthreads();
        }
    }

    // ---- forwards ----
    double executed = 0.0, total = INFINITY;
    int cell = 0;        // strategy of the cell, counted among those that stay
    int32_t v = -1;      // its budget
    bool walks = false;
    if (wave < WORKERS) {
        double lam[KEYS_HELD ? KEYS_HELD : 1][WINDOW], ub[KEYS_HELD ? KEYS_HELD : 1];
        int32_t budget[KEYS_HELD ? KEYS_HELD : 1];
#pragma unroll
        for (int k = 0; k < KEYS_HELD; ++k) {
#pragma unroll
            for (int i = 0; i < WINDOW; ++i) lam[k][i] = sh.lam[k][i];
            ub[k] = sh.ub[k];
            budget[k] = sh.budget[k];
        }
        int before = 1, at = 0, ns = 0;   // labels of the layer before, and where this layer's begin in memory
        // (before the first layer: one, no memory used, for each strategy the cheapest way in)
        __syncthreads();
        int4 here = sh.layer[0];
        for (int l = 0, slot = 0; l < L; ++l, slot = slot == 2 ? 0 : slot + 1) {
            const int now = l & 1, n = uniform(here.x), kept_at = uniform(here.y);
            here = sh.layer[l + 1];
            // what can still be part of a path that fits and is no worse than the best one known
            auto alive = [&](const double2 *line, const double2 *row, double c, int32_t w) {
                const double dw = (double)w;
                bool any = false;
#pragma unroll
                for (int k = 0; k < KEYS; ++k) {
                    const bool held = k < KEYS_HELD;
                    const double *const by = held ? lam[held ? k : 0] : sh.lam[k];
                    const double2 *const at = k < LINES_HELD ? line : row;
                    const double b0 = __builtin_fma(by[0], dw, at[2 * k].x), b1 = __builtin_fma(by[1], dw, at[2 * k].y),
                                 b2 = __builtin_fma(by[2], dw, at[2 * k + 1].x), b3 = __builtin_fma(by[3], dw, at[2 * k + 1].y);
                    const double bound = max_f64(max_f64(b0, b1), max_f64(b2, b3));
                    any |= (w <= (held ? budget[held ? k : 0] : sh.budget[k])) & (c + bound <= (held ? ub[held ? k : 0] : sh.ub[k]));
                }
                return any;
            };
            // Of labels that need the same memory the cheapest counts, with the last of them.  c: the least up to each label;
            // returns the least up to the last label that needs less than this one, `last` for the first ones of a turn, and
            // moves `last` on.
            auto step_from = [&](double c, bool ends, double &last) {
                const unsigned long long goes_on = __builtin_amdgcn_ballot_w64(!ends);
                double from = moved<0x138, 0xf>(last, c);   // wave_shr:1
                if (goes_on) {
                    const unsigned long long starts = ~(goes_on << 1) & ((2ull << lane) - 1);   // up to this lane; bit 0 is set
                    const int start = 63 - __builtin_clzll(starts | 1);
                    const int2v w = __builtin_bit_cast(int2v, from);
                    const int2v f = {__builtin_amdgcn_ds_bpermute(4 * start, w.x), __builtin_amdgcn_ds_bpermute(4 * start, w.y)};
                    from = __builtin_bit_cast(double, f);
                }
                last = goes_on >> 63 ? lane_of(from, 63) : lane_of(c, 63);
                return from;
            };
            // Labels of strategy b, `before_these` of which there are already: where the next `count` go.
            auto room = [&](int count) {
                int to = 0;
                if (lane == 0) to = draw(sh.found + slot, count);
                return uniform(to);
            };
            auto emit = [&](bool stays, unsigned long long these, int b, int before_these, int to, double c, int32_t w) {
                const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(these >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)these, 0));
                to += below;
                if (n == 1) {   // one strategy: these are in order, and none is read any more where they go
                    const Label label = {c, w, 0};
                    if (stays && at + to < n_hist) {
                        put(sh.f.label + to, label);
                        hist[(uint32_t)(at + to)] = words(label);
                    }
                } else if (stays && to < LABELS) {
                    sh.f.key[now][to] = __builtin_fma((double)w, KEY_W, (double)(b * (int)KEY_S + before_these + below));
                    sh.f.cost[to] = c;
                }
            };
            // the labels of strategy b: from those of the layer before in turn, 64 at a time
            if (l && before <= 64) {   // a turn is all there is
                for (int b = wave; b < n; b += WORKERS) {
                    const Label old = label_at(sh.f.label + min(lane, before - 1));
                    const int32_t next_w = sh.f.label[min(lane + 1, before - 1)].w;
                    const double turn = sh.f.turns[now][old.s * n + b];
                    const double2 *row = reinterpret_cast<const double2 *>(sh.f.lines[now] + b * LINE);
                    double2 line[LINES_HELD ? LINES_HELD * WINDOW / 2 : 1];
#pragma unroll
                    for (int i = 0; i < LINES_HELD * WINDOW / 2; ++i) line[i] = row[i];
                    const double2 costs = row[KEYS * WINDOW / 2];
                    const int32_t w = old.w + __builtin_bit_cast(int2v, costs.y).x;
                    const double c = prefix_min(lane < before ? old.c + turn : INFINITY, before) + costs.x;
                    const bool ends = lane >= before - 1 || next_w != old.w;
                    double last = INFINITY;
                    const double from = step_from(c, ends, last);   // (by all lanes)
                    const bool stays = (lane < before) & ends & (c < from) & alive(line, row, c, w);
                    const unsigned long long these = __builtin_amdgcn_ballot_w64(stays);
                    emit(stays, these, b, 0, room(__popcll(these)), c, w);
                }
            } else {
                for (int b = wave; b < n; b += WORKERS) {
                    const double2 *row = reinterpret_cast<const double2 *>(sh.f.lines[now] + b * LINE);
                    double2 line[LINES_HELD ? LINES_HELD * WINDOW / 2 : 1];
#pragma unroll
                    for (int i = 0; i < LINES_HELD * WINDOW / 2; ++i) line[i] = row[i];
                    const double2 costs = row[KEYS * WINDOW / 2];
                    const double own = costs.x;
                    const int32_t m = __builtin_bit_cast(int2v, costs.y).x;
                    double least = INFINITY, last = INFINITY;   // up to the labels before these: of the sums, of the costs
                    int found = 0;
                    // two turns side by side: each is a chain of dependent instructions
                    for (int j0 = 0; j0 < before; j0 += 128) {
                        double c[2];
                        int32_t w[2];
                        bool ends[2], stays[2];
                        unsigned long long these[2];
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            const int j = j0 + 64 * u + lane;
                            double x;
                            w[u] = m;
                            ends[u] = true;
                            if (l) {
                                const Label old = label_at(sh.f.label + min(j, before - 1));
                                ends[u] = j >= before - 1 || sh.f.label[min(j + 1, before - 1)].w != old.w;
                                x = old.c + sh.f.turns[now][old.s * n + b];
                                w[u] += old.w;
                            } else {
                                const gdouble M = inter + (size_t)sh.mat[0] * S * S + sh.kept[kept_at + b];
                                x = 0.0 + M[(size_t)min(lane, S - 1) * S];
                                x = min_f64(x, 0.0 + M[(size_t)min(lane + 64, S - 1) * S]);
                                x = lane_of(prefix_min(x), 63);
                            }
                            c[u] = prefix_min(j < before ? x : INFINITY);
                        }
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            c[u] = min_f64(c[u], least);
                            least = lane_of(c[u], 63);
                            c[u] += own;
                            const double from = step_from(c[u], ends[u], last);   // (by all lanes)
                            stays[u] = (j0 + 64 * u + lane < before) & ends[u] & (c[u] < from) & alive(line, row, c[u], w[u]);
                            these[u] = __builtin_amdgcn_ballot_w64(stays[u]);
                        }
                        const int first = __popcll(these[0]), count = first + __popcll(these[1]), to = room(count);
                        emit(stays[0], these[0], b, found, to, c[0], w[0]);
                        emit(stays[1], these[1], b, found + first, to + first, c[1], w[1]);
                        found += count;
                    }
                }
            }
            executed += (double)(l ? before : S) * n;
            __syncthreads();
            const int sum = uniform(sh.found[slot]);
            ns += layer_ns(n, before);
            if (sum == 0 || sum > LABELS || at + sum > n_hist || hopeless(ns, l, n, sum)) {
                give_up(sum == 0 ? 3 : 4);
                return;
            }
            const int32_t first_w = sh.f.label[0].w, last_w = sh.f.label[before - 1].w;   // of the layer before
            before = sum;
            if (t == 0) {
                sh.labels_at[l + 1] = at + sum;
                sh.found[slot == 0 ? 2 : slot - 1] = 0;   // of the layer after the next: all have read what it was
            }
            if (n == 1) {
                at += sum;
                continue;
            }
            // In the order of their memory: a label's place is how many keys are lower.
            auto lay_down = [&](double key, double c, int place) {
                const long long k = (long long)key;
                const Label label = {c, (int32_t)(k >> 17), (int32_t)(k >> 11) & 63};
                put(sh.f.label + place, label);
                hist[(uint32_t)(at + place)] = words(label);
            };
            if (sum > SORTED_FROM) {
                // Many: into 512 buckets of memory, and among the few of a bucket.  All lie between the lowest and the highest
                // of the layer before and what the strategies add to them.
                int32_t most = INT32_MIN, least_m = INT32_MAX;
                if (lane < n) most = least_m = __builtin_bit_cast(int2v, sh.f.lines[now][lane * LINE + KEYS * WINDOW + 1]).x;
                least_m = lanes_min(least_m);
                most = -lanes_min(-max(most, -INT32_MAX));
                const int32_t low = l ? first_w + least_m : least_m;
                const float scale = (float)BUCKETS / (float)((l ? last_w + most : most) - low + 1);
                constexpr int TIMES = (LABELS + 64 * WORKERS - 1) / (64 * WORKERS);
                double key[TIMES], c[TIMES];
                int q[TIMES], r[TIMES];
#pragma unroll
                for (int i = 0; i < TIMES; ++i) {
                    const int e = t + i * 64 * WORKERS;
                    if (e >= sum) continue;
                    key[i] = sh.f.key[now][e];
                    c[i] = sh.f.cost[e];
                    q[i] = min(max((int)((float)((int32_t)((long long)key[i] >> 17) - low) * scale), 0), BUCKETS - 1);
                    r[i] = atomicAdd(sh.f.bucket + q[i], 1);
                }
                __syncthreads();
                {
                    const int own = sh.f.bucket[t];
                    int x = own;
#pragma unroll
                    for (int w = 1; w < 64; w <<= 1) {
                        const int y = __shfl_up(x, w);
                        if (lane >= w) x += y;
                    }
                    sh.f.bucket_at[t] = x - own;
                    if (lane == 63) sh.f.buckets_of[wave] = x;
                }
                __syncthreads();
                int of[WORKERS];
#pragma unroll
                for (int w = 0; w < WORKERS; ++w) of[w] = sh.f.buckets_of[w];
#pragma unroll
                for (int i = 0; i < TIMES; ++i) {
                    if (t + i * 64 * WORKERS >= sum) continue;
                    int base = sh.f.bucket_at[q[i]];
#pragma unroll
                    for (int w = 0; w < WORKERS - 1; ++w) base += w < q[i] >> 6 ? of[w] : 0;
                    sh.f.sorted[base + r[i]] = key[i];
                    r[i] = base;
                }
                __syncthreads();
#pragma unroll
                for (int i = 0; i < TIMES; ++i) {
                    if (t + i * 64 * WORKERS >= sum) continue;
                    const int have = sh.f.bucket[q[i]];
                    int place = r[i];
                    for (int k = 0; k < have; ++k) place += sh.f.sorted[r[i] + k] < key[i];
                    lay_down(key[i], c[i], place);
                }
            } else {
                // Few: up to 8 lanes share the keys.
                const int share = sum <= 64 ? 3 : sum <= 128 ? 2 : sum <= 256 ? 1 : 0, lanes = 1 << share;   // (bits)
                const int part = ((sum + lanes - 1) >> share) + 7 & ~7;
                for (int e0 = wave << (6 - share); e0 < sum; e0 += WORKERS << (6 - share)) {
                    const int e = e0 + (lane >> share), from = (lane & (lanes - 1)) * part;
                    const double key = sh.f.key[now][min(e, sum - 1)], c = sh.f.cost[min(e, sum - 1)];
                    const double2 *p = reinterpret_cast<const double2 *>(sh.f.key[now] + from);
                    int to[4] = {};
                    for (int i = 0; i < part; i += 8, p += 4) {
                        const double2 x0 = p[0], x1 = p[1], x2 = p[2], x3 = p[3];
                        to[0] += x0.x < key;
                        to[1] += x0.y < key;
                        to[2] += x1.x < key;
                        to[3] += x1.y < key;
                        to[0] += x2.x < key;
                        to[1] += x2.y < key;
                        to[2] += x3.x < key;
                        to[3] += x3.y < key;
                    }
                    int place = to[0] + to[1] + to[2] + to[3];
                    if (share > 0) place += __builtin_amdgcn_mov_dpp(place, 0xb1, 0xf, 0xf, true);    // lane ^ 1
                    if (share > 1) place += __builtin_amdgcn_mov_dpp(place, 0x4e, 0xf, 0xf, true);    // lane ^ 2
                    if (share > 2) place += __builtin_amdgcn_mov_dpp(place, 0x141, 0xf, 0xf, true);   // mirrored within 8
                    if (e < sum && (lane & (lanes - 1)) == 0) lay_down(key, c, place);
                }
            }
            at += sum;
            __syncthreads();
        }
        // the start rows: a wave per key
        walks = wave < K && uniform(sh.budget[min(wave, K - 1)]) >= 0;
        if (walks) {
            v = uniform(sh.budget[wave]);
            double c = INFINITY;
            int s = INT32_MAX;
            for (int j = lane; j < before; j += 64) {
                const Label label = label_at(sh.f.label + j);
                if (label.w <= v && (label.c < c || (label.c == c && label.s < s))) {
                    c = label.c;
                    s = label.s;
                }
            }
            cheapest(c, s, before);
            total = c;
            cell = s;
            if (!(total < INFINITY) && lane == 0) sh.lost = 1;
        }
    }
    __syncthreads();
    if (sh.lost) {
        give_up(5);
        return;
    }

    // ---- backwards ----
    const giout res = GLOBAL(giout, I.res) + (size_t)min(wave, K - 1) * L;
    if (walks && lane == 0) res[L - 1] = sh.kept[sh.layer[L - 1].y + cell];
    for (int top = L - 1; top >= 0;) {
        // layers low .. top: their costs, the transitions into them and the labels before them lie in LDS together
        const int4 end = sh.layer[top + 1];
        const int low_of_lane = top - lane;
        const int4 begin = sh.layer[max(low_of_lane, 0)];
        const bool fits = low_of_lane >= 0 && end.y - begin.y <= BACK_KEPT && end.z - begin.z <= BACK_TURNS &&
                          sh.labels_at[top] - sh.labels_at[max(low_of_lane - 1, 0)] <= BACK_LABELS;
        const int low = top + 1 - __popcll(__builtin_amdgcn_ballot_w64(fits));
        const int kept0 = uniform(sh.layer[low].y), turns0 = uniform(sh.layer[low].z), labels0 = uniform(sh.labels_at[max(low - 1, 0)]);
        const int labels = uniform(sh.labels_at[top]) - labels0;
        __syncthreads();   // what lay there is not read any more
        for (int e = t; e < end.y - kept0; e += THREADS) {
            sh.b.mem[e] = hist_mem[(uint32_t)(kept0 + e)];
            sh.b.intra[e] = hist_intra[(uint32_t)(kept0 + e)];
        }
        for (int e = t; e < end.z - turns0; e += THREADS) sh.b.turns[e] = hist_turns[(uint32_t)(turns0 + e)];
        for (int e = t; e < labels; e += THREADS) *reinterpret_cast<int4v *>(sh.b.label + e) = hist[(uint32_t)(labels0 + e)];
        __syncthreads();
        if (walks) {
            // what a step needs beside the cell is fetched a step ahead: the layer, the first 64 labels before it
            int4 here = sh.layer[top], next = sh.layer[max(top - 1, 0)];
            int first = uniform(sh.labels_at[max(top - 1, 0)]) - labels0, end_of = labels;
            Label label = label_at(sh.b.label + min(first + lane, max(end_of, 1) - 1));
            for (int l = top; l >= low; --l) {
                const int n = uniform(here.x), kept_at = uniform(here.y) - kept0 + cell, turns_at = uniform(here.z) - turns0 + cell;
                const int32_t m = sh.b.mem[kept_at];
                const double own = sh.b.intra[kept_at];
                if (l == 0) {
                    v -= uniform(m);
                    break;
                }
                const double turn = sh.b.turns[turns_at + label.s * n];
                const int begin = first, all = end_of - first, kept_n = uniform(next.x), list = uniform(next.y);
                here = next;
                next = sh.layer[max(l - 2, 0)];
                end_of = first;
                first = max(uniform(sh.labels_at[max(l - 2, 0)]) - labels0, 0);
                v -= uniform(m);
                double c = lane < all && label.w <= v ? (label.c + turn) + own : INFINITY;
                int s = c < INFINITY ? label.s : INT32_MAX;
                for (int j = lane + 64; j < all; j += 64) {
                    const Label other = label_at(sh.b.label + begin + j);
                    const double x = other.w <= v ? (other.c + sh.b.turns[turns_at + other.s * n]) + own : INFINITY;
                    if (x < c || (x == c && other.s < s)) {
                        c = x;
                        s = other.s;
                    }
                }
                label = label_at(sh.b.label + min(first + lane, max(end_of, 1) - 1));
                if (all == 1) s = __builtin_amdgcn_readlane(s, 0);
                else cheapest(c, s, all);
                cell = min(s, kept_n - 1);   // (there is one: the cell has a cost)
                if (lane == 0) res[l - 1] = sh.kept[list + cell];
            }
        }
        top = low - 1;
    }
    if (wave < K && lane == 0) {
        out->total[wave] = walks ? total + GLOBAL(gdouble, I.other_time)[wave] : INFINITY;
        out->remaining[wave] = walks ? v : -1;
        out->executed[wave] = wave == 0 ? executed : 0.0;
        out->status[wave] = 0;
    }
}

}  // namespace

hipError_t bounds::launch_labels(const GdpBoundInst *inst, int n, int max_K, hipStream_t stream)
{
    const dim3 grid((unsigned)n);
    // 5 keys have a kernel of their own: its registers hold what that of 8 reads from LDS (L = 80, S = 64 298 us against 370)
    if (max_K <= 2) gdp_frontier_kernel<2><<<grid, THREADS, sizeof(Shared), stream>>>(inst);
    else if (max_K <= 4) gdp_frontier_kernel<4><<<grid, THREADS, sizeof(Shared), stream>>>(inst);
    else if (max_K == 5) gdp_frontier_kernel<5><<<grid, THREADS, sizeof(Shared), stream>>>(inst);
    else gdp_frontier_kernel<8><<<grid, THREADS, sizeof(Shared), stream>>>(inst);
    return hipGetLastError();
}
