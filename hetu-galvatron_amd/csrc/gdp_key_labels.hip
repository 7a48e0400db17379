// The DP over labels (gdp_frontier.hip) with a workgroup for every key of an instance.
//
// Between the layers of a call lies latency, not work: a wave issues one instruction in 4 clocks at best, one that waits for
// the one before in 9, one that waits for LDS in 120, a round trip to memory is 2000.  What this kernel does about it:
// * The labels of a key by itself are fewer than those of 4 keys together, and are held against one upper bound, by 8
//   multipliers instead of 4, wider apart (L = 80, S = 64, labels per layer: 42 of all keys, 10 of one).
// * The upper bound becomes better on the way: every label, completed by the cheapest ways on from its strategy under two
//   multipliers, is a path (30 layers of two kinds that trade memory for time: a third of the labels of the first bound).
// * What the layers need of the matrices is in LDS before the first one begins, of as many layers as fit together.
// * Where one strategy follows one strategy, which is most layers of random costs, labels only move: additions in
//   registers.  A layer's labels from up to 64 of the layer before are one wave's, without a barrier, while two passes of 64 lanes
//   do for them (16 labels and 8 strategies, 64 and 2); more are all 8 waves'.  A layer of those takes 3700 clocks for its labels
//   and 2500 for their order, of one wave 900.
// us, a workgroup for an instance (gdp_frontier.hip) -> one for each key: L = 80, S = 64 200 -> 71, L = 48, S = 88 83 -> 13, 256 instances of
// S = 44 136 -> 81.
#include "gdp_bounds.h"
#include "gdp_label_ops.h"

#include <math.h>

namespace {

constexpr int WAVES = 8, THREADS = 64 * WAVES;
constexpr int LABELS = 1536;      // of a layer
constexpr int KEPT = 64;          // strategies of a layer
constexpr int ALL_KEPT = 4096;    // ... and of all layers
constexpr int STAGED = 448, STAGED_TURNS = 3072;   // strategies, transitions in LDS at a time
constexpr int SOLO = 2;           // passes over the labels of a layer that one wave takes by itself
constexpr int WINDOW = 8, WAYS = 2;   // multipliers that labels are held against, and whose ways on complete them
constexpr int FIRST_WAY = WINDOW, COSTS = FIRST_WAY + 2 * WAYS, ROW = COSTS + 2;   // of a strategy: bounds; time and memory of the ways on; intra, memory
constexpr int KEY_PAD = 72;       // 8 lanes look at 8 keys at a time each
constexpr int BUCKETS = THREADS;
constexpr int SORTED_FROM = 192;  // labels of a layer that are laid down through buckets
constexpr int PER_ROW = THREADS / WINDOW, PER_COST = THREADS / 4;
constexpr int STAGE_ROWS = STAGED / PER_ROW, STAGE_COSTS = (STAGED + PER_COST - 1) / PER_COST;
static_assert(STAGED % PER_ROW == 0 && STAGED >= KEPT && WAYS == 2 && ROW % 2 == 0 && GDP_BOUND_MAX_S <= 128 && GDP_KEY_LABELS_MAX_L <= 128, "");

// Where those lie among more than 64 multipliers, around the best one, 8 below it and on, a byte each: close by, where most labels have
// theirs, and wider apart.
constexpr unsigned long long SPREAD = 0x0e0b090807060400ull;

// Of a label as it is found: w, strategy, number within the strategy in one whole number below 2^53.
constexpr double KEY_W = 0x1p17, KEY_S = 0x1p11;
static_assert(KEPT <= 64 && LABELS <= 2048, "6 bits and 11");

struct Forward {
    Label label[LABELS];
    __align__(16) double key[2][LABELS + KEY_PAD];   // +inf behind the last
    double cost[LABELS];
    int32_t bucket[BUCKETS], bucket_at[BUCKETS];
    __align__(16) int32_t buckets_of[WAVES];
};
constexpr int BACK_LABELS = sizeof(Forward) / sizeof(Label);

struct Shared {
    union {
        Forward f;
        Label back[BACK_LABELS];   // of the walk back
    };
    __align__(16) double rows[STAGED * ROW];
    double turns[STAGED_TURNS];
    __align__(16) double solo_key[64 * SOLO + 16], solo_cost[64 * SOLO];
    double single[GDP_KEY_LABELS_MAX_L + 1];         // memory of the layers before this one that have one strategy
    __align__(16) double ub_of[3][WAVES];            // of the best paths that the waves have completed in a layer
    double ub, executed;
    // Per layer: strategies that stay, where their list begins, where the transitions into them would in one list, the matrix.  One
    // more at the end for the sums.
    int4 layer[GDP_KEY_LABELS_MAX_L + 1];
    int4 mark[GDP_KEY_LABELS_MAX_L];
    int4 state;                                      // what a wave by itself leaves: layer, labels before it, their sum, why it ends
    int32_t labels_at[GDP_KEY_LABELS_MAX_L + 1];     // where the labels of a layer begin in memory; of one strategy: none lie there
    int32_t labels_of[GDP_KEY_LABELS_MAX_L];         // how many there are
    int2 step[GDP_KEY_LABELS_MAX_L + 1];             // strategies of a layer, and how many layers from it on have one behind one
    int32_t res[GDP_KEY_LABELS_MAX_L];               // the strategies of the best path
    int32_t several_before[GDP_KEY_LABELS_MAX_L];    // the last layer before it of more than one, -1: none
    int32_t found[3];                                // labels of a layer, of the next one of all waves and the one after that
    int32_t lost, unsorted, told;
    uint16_t chunk[GDP_KEY_LABELS_MAX_L + 1];        // first layers of what lies in LDS together
    uint16_t kept[ALL_KEPT];                         // layer * 128 + strategy
};
static_assert(sizeof(Shared) <= 160 * 1024, "LDS of a compute unit");

constexpr unsigned long long GIVEN_UP = ~0ull - 1;   // (as a bound it would be a NaN)
enum { GOES_ON = 0, NO_PATH = 1, TOO_MANY_KEPT = 2, NONE_LEFT = 3, TOO_MANY = 4, UNSORTED = -1 };

__device__ __forceinline__ int prefix_sum(int x)
{
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
    return x;
}

// The same of a whole number as a double.
__device__ __forceinline__ double prefix_sum(double x)
{
    x += moved<0x111, 0xf>(0.0, x);
    x += moved<0x112, 0xf>(0.0, x);
    x += moved<0x114, 0xf>(0.0, x);
    x += moved<0x118, 0xf>(0.0, x);
    x += moved<0x142, 0xa>(0.0, x);
    x += moved<0x143, 0xc>(0.0, x);
    return x;
}

// Minimum over the lanes up to this one, of each 16, 32 or 64 (bits: 4, 5, 6).  What a lane without a source keeps of the step before is
// one of those it is the minimum of, so that nothing has to be put there.
__device__ __forceinline__ double prefix_min_of(double x, int bits)
{
    double m = moved<0x111, 0xf>(INFINITY, x);
    x = min_f64(x, m);
    m = moved<0x112, 0xf>(m, x);
    x = min_f64(x, m);
    m = moved<0x114, 0xf>(m, x);
    x = min_f64(x, m);
    m = moved<0x118, 0xf>(m, x);
    x = min_f64(x, m);
    if (bits > 4) {
        m = moved<0x142, 0xa>(m, x);
        x = min_f64(x, m);
    }
    if (bits > 5) {
        m = moved<0x143, 0xc>(m, x);
        x = min_f64(x, m);
    }
    return x;
}

__device__ __forceinline__ unsigned long long lanes_where(bool x) { return __builtin_amdgcn_ballot_w64(x); }
__device__ __forceinline__ int lanes_below(unsigned long long m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
}
// A label's memory and strategy from its key: 2^52 more, and the whole number is the low bits of the double.
__device__ __forceinline__ Label label_of(double key, double c)
{
    const int2v w = __builtin_bit_cast(int2v, key + 0x1p52);
    return Label{c, (int32_t)__builtin_amdgcn_alignbit((uint32_t)w.y, (uint32_t)w.x, 17), w.x >> 11 & 63};
}

// What the lanes of a wave have written before is read by others of them from here on.  LDS is in order for a wave; this keeps the compiler
// to it, too.
__device__ __forceinline__ void in_order() { __builtin_amdgcn_wave_barrier(); }

__device__ __forceinline__ int32_t low_word(double x) { return __builtin_bit_cast(int2v, x).x; }

// grid (keys, instances).
__global__ __launch_bounds__(THREADS) void gdp_key_labels_kernel(const GdpBoundInst *inst)
{
    extern __shared__ __align__(16) char lds[];
    Shared &sh = *reinterpret_cast<Shared *>(lds);
    const GdpBoundInst &I = inst[blockIdx.y];
    const int own_key = (int)blockIdx.x;
    if (own_key >= I.K) return;   // the whole workgroup
    const int L = uniform(I.L), S = uniform(I.S), LS = L * S;
    const int t = (int)threadIdx.x, lane = t & 63, wave = uniform(t >> 6);
    GdpFrontierOut *const out = I.out;
    // By the whole workgroup.  The other keys of the instance are told, in the place of their upper bound, and look there every 4th
    // layer: nothing of it is kept.  (15 stages of a fit, L = 30, S = 37, 4 keys, one or two given up: 712 -> 574 us, 824 -> 591; where
    // none is, nothing: 420 and 422.)
    auto give_up = [&](int why) {
        if (t == 0) out->status[own_key] = why;
        if (t < I.K && t != own_key) {
            unsigned long long *const of = I.ub + t;
            if (__hip_atomic_load(of, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != ~0ull)   // (no path: its status says so)
                __hip_atomic_store(of, GIVEN_UP, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    const int64_t B = GLOBAL(const __attribute__((address_space(1))) int64_t *, I.budget)[own_key];
    unsigned long long known = 0;   // the workgroup of another key may write here by now: one wave asks, and decides for all
    if (t < 64) known = __hip_atomic_load(I.ub + own_key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    const int best = GLOBAL(gint, I.best)[own_key];
    const __attribute__((address_space(1))) int4v *marks = GLOBAL(const __attribute__((address_space(1))) int4v *, I.marks) + (size_t)own_key * L;
    int4v mark = marks[min(lane, L - 1)];
    int32_t matrix = GLOBAL(gint, I.index)[min(lane, L - 1)];
    if (B < 0) {   // no solution
        if (t == 0) {
            out->total[own_key] = INFINITY;
            out->remaining[own_key] = -1;
            out->executed[own_key] = 0.0;
            out->status[own_key] = 0;
        }
        return;
    }
    const int32_t budget = uniform((int32_t)B);
    const gdouble Q = GLOBAL(gdouble, I.Q), intra = GLOBAL(gdouble, I.intra), inter = GLOBAL(gdouble, I.inter_f);
    const gint Q_mem = GLOBAL(gint, I.Q_mem), mem = GLOBAL(gint, I.mem);
    const glabel hist = GLOBAL(glabel, I.hist) + (size_t)own_key * I.n_hist;
    const int n_hist = uniform(I.n_hist);
    const double limit = uniform(I.limit);

    // ---- the multipliers: a thread has the same of 8, and of the 2 ways on, wherever it fetches what belongs to one ----
    const int n_lam = I.n_lam;
    auto multiplier = [&](int by) { return min(max(best + by, 0), n_lam - 1); };
    const int bound_multiplier = multiplier(n_lam > 64 ? (int)(SPREAD >> 8 * (t % WINDOW) & 0xff) - 8 : t % WINDOW - WINDOW / 2), bound_at = bound_multiplier * LS;
    const int way = t & 3, way_multiplier = multiplier(way == 0 ? 0 : n_lam > 64 ? 2 : 1), way_at = way_multiplier * LS;
    const double bound_lam = GLOBAL(gdouble, I.lam)[bound_multiplier], way_lam = GLOBAL(gdouble, I.lam)[way_multiplier];
    const double shift = bound_lam * (double)budget + gdp_bound_margin(L, I.V, I.magnitude, bound_lam),
                 way_margin = gdp_bound_margin(L, I.V, I.magnitude, way_lam);
    double lam[WINDOW];
#pragma unroll
    for (int i = 0; i < WINDOW; ++i) lam[i] = lane_of(bound_lam, i);

    // ---- what stays, as lists ----
    if (wave == 0) {
        int sum = 0, turns = 0, before = 1;
        bool bad = false;
        for (int l0 = 0; l0 < L; l0 += 64) {
            const int l = l0 + lane;
            if (l0) {
                mark = marks[min(l, L - 1)];
                matrix = GLOBAL(gint, I.index)[min(l, L - 1)];
            }
            const int4v m = mark;
            const int n = l < L ? __popc(m.x) + __popc(m.y) + __popc(m.z) + __popc(m.w) : 0;
            const int y = n * __builtin_amdgcn_update_dpp(before, n, 0x138, 0xf, 0xf, false);   // wave_shr:1
            bad |= l < L && (n < 1 || n > KEPT || y > STAGED_TURNS);
            before = __builtin_amdgcn_readlane(n, 63);
            const int xs = prefix_sum(n), ys = prefix_sum(y);
            if (l < L) {
                sh.layer[l] = make_int4(n, sum + xs - n, turns + ys - y, matrix);
                sh.mark[l] = make_int4(m.x, m.y, m.z, m.w);
            }
            sum += __builtin_amdgcn_readlane(xs, 63);
            turns += __builtin_amdgcn_readlane(ys, 63);
        }
        const bool any_bad = lanes_where(bad) != 0;   // (of all lanes)
        if (lane == 0) {
            sh.layer[L] = make_int4(0, sum, turns, 0);
            sh.lost = known == ~0ull ? NO_PATH : known == GIVEN_UP ? TOO_MANY : any_bad || sum > ALL_KEPT ? TOO_MANY_KEPT : GOES_ON;
            sh.ub = gdp_unordered(known);
        }
    }
    for (int e = t; e < 2 * (LABELS + KEY_PAD); e += THREADS) sh.f.key[0][e] = INFINITY;   // both
    sh.f.bucket[t] = 0;
    if (t < 3) sh.found[t] = 0;
    if (t == 3) sh.told = 0;
    if (t == 0) {
        sh.f.label[0] = Label{0.0, 0, 0};   // before the first layer: one, no memory used
        sh.labels_at[0] = 0;
        sh.single[0] = 0.0;
    }
    __syncthreads();
    if (const int why = uniform(sh.lost); why != GOES_ON) {
        give_up(why);
        return;
    }
    double ub = uniform(sh.ub);
    for (int l = wave; l < L; l += WAVES) {
        const int4 m = sh.mark[l];
        const unsigned long long lo = (unsigned long long)(uint32_t)uniform(m.y) << 32 | (uint32_t)uniform(m.x),
                                 hi = (unsigned long long)(uint32_t)uniform(m.w) << 32 | (uint32_t)uniform(m.z);
        const int at = sh.layer[l].y;
        if (lo >> lane & 1) sh.kept[at + lanes_below(lo)] = (uint16_t)(l * 128 + lane);
        if (hi >> lane & 1) sh.kept[at + __popcll(lo) + lanes_below(hi)] = (uint16_t)(l * 128 + 64 + lane);
    }
    __syncthreads();

    if (wave < 2) {   // layers of more than one strategy, and those whose labels only move: one strategy behind one
        unsigned long long several[2], moves[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int l = 64 * h + lane, n = l < L ? sh.layer[min(l, L)].x : 0, n_prev = l && l <= L ? sh.layer[l - 1].x : 1;
            several[h] = lanes_where(n > 1);
            moves[h] = lanes_where(n == 1 && n_prev == 1);
        }
        const int l = t;
        const unsigned long long ends = ~(moves[wave] >> lane | (wave == 0 && lane ? moves[1] << (64 - lane) : 0)),
                                 lower = several[wave] & ((1ull << lane) - 1);
        const int before = lower ? 63 - __builtin_clzll(lower) + 64 * wave : wave && several[0] ? 63 - __builtin_clzll(several[0]) : -1;
        if (l <= L) sh.step[l] = make_int2(sh.layer[l].x, ends ? __builtin_ctzll(ends) : 64);
        if (l < L) sh.several_before[l] = before;
    }
    if (t == 128) sh.step[128] = make_int2(0, 0);
    if (t < L && sh.layer[t].x == 1) sh.res[t] = sh.kept[sh.layer[t].y] & 127;
    __syncthreads();

    // ---- what the layers need, in LDS ----
    // Layers from `low` on whose strategies and transitions fit together: the first that does not.
    auto chunk_end = [&](int low) {
        const int4 begin = sh.layer[low];
        for (int l0 = low;; l0 += 64) {
            const int4 end = sh.layer[min(l0 + lane + 1, L)];
            const int fit = __popcll(lanes_where(l0 + lane < L && end.y - begin.y <= STAGED && end.z - begin.z <= STAGED_TURNS));
            if (fit < 64) return l0 + fit;
        }
    };
    auto stage = [&](int low, int high) {
        const int k0 = uniform(sh.layer[low].y), all = uniform(sh.layer[high].y) - k0, t0 = uniform(sh.layer[low].z);
        auto at_of = [&](int g) {
            const int id = sh.kept[k0 + min(g, all - 1)];
            return (uint32_t)((id >> 7) * S + (id & 127));
        };
        double bound[STAGE_ROWS], time[STAGE_COSTS];
        int32_t need[STAGE_COSTS];
#pragma unroll
        for (int i = 0; i < STAGE_ROWS; ++i)
            if (i * PER_ROW < all) bound[i] = Q[bound_at + at_of(t / WINDOW + i * PER_ROW)];
#pragma unroll
        for (int i = 0; i < STAGE_COSTS; ++i) {
            if (i * PER_COST >= all) break;
            const uint32_t at = at_of(t / 4 + i * PER_COST);
            if (way < WAYS) {
                time[i] = Q[way_at + at];
                need[i] = Q_mem[way_at + at];
            } else {
                time[i] = intra[at];
                need[i] = mem[at];
            }
        }
        // transitions: 8 threads have the sources of a strategy
        double turn[STAGE_ROWS];
        int to[STAGE_ROWS];
        auto fetch_turns = [&](int from0) {
#pragma unroll
            for (int i = 0; i < STAGE_ROWS; ++i) {
                const int g = t / 8 + i * PER_ROW, from = from0 + t % 8;
                to[i] = -1;
                if (g >= all) continue;
                const int id = sh.kept[k0 + g], l = id >> 7;
                const int4 here = sh.layer[l], before = sh.layer[max(l - 1, 0)];
                if (l == 0 || from >= before.x) continue;
                const int source = sh.kept[before.y + from] & 127;
                turn[i] = inter[(size_t)here.w * S * S + (uint32_t)(source * S + (id & 127))];
                to[i] = here.z - t0 + from * here.x + (k0 + g - here.y);
            }
        };
        auto place_turns = [&]() {
#pragma unroll
            for (int i = 0; i < STAGE_ROWS; ++i)
                if (to[i] >= 0) sh.turns[to[i]] = turn[i];
        };
        fetch_turns(0);
#pragma unroll
        for (int i = 0; i < STAGE_ROWS; ++i) {
            const int g = t / WINDOW + i * PER_ROW;
            if (g < all) sh.rows[g * ROW + t % WINDOW] = bound[i] - shift;
        }
#pragma unroll
        for (int i = 0; i < STAGE_COSTS; ++i) {
            const int g = t / 4 + i * PER_COST;
            if (g >= all || way > WAYS) continue;
            const double x = way < WAYS ? time[i] - way_lam * (double)need[i] + way_margin : time[i];
            *reinterpret_cast<double2 *>(sh.rows + g * ROW + FIRST_WAY + 2 * way) = make_double2(x, __builtin_bit_cast(double, int2v{need[i], 0}));
        }
        place_turns();
        int widest = 0;
        for (int l = max(low, 1) + lane; l < high; l += 64) widest = max(widest, sh.layer[l - 1].x);
        widest = -lanes_min(-widest);
        for (int from0 = 8; from0 < widest; from0 += 8) {
            fetch_turns(from0);
            place_turns();
        }
        if (low == 0) {   // into the first layer from the zeros before it: the cheapest transition
            const gdouble M = inter + (size_t)uniform(sh.layer[0].w) * S * S;
            const int n = uniform(sh.layer[0].x);
            for (int b0 = wave; b0 < n; b0 += 2 * WAVES) {
                double x[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int s = sh.kept[min(b0 + u * WAVES, n - 1)] & 127;
                    x[u] = 0.0 + M[(uint32_t)(min(lane, S - 1) * S + s)];
                    x[u] = min_f64(x[u], 0.0 + M[(uint32_t)(min(lane + 64, S - 1) * S + s)]);
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    x[u] = prefix_min_of(x[u], 6);
                    if (lane == 63 && b0 + u * WAVES < n) sh.turns[b0 + u * WAVES] = x[u];
                }
            }
        }
    };

    // The sums of the layers with one strategy, behind stage(); by one wave.
    auto sum_singles = [&](int low, int high) {
        const int k0 = uniform(sh.layer[low].y);
        double before = low ? sh.single[low] : 0.0;
        for (int l0 = low; l0 < high; l0 += 64) {
            const int l = l0 + lane;
            const int4 of = sh.layer[min(l, high - 1)];
            const double x = prefix_sum(l < high && of.x == 1 ? (double)low_word(sh.rows[(of.y - k0) * ROW + COSTS + 1]) : 0.0);
            if (l < high) sh.single[l + 1] = before + x;
            before += lane_of(x, 63);
        }
    };

    // ---- forwards ----
    // The bound of what can still be part of a path that fits and is no worse than the best one known.
    auto bound_of = [&](const double2 *row, double w) {
        double b[WINDOW];
#pragma unroll
        for (int i = 0; i < WINDOW; i += 2) {
            const double2 r = row[i / 2];
            b[i] = __builtin_fma(lam[i], w, r.x);
            b[i + 1] = __builtin_fma(lam[i + 1], w, r.y);
        }
        return max_f64(max_f64(max_f64(b[0], b[1]), max_f64(b[2], b[3])), max_f64(max_f64(b[4], b[5]), max_f64(b[6], b[7])));
    };
    // The best path that a label of cost c, memory w is completed to.
    auto completed = [&](const double2 *row, double c, int32_t w) {
        const double2 a = row[FIRST_WAY / 2], b = row[FIRST_WAY / 2 + 1];
        const double x = c + a.x, y = c + b.x;
        const double fits_x = (uint32_t)w + (uint32_t)low_word(a.y) <= (uint32_t)budget ? x : INFINITY,
                     fits_y = (uint32_t)w + (uint32_t)low_word(b.y) <= (uint32_t)budget ? y : INFINITY;
        return min_f64(fits_x, fits_y);
    };
    // Of labels that need the same memory the cheapest counts, with the last of them: `from`, the least up to the label before, as it
    // is for the first of them.
    auto from_last_other = [&](double from, unsigned long long goes_on) {
        const unsigned long long starts = ~(goes_on << 1) & ((2ull << lane) - 1);   // up to this lane; bit 0 is set
        const int start = 63 - __builtin_clzll(starts | 1);
        const int2v w = __builtin_bit_cast(int2v, from);
        const int2v f = {__builtin_amdgcn_ds_bpermute(4 * start, w.x), __builtin_amdgcn_ds_bpermute(4 * start, w.y)};
        return __builtin_bit_cast(double, f);
    };
    // A pass over up to 64 labels, 1 << bits lanes for them, and as many strategies of the layer from b0 on beside each other as that
    // leaves room for.  own: the lane's label, alike for all strategies; goes_on: the next one needs the same memory.  Leaves cost and memory of
    // the lane's new label, its strategy, and which are to stay.
    struct Found {
        double c;
        int32_t w;
        int b;
        bool stays;
        unsigned long long these;   // ... of all lanes
    };
    auto pass = [&](const double *rows, const double *turns, int n, int n_prev, int labels, const Label &own, unsigned long long goes_on, int bits, int b0,
                    bool completes, double &best_path) {
        Found f;
        const int j = lane & ((1 << bits) - 1);
        f.b = b0 + (lane >> bits);
        const bool there = (j < labels) & (f.b < n);
        f.b = min(f.b, n - 1);
        const double2 *const row = reinterpret_cast<const double2 *>(rows + f.b * ROW);
        const double x = own.c + turns[own.s * n + f.b];
        const double2 cost = row[COSTS / 2];
        f.w = own.w + low_word(cost.y);
        const double bound = bound_of(row, (double)f.w);
        f.c = there ? x : INFINITY;
        if (n_prev > 1) f.c = prefix_min_of(f.c, bits);
        f.c += cost.x;
        double from = moved<0x138, 0xf>(INFINITY, f.c);   // wave_shr:1
        from = j == 0 ? INFINITY : from;
        if (goes_on) from = from_last_other(from, goes_on);
        f.stays = there & (f.c < from) & (f.w <= budget) & (f.c + bound <= ub);
        if (goes_on) f.stays &= !(goes_on >> lane & 1);
        f.these = lanes_where(f.stays);
        if (completes) best_path = min_f64(best_path, completed(row, f.c, f.w));
        return f;
    };
    auto key_of = [&](int32_t w, int b, int number) { return __builtin_fma((double)w, KEY_W, (double)(b * (int)KEY_S + number)); };
    auto bits_for = [](int labels) { return labels <= 16 ? 4 : labels <= 32 ? 5 : 6; };
    // What a layer takes, in ns, where all waves take part.  An instance whose other layers would take longer than the dense
    // recurrence is left to that one; what its labels have taken by then does not come back either way (gdp_frontier.hip).
    auto layer_ns = [](int n, int before) {
        return (before > SORTED_FROM ? 3000 : 1500) + ((n + WAVES - 1) / WAVES) * ((before + 127) / 128) * 700;
    };
    auto hopeless = [&](int ns, int l, int n, int labels) {
        if (labels <= 64) return false;
        const int ahead = L - 1 - l;
        if ((double)ns * (double)ahead > limit * (double)(l + 1)) return true;
        if (l >= L / 2) return (double)ahead * layer_ns(n, labels / 2) > limit;
        if (l < max(2, L / 16)) return false;
        const int half = (l - 1) / 2, grown = labels - uniform(sh.labels_of[half]);
        const int top = labels + max(grown, 0) * (L / 2 - l) / (l - half);
        return top > 2 * LABELS || (double)ns + (double)(L - l) * layer_ns(n, top / 2) > 0.9 * limit;
    };

    int l = 0, before = 1, at = 0, chunks = 0, high = 0, ns = 0;
    int keys_in = 0, others = 0, slot = 0;   // where the next keys go, how many lie in the other place; of the counts
    double executed = 0.0;
    while (l < L) {
        const int low = l;
        if (t == 0) sh.chunk[chunks] = (uint16_t)low;
        ++chunks;
        high = uniform(chunk_end(low));
        stage(low, high);
        __syncthreads();
        if (wave == 0) {
            sum_singles(low, high);
            in_order();
        }
        const int k0 = uniform(sh.layer[low].y), t0 = uniform(sh.layer[low].z);
        while (l < high) {
            int n = uniform(sh.layer[l].x), sum = 0;
            if (before <= 64 && (n << bits_for(before)) <= 64 * SOLO) {
                // ---- one wave, its labels in registers ----
                if (wave == 0) {
                    int bits = bits_for(before), why = GOES_ON, n_prev = l ? uniform(sh.layer[l - 1].x) : 1;
                    Label own = label_at(sh.f.label + min(lane & ((1 << bits) - 1), before - 1));
                    const double *rows = sh.rows + (uniform(sh.layer[l].y) - k0) * ROW, *turns = sh.turns + (uniform(sh.layer[l].z) - t0);
                    if (l == 0) executed += (double)((S - 1) * n);   // before the first layer there is one of each strategy
                    int moving = uniform(sh.step[l].y);
                    for (;;) {
                        const int run = min(moving, high - l);
                        const int2 step = sh.step[l + max(run, 1)];
                        if (run > 0) {   // the labels move; those beyond the budget are the last ones
                            const int i = min(lane, run - 1);
                            const double intra_of = rows[i * ROW + COSTS], turn_of = turns[i];
                            const double more = sh.single[l + run] - sh.single[l];
                            for (int k = 0; k < run; ++k) own.c = (own.c + lane_of(turn_of, k)) + lane_of(intra_of, k);
                            executed += (double)(before * run);
                            const double w = (double)own.w + more;
                            before = __popcll(lanes_where(((lane & ((1 << bits) - 1)) < before) & (w <= (double)budget))) >> (6 - bits);
                            own.w = (int32_t)w;
                            if (before == 0) {
                                why = NONE_LEFT;
                                break;
                            }
                            if (lane < run) {
                                sh.labels_at[l + 1 + lane] = at;
                                sh.labels_of[l + lane] = before;
                            }
                            if (bits_for(before) != bits) {   // fewer: more strategies beside each other again
                                if (lane < before) put(sh.f.label + lane, own);
                                in_order();
                                bits = bits_for(before);
                                own = label_at(sh.f.label + min(lane & ((1 << bits) - 1), before - 1));
                            }
                            l += run;
                            rows += run * ROW;
                            turns += run;
                            n_prev = 1;
                        } else {
                            const int32_t next_w = __builtin_amdgcn_update_dpp(0, own.w, 0x130, 0xf, 0xf, false);   // wave_shl:1
                            const unsigned long long goes_on = n_prev > 1 ? lanes_where(((lane & ((1 << bits) - 1)) < before - 1) & (next_w == own.w)) : 0;
                            double best_path = INFINITY;
                            int found = 0;
                            for (int b0 = 0; b0 < n; b0 += 64 >> bits) {
                                const Found f = pass(rows, turns, n, n_prev, before, own, goes_on, bits, b0, before > 8, best_path);
                                const int below = lanes_below(f.these);
                                if (f.stays) {
                                    if (n == 1) put(sh.f.label + below, Label{f.c, f.w, 0});
                                    else {
                                        sh.solo_key[found + below] = key_of(f.w, f.b, below);
                                        sh.solo_cost[found + below] = f.c;
                                    }
                                }
                                found += __popcll(f.these);
                            }
                            in_order();
                            executed += (double)(before * n);
                            if (before > 8) ub = min_f64(ub, lane_of(prefix_min_of(best_path, 6), 63));
                            if (found > 64) {   // all waves lay them down
                                for (int e = lane; e < found; e += 64) {
                                    sh.f.key[keys_in][e] = sh.solo_key[e];
                                    sh.f.cost[e] = sh.solo_cost[e];
                                }
                                if (lane == 0) sh.unsorted = found;
                                why = UNSORTED;
                                break;
                            }
                            if (found == 0 || at + found > n_hist) {
                                why = found == 0 ? NONE_LEFT : TOO_MANY;
                                break;
                            }
                            if (n > 1) {   // a label's place is how many keys are lower; 4 or 2 lanes share the keys where they are few
                                if (lane < 16) sh.solo_key[found + lane] = INFINITY;
                                in_order();
                                const int share = found <= 16 ? 2 : found <= 32 ? 1 : 0, lanes = 1 << share;   // (bits)
                                const int part = ((found + lanes - 1) >> share) + 3 & ~3, e = min(lane >> share, found - 1);
                                const double key = sh.solo_key[e], c = sh.solo_cost[e];
                                const double2 *p = reinterpret_cast<const double2 *>(sh.solo_key + (lane & (lanes - 1)) * part);
                                int place = 0, place2 = 0;
                                for (int i = 0; i < part; i += 4, p += 2) {
                                    const double2 x0 = p[0], x1 = p[1];
                                    place += x0.x < key;
                                    place2 += x0.y < key;
                                    place += x1.x < key;
                                    place2 += x1.y < key;
                                }
                                place += place2;
                                if (share > 0) place += __builtin_amdgcn_mov_dpp(place, 0xb1, 0xf, 0xf, true);    // lane ^ 1
                                if (share > 1) place += __builtin_amdgcn_mov_dpp(place, 0x4e, 0xf, 0xf, true);    // lane ^ 2
                                const Label label = label_of(key, c);
                                if (lane >> share < found && (lane & (lanes - 1)) == 0) {
                                    put(sh.f.label + place, label);
                                    hist[(uint32_t)(at + place)] = words(label);
                                }
                                at += found;
                                in_order();
                            }
                            before = found;
                            bits = bits_for(before);
                            own = label_at(sh.f.label + min(lane & ((1 << bits) - 1), before - 1));
                            if (lane == 0) {
                                sh.labels_at[l + 1] = at;
                                sh.labels_of[l] = before;
                            }
                            ++l;
                            rows += n * ROW;
                            turns += n * n_prev;
                            n_prev = n;
                        }
                        n = uniform(step.x);
                        moving = uniform(step.y);
                        if (l >= high || (n << bits) > 64 * SOLO) break;
                    }
                    if (why <= GOES_ON && lane < before) put(sh.f.label + lane, own);
                    if (lane == 0) {
                        sh.state = make_int4(l, before, at, why);
                        sh.ub = ub;
                        sh.executed = executed;
                    }
                }
                __syncthreads();
                const int4 state = sh.state;
                const int why = uniform(state.w);
                ns += 600 * (uniform(state.x) - l);
                l = uniform(state.x);
                at = uniform(state.z);
                ub = uniform(sh.ub);
                executed = sh.executed;
                if (why > GOES_ON) {
                    give_up(why);
                    return;
                }
                before = uniform(state.y);
                if (why == GOES_ON) continue;
                sum = uniform(sh.unsorted);
                n = uniform(sh.layer[l].x);
                sh.f.bucket[t] = 0;
                __syncthreads();
            } else {
                // ---- all waves ----
                const int n_prev = l ? uniform(sh.layer[l - 1].x) : 1;
                const double *const rows = sh.rows + (uniform(sh.layer[l].y) - k0) * ROW, *const turns = sh.turns + (uniform(sh.layer[l].z) - t0);
                const bool completes = l & 1, asks = l % 4 == 3;
                unsigned long long told = 0;
                if (asks && t == 0) told = __hip_atomic_load(I.ub + own_key, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                sh.f.bucket[t] = 0;
                double best_path = INFINITY;
                auto room = [&](int count) {
                    int to = 0;
                    if (lane == 0) to = draw(sh.found + slot, count);
                    return uniform(to);
                };
                auto emit = [&](const Found &f, int place, int number) {
                    if (!f.stays) return;
                    if (n == 1) put(sh.f.label + place, Label{f.c, f.w, 0});   // these are in order, and none is read any more where they go
                    else if (place < LABELS) {
                        sh.f.key[keys_in][place] = key_of(f.w, f.b, number);
                        sh.f.cost[place] = f.c;
                    }
                };
                if (before <= 64) {
                    const int bits = bits_for(before), j = min(lane & ((1 << bits) - 1), before - 1);
                    const Label own = label_at(sh.f.label + j);
                    const unsigned long long goes_on = lanes_where(j < before - 1 && sh.f.label[min(j + 1, before - 1)].w == own.w);
                    for (int b0 = wave * (64 >> bits); b0 < n; b0 += WAVES * (64 >> bits)) {
                        const Found f = pass(rows, turns, n, n_prev, before, own, goes_on, bits, b0, completes, best_path);
                        const int below = lanes_below(f.these);
                        emit(f, room(__popcll(f.these)) + below, below);
                    }
                } else {
                    for (int b = wave; b < n; b += WAVES) {
                        const double2 *row = reinterpret_cast<const double2 *>(rows + b * ROW);
                        const double2 cost = row[COSTS / 2];
                        double least = INFINITY, last = INFINITY;   // up to the labels before these: of the sums, of the costs
                        int found = 0;
                        for (int j0 = 0; j0 < before; j0 += 128) {   // two turns of them side by side: each is a chain of dependent instructions
                            Found f[2];
                            unsigned long long goes_on[2];
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                const int j = j0 + 64 * u + lane;
                                const Label old = label_at(sh.f.label + min(j, before - 1));
                                goes_on[u] = lanes_where(j < before - 1 && sh.f.label[min(j + 1, before - 1)].w == old.w);
                                const double x = old.c + turns[old.s * n + b];
                                f[u].b = b;
                                f[u].w = old.w + low_word(cost.y);
                                f[u].c = prefix_min_of(j < before ? x : INFINITY, 6);
                            }
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                f[u].c = min_f64(f[u].c, least);
                                least = lane_of(f[u].c, 63);
                                f[u].c += cost.x;
                                double from = moved<0x138, 0xf>(last, f[u].c);   // wave_shr:1
                                if (goes_on[u]) from = from_last_other(from, goes_on[u]);
                                last = goes_on[u] >> 63 ? lane_of(from, 63) : lane_of(f[u].c, 63);
                                const bool there = (j0 + 64 * u + lane < before) & !(goes_on[u] >> lane & 1);
                                const double bound = bound_of(row, (double)f[u].w);
                                f[u].stays = there & (f[u].c < from) & (f[u].w <= budget) & (f[u].c + bound <= ub);
                                f[u].these = lanes_where(f[u].stays);
                                if (completes) best_path = min_f64(best_path, there ? completed(row, f[u].c, f[u].w) : INFINITY);
                            }
                            const int first = __popcll(f[0].these), count = first + __popcll(f[1].these), to = room(count);
                            emit(f[0], to + lanes_below(f[0].these), found + lanes_below(f[0].these));
                            emit(f[1], to + first + lanes_below(f[1].these), found + first + lanes_below(f[1].these));
                            found += count;
                        }
                    }
                }
                if (completes) {
                    best_path = lane_of(prefix_min_of(best_path, 6), 63);
                    if (lane == 0) sh.ub_of[slot][wave] = best_path;
                }
                executed += (double)((l ? before : S) * n);
                ns += layer_ns(n, before);
                if (asks && t == 0) sh.told = told == GIVEN_UP;
                __syncthreads();
                sum = uniform(sh.found[slot]);
                if (completes) {
                    const double2 *of = reinterpret_cast<const double2 *>(sh.ub_of[slot]);
                    const double2 a = of[0], c = of[1], d = of[2], e = of[3];
                    ub = uniform(min_f64(ub, min_f64(min_f64(min_f64(a.x, a.y), min_f64(c.x, c.y)), min_f64(min_f64(d.x, d.y), min_f64(e.x, e.y)))));
                }
                if (t == 0) sh.found[slot == 0 ? 2 : slot - 1] = 0;   // all have read what it was
                slot = slot == 2 ? 0 : slot + 1;
            }
            if (sum == 0 || sum > LABELS || at + sum > n_hist || (l % 4 == 3 && (uniform(sh.told) != 0 || hopeless(ns, l, n, sum)))) {
                give_up(sum == 0 ? NONE_LEFT : TOO_MANY);
                return;
            }
            if (n > 1) {
                // In the order of their memory: a label's place is how many keys are lower.
                auto lay_down = [&](double key, double c, int place) {
                    const Label label = label_of(key, c);
                    put(sh.f.label + place, label);
                    hist[(uint32_t)(at + place)] = words(label);
                };
                double *const keys = sh.f.key[keys_in];
                for (int e = t; e < others; e += THREADS) sh.f.key[keys_in ^ 1][e] = INFINITY;
                others = sum;
                keys_in ^= 1;
                if (sum > SORTED_FROM) {
                    // Many: into 512 buckets of memory, and among the few of a bucket.
                    constexpr int TIMES = LABELS / THREADS;
                    double key[TIMES], c[TIMES];
                    int q[TIMES], r[TIMES];
                    const int32_t low_w = sh.f.label[0].w, high_w = sh.f.label[before - 1].w;   // of the layer before
                    int32_t most = INT32_MIN + 1, least_m = INT32_MAX;
                    const int row = uniform(sh.layer[l].y) - k0 + lane;
                    if (lane < n) most = least_m = low_word(sh.rows[row * ROW + COSTS + 1]);
                    least_m = lanes_min(least_m);
                    most = -lanes_min(-most);
                    const float scale = (float)BUCKETS / (float)(high_w + most - (low_w + least_m) + 1);
#pragma unroll
                    for (int i = 0; i < TIMES; ++i) {
                        const int e = t + i * THREADS;
                        if (e >= sum) continue;
                        key[i] = keys[e];
                        c[i] = sh.f.cost[e];
                        q[i] = min(max((int)((float)(label_of(key[i], 0.0).w - (low_w + least_m)) * scale), 0), BUCKETS - 1);
                        r[i] = atomicAdd(sh.f.bucket + q[i], 1);
                    }
                    __syncthreads();
                    {
                        const int own = sh.f.bucket[t], x = prefix_sum(own);
                        sh.f.bucket_at[t] = x - own;
                        if (lane == 63) sh.f.buckets_of[wave] = x;
                    }
                    __syncthreads();
                    int of[WAVES];
#pragma unroll
                    for (int w = 0; w < WAVES; ++w) of[w] = sh.f.buckets_of[w];
#pragma unroll
                    for (int i = 0; i < TIMES; ++i) {
                        if (t + i * THREADS >= sum) continue;
                        int base = sh.f.bucket_at[q[i]];
#pragma unroll
                        for (int w = 0; w < WAVES - 1; ++w) base += w < q[i] >> 6 ? of[w] : 0;
                        keys[base + r[i]] = key[i];   // in the place of the keys as they were found, which all have read
                        r[i] = base;
                    }
                    __syncthreads();
#pragma unroll
                    for (int i = 0; i < TIMES; ++i) {
                        if (t + i * THREADS >= sum) continue;
                        const int have = sh.f.bucket[q[i]];
                        int place = r[i];
                        for (int k = 0; k < have; ++k) place += keys[r[i] + k] < key[i];
                        lay_down(key[i], c[i], place);
                    }
                } else {
                    // Few: up to 8 lanes share the keys.
                    const int share = sum <= 64 ? 3 : sum <= 128 ? 2 : 1, lanes = 1 << share;   // (bits)
                    const int part = ((sum + lanes - 1) >> share) + 7 & ~7;
                    const int e = t >> share, from = (lane & (lanes - 1)) * part;   // (512 threads: all labels at a time)
                    if (e < sum) {
                        const double key = keys[e], c = sh.f.cost[e];
                        const double2 *p = reinterpret_cast<const double2 *>(keys + from);
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
                        place += __builtin_amdgcn_mov_dpp(place, 0xb1, 0xf, 0xf, true);                    // lane ^ 1
                        if (share > 1) place += __builtin_amdgcn_mov_dpp(place, 0x4e, 0xf, 0xf, true);    // lane ^ 2
                        if (share > 2) place += __builtin_amdgcn_mov_dpp(place, 0x141, 0xf, 0xf, true);   // mirrored within 8
                        if ((lane & (lanes - 1)) == 0) lay_down(key, c, place);
                    }
                }
                __syncthreads();
            }
            if (n > 1) at += sum;   // (labels of layers with one strategy are not looked at again)
            before = sum;
            if (t == 0) {
                sh.labels_at[l + 1] = at;
                sh.labels_of[l] = sum;
            }
            ++l;
        }
        __syncthreads();   // what lies in LDS is not read any more
    }

    // ---- the start row: the cheapest label that fits, of those the lowest strategy ----
    int cell = 0;          // strategy of the cell, counted among those that stay
    int32_t v = budget;    // its budget
    double total = INFINITY;
    if (wave == 0) {
        int s = INT32_MAX;
        for (int j = lane; j < before; j += 64) {
            const Label label = label_at(sh.f.label + j);
            if (label.w <= v && (label.c < total || (label.c == total && label.s < s))) {
                total = label.c;
                s = label.s;
            }
        }
        cheapest(total, s, before);
        cell = s;
        if (lane == 0) sh.lost = !(total < INFINITY);
    }
    __syncthreads();
    if (sh.lost) {
        give_up(5);
        return;
    }

    // ---- backwards ----
    // Layers with one strategy are passed by in one step; of the others wave 0 looks for the cheapest label that leads to the cell.
    if (t == 0) sh.res[L - 1] = sh.kept[sh.layer[L - 1].y + cell] & 127;
    int walk = L - 1;        // the layer of the cell
    bool paid = false;       // whether its budget is that before it already
    for (int chunk = chunks - 1, top = L - 1; chunk >= 0; --chunk) {
        const int low = uniform((int)sh.chunk[chunk]);
        if (chunk != chunks - 1) {
            __syncthreads();
            stage(low, top + 1);
        }
        const int k0 = uniform(sh.layer[low].y), t0 = uniform(sh.layer[low].z);
        while (top >= low) {
            // layers from `lowest` on whose labels before them lie in LDS together
            int lowest = top + 1;
            for (;;) {
                const int l = lowest - 1 - lane;
                const int fit = __popcll(lanes_where(l >= low && sh.labels_at[top] - sh.labels_at[max(l - 1, 0)] <= BACK_LABELS));
                lowest -= fit;
                if (fit < 64) break;
            }
            lowest = uniform(lowest);
            const int first = uniform(sh.labels_at[max(lowest - 1, 0)]), labels = uniform(sh.labels_at[top]) - first;
            __syncthreads();
            for (int e = t; e < labels; e += THREADS) *reinterpret_cast<int4v *>(sh.back + e) = hist[(uint32_t)(first + e)];
            __syncthreads();
            if (wave == 0 && walk >= lowest) {
                // What a step needs beside the cell, fetched a step ahead: the last layer before of several strategies, `next`; the one
                // behind it, whose matrix leads there; their labels; the memory of the layers with one strategy between.
                struct Step {
                    int next, begin, end;
                    int4 behind;
                    double between;
                    Label label;
                };
                auto step_of = [&](int l) {
                    Step s;
                    s.next = uniform(sh.several_before[max(l, 0)]);
                    s.behind = sh.layer[s.next + 1];
                    s.begin = uniform(sh.labels_at[max(s.next, 0)]) - first;
                    s.end = uniform(sh.labels_at[s.next + 1]) - first;
                    s.between = sh.single[max(l, 0)] - sh.single[s.next + 1];
                    s.label = label_at(sh.back + max(min(s.begin + lane, BACK_LABELS - 1), 0));   // (of a layer that is not here: of no use)
                    return s;
                };
                Step step = step_of(walk);
                int row = uniform(sh.layer[walk].y) - k0;
                while (walk >= lowest) {
                    double2 costs = *reinterpret_cast<const double2 *>(sh.rows + (row + cell) * ROW + COSTS);
                    if (!paid) v -= uniform(low_word(costs.y));
                    if (step.next < walk - 1 || step.next < 0) {   // one strategy each, down to the layer behind the next of several
                        v -= (int32_t)uniform(step.between);
                        walk = step.next < 0 ? -1 : step.next + 1;
                        cell = 0;
                        paid = true;
                        if (walk < lowest) break;
                        row = uniform(step.behind.y) - k0;
                        costs = *reinterpret_cast<const double2 *>(sh.rows + row * ROW + COSTS);
                    }
                    const Step after = step_of(step.next);
                    const int n = uniform(step.behind.x), count = step.end - step.begin;
                    const double *const turns = sh.turns + (uniform(step.behind.z) - t0) + cell;
                    double c = lane < count && step.label.w <= v ? (step.label.c + turns[step.label.s * n]) + costs.x : INFINITY;
                    int s = c < INFINITY ? step.label.s : INT32_MAX;
                    for (int j = lane + 64; j < count; j += 64) {
                        const Label label = label_at(sh.back + step.begin + j);
                        const double x = label.w <= v ? (label.c + turns[label.s * n]) + costs.x : INFINITY;
                        if (x < c || (x == c && label.s < s)) {
                            c = x;
                            s = label.s;
                        }
                    }
                    cheapest(c, s, count);
                    walk = step.next;
                    const int4 at_walk = sh.layer[walk];
                    cell = min(s, uniform(at_walk.x) - 1);   // (there is one: the cell has a cost)
                    if (lane == 0) sh.res[walk] = sh.kept[at_walk.y + cell] & 127;
                    row = uniform(at_walk.y) - k0;
                    paid = false;
                    step = after;
                }
            }
            top = lowest - 1;
        }
    }
    __syncthreads();
    const giout res = GLOBAL(giout, I.res) + (size_t)own_key * L;
    if (t < L) res[t] = sh.res[t];
    if (t == 0) {
        out->total[own_key] = total + GLOBAL(gdouble, I.other_time)[own_key];
        out->remaining[own_key] = v;
        out->executed[own_key] = executed;
        out->status[own_key] = 0;
    }
}

}  // namespace

hipError_t bounds::launch_key_labels(const GdpBoundInst *inst, int n, int max_K, hipStream_t stream)
{
    gdp_key_labels_kernel<<<dim3((unsigned)max_K, (unsigned)n), THREADS, sizeof(Shared), stream>>>(inst);
    return hipGetLastError();
}
