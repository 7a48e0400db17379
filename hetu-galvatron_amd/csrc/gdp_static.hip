// gdp_solve_static: one DP instance solved without obtaining any memory.
//
// Every other compute entry point of the library gets device memory for its cost buffers, argmin
// table, layer records and results (hipMalloc, or an allocation kept from an earlier plan), a stream,
// events and page-locked host memory.  Some callers may do none of that: tight serving loops that must
// not touch the allocator, harnesses that forbid it.  (It is no call for a process in which a stream is
// being captured in the global capture mode: synchronous copies and null-stream launches are prohibited
// then.)  For them this entry point keeps all of its device-side working
// memory in ONE file-scope device array of GDP_STATIC_SCRATCH_BYTES, builds the device layout of the
// inputs in a fixed host array, runs on the null stream with synchronous copies, and calls no
// hipMalloc / hipFree / hipHostMalloc / stream or event creation and no host allocator.
//
// An instance that has the form is solved by bounds and the DP over what they leave (gdp_bounds.hip, gdp_frontier.hip).  Any
// other, and what stays of one that is left with too many labels, by the kernels of the other entry points in the layout
// that needs the least memory: two cost buffers used in turn plus the one-byte argmin table (what GDP_KEEP_MARKS selects), one
// launch per layer, every cell computed.  Results are the same bits as gdp_solve's.
//
// The array is per process and per device (every device the library's code object is loaded on holds
// its own copy at its own address) and keeps the contents of the last call; a call rewrites everything
// it reads (pads, zeros of the initial costs, tables), so nothing of an earlier call is ever read.  Calls
// take a process-wide lock for their whole duration: two of them never work in the array at once.
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "gdp_bounds.h"
#include "gdp_host.h"
#include "gdp_kernels.h"

// Device working memory of gdp_solve_static.  In host code this name is only a handle for
// hipGetSymbolAddress; the address the kernels get is the one that call returns (scratch_of_device).
static __device__ __align__(256) unsigned char scratch[GDP_STATIC_SCRATCH_BYTES];

namespace {

constexpr int MAX_DEVICES = 64;
std::mutex g_mu;                       // one call at a time: the arrays below and `scratch` are shared
unsigned char *g_scratch_ptr[MAX_DEVICES];  // device address of `scratch` on device d, once asked for

// Host side: the device layout of the inputs is built here and uploaded in one copy; the results are
// copied back into it.
constexpr size_t STAGE_BYTES = (size_t)8 << 20;
alignas(256) unsigned char g_stage[STAGE_BYTES];

// What stays of an instance: the marks that the device found, and the smaller instance they leave.
uint8_t g_keep[GDP_BOUND_MAX_LS];
constexpr size_t KEPT_BYTES = (size_t)4 << 20;
alignas(256) unsigned char g_kept[KEPT_BYTES];

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// The address of `scratch` on the current device; asked for once per device, with that device current.
int scratch_of_device(unsigned char **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return gdp_fail_hip(e, "hipGetDevice");
    if (dev < 0 || dev >= MAX_DEVICES) return gdp_fail(GDP_E_HIP, "gdp_solve_static: device index above 63");
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return gdp_fail_hip(e, "hipGetSymbolAddress(scratch)");
        if (!p) return gdp_fail(GDP_E_HIP, "hipGetSymbolAddress(scratch) returned a null address");
        g_scratch_ptr[dev] = static_cast<unsigned char *>(p);
    }
    *out = g_scratch_ptr[dev];
    return GDP_OK;
}

struct Layout {
    int L, V, S, T, n_key, ts, variant, SP, SU, rows, P, ntile;
    int64_t ld, ldm;
    size_t off_inst, off_keys, off_lay, off_inter, off_intra, off_index, off_roff, off_mem, off_zcols, small_bytes;
    bool has_zero;
    size_t off_out, off_res, back_bytes, off_H, off_M, total_bytes;
};

// Strategies of S in register tiles of those built with the argmin table (11 or 8 wide, 64 rows): the least padding, then the
// wider one.
int padded(int S) { return (int)std::min(align_up((size_t)S, 11), align_up((size_t)S, 8)); }

// Shapes and offsets (bytes from the start of `scratch`); the same rules as a plan laid out with
// GDP_KEEP_MARKS and one launch per layer.
void lay_out(const gdp_problem *p, Layout *y)
{
    y->L = p->L; y->V = p->V; y->S = p->S;
    y->T = p->inter_index ? p->n_inter : p->L;
    y->n_key = p->n_key;
    y->SP = padded(p->S);
    y->ts = y->SP % 11 == 0 ? 11 : 8;
    y->variant = gdp_find_variant(y->ts, 1);
    y->SU = (int)align_up((size_t)p->S, GDP_SRC_UNROLL);
    y->rows = y->SU + GDP_SRC_PAD;
    int maxm = 1;
    y->has_zero = false;
    for (size_t k = 0; k < (size_t)p->L * p->S; ++k) {
        if (p->mem[k] < p->V) maxm = std::max(maxm, p->mem[k]);
        if (p->mem[k] == 0) y->has_zero = true;
    }
    y->P = (int)align_up((size_t)maxm, 64);
    y->ntile = (p->V + 63) / 64;
    y->ldm = (int64_t)align_up((size_t)y->ntile * 64, 256);
    y->ld = y->P + y->ldm;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t o = off;
        off = align_up(off + bytes, 256);
        return o;
    };
    y->off_inst = take(sizeof(GdpDevInst));
    y->off_keys = take(sizeof(GdpDevKey) * (size_t)std::max(y->n_key, 1));
    y->off_lay = take(sizeof(GdpDevLayer) * (size_t)y->L);
    y->off_inter = take(sizeof(double) * (size_t)y->T * y->rows * y->SP);
    y->off_intra = take(sizeof(double) * (size_t)y->L * y->SP);
    y->off_index = take(sizeof(int32_t) * (size_t)y->L);
    y->off_roff = take(sizeof(int64_t) * (size_t)(y->L + 1) * y->rows);
    y->off_mem = take(sizeof(int32_t) * (size_t)y->L * y->S);
    y->off_zcols = y->has_zero ? take(sizeof(int32_t) * (size_t)y->L * (size_t)(y->S + 1)) : 0;
    y->small_bytes = off;
    y->off_out = take(sizeof(GdpDevOut) * (size_t)std::max(y->n_key, 1));
    y->off_res = take(sizeof(int32_t) * std::max<size_t>((size_t)y->n_key * y->L, 1));
    y->back_bytes = off - y->off_out;
    y->off_H = take(sizeof(double) * 2 * (size_t)(y->S + 1) * (size_t)y->ld);
    y->off_M = take((size_t)y->L * y->S * (size_t)y->ldm);
    y->total_bytes = off;
}

// The device layout of the inputs, written into g_stage; `base` is the device address of `scratch`.
void build(const gdp_problem *p, const Layout &y, unsigned char *base)
{
    memset(g_stage, 0, y.small_bytes);
    GdpDevInst &d = *reinterpret_cast<GdpDevInst *>(g_stage + y.off_inst);
    d.H = reinterpret_cast<double *>(base + y.off_H);
    d.hstride = (int64_t)(y.S + 1) * y.ld;
    d.M = base + y.off_M;
    d.inter = reinterpret_cast<const double *>(base + y.off_inter);
    d.intra = reinterpret_cast<const double *>(base + y.off_intra);
    d.inter_index = reinterpret_cast<const int32_t *>(base + y.off_index);
    d.roff = reinterpret_cast<const int64_t *>(base + y.off_roff);
    d.mem = reinterpret_cast<const int32_t *>(base + y.off_mem);
    d.ld = y.ld; d.ldm = y.ldm;
    d.L = y.L; d.V = y.V; d.S = y.S; d.SP = y.SP; d.SU = y.SU; d.P = y.P; d.ntile = y.ntile;
    d.nbuf = 2;
    // transition matrices [T][rows][SP] and intra [L][SP], zero padded
    double *it = reinterpret_cast<double *>(g_stage + y.off_inter);
    for (int t = 0; t < y.T; ++t)
        for (int a = 0; a < y.S; ++a)
            memcpy(it + ((size_t)t * y.rows + a) * y.SP, p->inter + ((size_t)t * y.S + a) * y.S,
                   sizeof(double) * (size_t)y.S);
    double *ia = reinterpret_cast<double *>(g_stage + y.off_intra);
    for (int l = 0; l < y.L; ++l) memcpy(ia + (size_t)l * y.SP, p->intra + (size_t)l * y.S, sizeof(double) * (size_t)y.S);
    int32_t *ix = reinterpret_cast<int32_t *>(g_stage + y.off_index);
    for (int l = 0; l < y.L; ++l) ix[l] = p->inter_index ? p->inter_index[l] : l;
    memcpy(g_stage + y.off_mem, p->mem, sizeof(int32_t) * (size_t)y.L * y.S);
    d.zcols = nullptr;
    if (y.has_zero) {   // per layer: {n, the n strategies whose memory cost is 0} (see gdp_launch_zero_pass)
        d.zcols = reinterpret_cast<const int32_t *>(base + y.off_zcols);
        int32_t *z = reinterpret_cast<int32_t *>(g_stage + y.off_zcols);
        for (int l = 0; l < y.L; ++l) {
            int32_t *row = z + (size_t)l * (y.S + 1);
            row[0] = 0;
            for (int s = 0; s < y.S; ++s)
                if (p->mem[(size_t)l * y.S + s] == 0) row[++row[0]] = s;
        }
    }
    // roff[l][s']: element offset, from the base of a cost buffer, of "f after layer l-1, strategy s', row 0";
    // a strategy whose memory cost reaches V, and every padding source, reads the +inf row
    int64_t *ro = reinterpret_cast<int64_t *>(g_stage + y.off_roff);
    const int64_t inf_row = (int64_t)y.S * y.ld + y.P;
    for (int l = 0; l <= y.L; ++l) {
        int64_t *row = ro + (size_t)l * y.rows;
        for (int s = 0; s < y.S; ++s) {
            if (l == 0) {
                row[s] = (int64_t)s * y.ld + y.P;
            } else {
                const int m = p->mem[(size_t)(l - 1) * y.S + s];
                row[s] = (m >= y.V) ? inf_row : (int64_t)s * y.ld + y.P - m;
            }
        }
        for (int s = y.S; s < y.rows; ++s) row[s] = inf_row;
    }
    GdpDevLayer *lay = reinterpret_cast<GdpDevLayer *>(g_stage + y.off_lay);
    for (int l = 0; l < y.L; ++l) {
        GdpDevLayer &r = lay[l];
        int maxm = 0;
        for (int s = 0; s < y.S; ++s) {
            const int m = p->mem[(size_t)l * y.S + s];
            if (m < y.V) maxm = std::max(maxm, m);
        }
        const int mat = p->inter_index ? p->inter_index[l] : l;
        r.src = d.H + (int64_t)(l % 2) * d.hstride;
        r.dst = d.H + (int64_t)((l + 1) % 2) * d.hstride + y.P;
        r.ro = d.roff + (int64_t)l * y.rows;
        memcpy(r.ro_head, ro + (size_t)l * y.rows, sizeof(r.ro_head));
        r.it = d.inter + (int64_t)mat * y.rows * y.SP;
        r.ia = d.intra + (int64_t)l * y.SP;
        r.m = d.M + (int64_t)l * y.S * y.ldm;
        r.ld = y.ld; r.ldm = y.ldm;
        r.S = y.S; r.SU = y.SU; r.SP = y.SP; r.ntile = y.ntile;
        r.dep = (maxm + 63) / 64;
        r.lo = 0;               // every tile is computed
        r.hi = y.ntile - 1;
    }
    GdpDevKey *keys = reinterpret_cast<GdpDevKey *>(g_stage + y.off_keys);
    for (int k = 0; k < y.n_key; ++k) {
        keys[k].other_mem = p->other_mem[k];
        keys[k].other_time = p->other_time[k];
        keys[k].inst = 0;
        keys[k].res_off = k * y.L;
    }
}

double work(const gdp_problem *p) { return (double)p->L * p->V * (double)p->S * p->S; }

// What the dense recurrence takes: one launch per layer, 4 us and 0.35 for each strategy in turn (V = 5437, S = 9 7.3 us,
// V = 18405, S = 26 13.3, V = 12602, S = 41 20).
double dense_ns(int L, int S) { return L * (4000.0 + 350.0 * S); }

// Where the arrays of the bounds lie from the start of `scratch`.  alone: with a workgroup for every key.
struct BoundLayout {
    int NL;
    size_t off_inst, off_matrices, off_mem, off_intra, off_inter, off_index, off_lam, off_budget, off_other_time, up_bytes;   // what is uploaded
    size_t off_out, off_res, back_bytes;   // what is copied back
    size_t off_keep, off_marks, off_inter_f, off_inter_t, off_P, off_Q, off_P_mem, off_Q_mem, off_end, off_best, off_ub, off_hist, off_turns, off_hist_mem,
        off_hist_intra, bytes, labels;
};

BoundLayout bound_layout(const gdp_problem *p, int matrices, int multipliers, bool alone)
{
    const size_t L = (size_t)p->L, K = (size_t)p->n_key, T = (size_t)matrices, NL = (size_t)multipliers, LS = L * p->S, SS = (size_t)p->S * p->S,
                 keys = alone ? K : 1;
    BoundLayout y;
    y.NL = multipliers;
    y.labels = L * (alone ? GDP_KEY_LABELS : GDP_FRONTIER_LABELS);
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t o = off;
        off = align_up(off + bytes, 256);
        return o;
    };
    y.off_inst = take(sizeof(GdpBoundInst));
    y.off_matrices = take(sizeof(GdpBoundMatrix) * T);
    y.off_mem = take(4 * LS);
    y.off_intra = take(8 * LS);
    y.off_inter = take(8 * SS * T);
    y.off_index = take(4 * L);
    y.off_lam = take(8 * NL);
    y.off_budget = take(8 * K);
    y.off_other_time = take(8 * K);
    y.up_bytes = off;
    y.off_out = take(sizeof(GdpFrontierOut));
    y.off_res = take(4 * K * L);
    y.back_bytes = off - y.up_bytes;
    y.off_keep = take(LS);
    y.off_marks = take(16 * K * L);
    y.off_inter_f = take(8 * SS * T);
    y.off_inter_t = take(8 * SS * T);
    y.off_P = take(8 * LS * NL);
    y.off_Q = take(8 * LS * NL);
    y.off_P_mem = take(4 * LS * NL);
    y.off_Q_mem = take(4 * LS * NL);
    y.off_end = take(8 * NL);
    y.off_best = take(4 * K);
    y.off_ub = take(8 * K);
    y.off_hist = take(sizeof(GdpFrontierLabel) * y.labels * keys);
    y.off_turns = take(alone ? 0 : 8 * y.labels);
    y.off_hist_mem = take(4 * GDP_FRONTIER_KEPT);
    y.off_hist_intra = take(8 * GDP_FRONTIER_KEPT);
    y.bytes = off;
    return y;
}

// Solves p by bounds if that is possible: *done.  Initial costs are zeros.  *marked: that is left to the dense recurrence, and
// g_keep says which strategies can matter to it.
int solve_by_bounds(const gdp_problem *p, double magnitude, unsigned char *base, gdp_result *r, bool *done, bool *marked)
{
    *done = *marked = false;
    bool forced = false;
    if (!bounds::allowed(&forced)) return GDP_OK;
    gdp_problem form = *p;
    form.flags = p->flags & GDP_COMPUTE_ALL;   // (the others are ignored)
    const int L = p->L, S = p->S, K = p->n_key, T = p->inter_index ? p->n_inter : p->L;
    if (!bounds::has_form(&form) || !(magnitude < 1e100)) return GDP_OK;
    // The bounds take 35 us at least (L = 5: S = 8 58 us whole, 60 with them, S = 11 79 and 60).
    if (dense_ns(L, S) < 36e3 && !forced) return GDP_OK;
    // (Calls of more keys have one workgroup for all of them.  21 of 5 keys would take 0.84 of their time with a workgroup each; that some
    // of 5, 6 and 8 are given up, or not, where the shared workgroup does is held by tests, no limit of the other kernel.)
    constexpr int MOST_ALONE = 4;
    int64_t budget[GDP_BOUND_MAX_KEY], least = 0;
    for (int l = 0; l < L; ++l) {
        int32_t m = INT32_MAX;
        for (int s = 0; s < S; ++s) m = std::min(m, p->mem[(size_t)l * S + s]);
        if (m == 0) return GDP_OK;
        least += m;
    }
    bool any = false;
    for (int k = 0; k < K; ++k) {
        const int64_t b = (int64_t)p->V - 1 - p->other_mem[k];
        budget[k] = b >= least ? b : -1;
        any = any || b >= least;
    }
    if (!any) return GDP_OK;
    const bool may = K <= MOST_ALONE && L <= GDP_KEY_LABELS_MAX_L;
    const double undominated = may ? bounds::undominated(p) : 1.0;
    const bool alone = may && undominated <= GDP_KEY_LABELS_MOST;
    BoundLayout y = bound_layout(p, T, alone ? bounds::key_multipliers(p, undominated) : 64, alone);
    // Where 128 multipliers do not fit into the workspace 64 do (L = 128, S = 128, 4 keys, 40 matrices: 70.6 MB, 45.4;
    // dense 4.9 ms, by these bounds 1.15).
    if (y.bytes > (size_t)GDP_STATIC_SCRATCH_BYTES && y.NL > 64) y = bound_layout(p, T, 64, alone);
    if (y.bytes > (size_t)GDP_STATIC_SCRATCH_BYTES || y.up_bytes > STAGE_BYTES || y.back_bytes > STAGE_BYTES) return GDP_OK;
    const size_t NL = (size_t)y.NL, LS = (size_t)L * S, SS = (size_t)S * S;
    memcpy(g_stage + y.off_mem, p->mem, 4 * LS);
    memcpy(g_stage + y.off_intra, p->intra, 8 * LS);
    memcpy(g_stage + y.off_inter, p->inter, 8 * SS * (size_t)T);
    int32_t *index = reinterpret_cast<int32_t *>(g_stage + y.off_index);
    int changes = 0;
    for (int l = 0; l < L; ++l) {
        index[l] = p->inter_index ? p->inter_index[l] : l;
        changes += l > 0 && index[l] != index[l - 1];
    }
    bounds::multipliers(p, (int)NL, reinterpret_cast<double *>(g_stage + y.off_lam));
    memcpy(g_stage + y.off_budget, budget, 8 * (size_t)K);
    memcpy(g_stage + y.off_other_time, p->other_time, 8 * (size_t)K);
    GdpBoundMatrix *matrices = reinterpret_cast<GdpBoundMatrix *>(g_stage + y.off_matrices);
    for (int t = 0; t < T; ++t)
        matrices[t] = {reinterpret_cast<const double *>(base + y.off_inter) + SS * (size_t)t, reinterpret_cast<double *>(base + y.off_inter_f) + SS * (size_t)t,
                       reinterpret_cast<double *>(base + y.off_inter_t) + SS * (size_t)t, S, 0};
    GdpBoundInst b;
    memset(&b, 0, sizeof b);
    b.mem = reinterpret_cast<const int32_t *>(base + y.off_mem);
    b.intra = reinterpret_cast<const double *>(base + y.off_intra);
    b.inter_f = reinterpret_cast<double *>(base + y.off_inter_f);
    b.inter_t = reinterpret_cast<double *>(base + y.off_inter_t);
    b.index = reinterpret_cast<const int32_t *>(base + y.off_index);
    b.lam = reinterpret_cast<const double *>(base + y.off_lam);
    b.budget = reinterpret_cast<const int64_t *>(base + y.off_budget);
    b.P = reinterpret_cast<double *>(base + y.off_P);
    b.Q = reinterpret_cast<double *>(base + y.off_Q);
    b.P_mem = reinterpret_cast<uint32_t *>(base + y.off_P_mem);
    b.Q_mem = reinterpret_cast<uint32_t *>(base + y.off_Q_mem);
    b.end = reinterpret_cast<double *>(base + y.off_end);
    b.ub = reinterpret_cast<unsigned long long *>(base + y.off_ub);
    b.best = reinterpret_cast<int32_t *>(base + y.off_best);
    b.keep = base + y.off_keep;
    b.marks = reinterpret_cast<unsigned long long *>(base + y.off_marks);
    b.other_time = reinterpret_cast<const double *>(base + y.off_other_time);
    b.hist = reinterpret_cast<GdpFrontierLabel *>(base + y.off_hist);
    b.hist_mem = reinterpret_cast<int32_t *>(base + y.off_hist_mem);
    b.hist_turns = reinterpret_cast<double *>(base + y.off_turns);
    b.hist_intra = reinterpret_cast<double *>(base + y.off_hist_intra);
    b.out = reinterpret_cast<GdpFrontierOut *>(base + y.off_out);
    b.res = reinterpret_cast<int32_t *>(base + y.off_res);
    b.magnitude = magnitude;
    // Half of it for keys with a workgroup each, whose account (gdp_key_labels.hip) says what is ahead but not the bounds behind them: 75 random
    // calls 10.2 ms dense or by the shared workgroup, 8.5 with the whole, 2 of them more than 5 % slower than before, the worst 1.58; 8.3
    // with half, none; 8.7 with 0.3, one 2.5.
    b.limit = (alone ? 0.5 : 1.0) * dense_ns(L, S);
    b.L = L; b.V = p->V; b.S = S; b.K = K; b.T = T;
    b.n_hist = b.n_hist_turns = (int32_t)y.labels;
    b.n_lam = (int32_t)NL;
    memcpy(g_stage + y.off_inst, &b, sizeof b);
    hipStream_t stream = nullptr;
    hipError_t e = hipMemcpy(base, g_stage, y.up_bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) return gdp_fail_hip(e, "gdp_solve_static: upload");
    const GdpBoundInst *inst = reinterpret_cast<const GdpBoundInst *>(base + y.off_inst);
    e = bounds::lay_out({reinterpret_cast<const GdpBoundMatrix *>(base + y.off_matrices), T, nullptr, nullptr, 0}, S, stream);
    if (e == hipSuccess) e = bounds::launch(inst, 1, (int)NL, (int)LS, L * ((S + 63) / 64), S, K, changes * 4 <= L, stream);
    if (e == hipSuccess) e = alone ? bounds::launch_key_labels(inst, 1, K, stream) : bounds::launch_labels(inst, 1, K, stream);
    if (e != hipSuccess) {
        (void)hipDeviceSynchronize();
        return gdp_fail_hip(e, "gdp_solve_static: kernel launch");
    }
    e = hipMemcpy(g_stage, base + y.off_out, y.back_bytes, hipMemcpyDeviceToHost);   // after the kernels, in stream order
    if (e != hipSuccess) return gdp_fail_hip(e, "gdp_solve_static: download");
    const GdpFrontierOut *out = reinterpret_cast<const GdpFrontierOut *>(g_stage);
    const int status = bounds::status_of(*out, K);
    if (status > 1) {
        e = hipMemcpy(g_keep, base + y.off_keep, LS, hipMemcpyDeviceToHost);
        if (e != hipSuccess) return gdp_fail_hip(e, "gdp_solve_static: download");
        *marked = true;
    }
    if (status != 0) return GDP_OK;
    const int32_t *res = reinterpret_cast<const int32_t *>(g_stage + (y.off_res - y.off_out));
    for (int k = 0; k < K; ++k) {
        r->total[k] = out->total[k];
        r->remaining[k] = out->remaining[k];
        if (out->remaining[k] >= 0) memcpy(r->res + (size_t)k * L, res + (size_t)k * L, sizeof(int32_t) * (size_t)L);
    }
    stats::count(work(p), bounds::executed_of(*out, K));
    *done = true;
    return GDP_OK;
}

// What stays of p (g_keep) as an instance of its own in g_kept, and its layout; false where it would not be a good deal
// smaller, or does not fit.  (L = 27, S = 37, V = 20011, two kinds of layers that trade memory for time, calls left with too
// many labels, us: without bounds 541; after them whole 642 to 790, what stays 360 to 480.)
bool lay_out_kept(const gdp_problem *p, const Layout &whole, gdp_problem *small, Layout *y)
{
    int most = 0;
    for (int l = 0; l < p->L; ++l) {
        int n = 0;
        for (int s = 0; s < p->S; ++s) n += g_keep[(size_t)l * p->S + s] != 0;
        if (n == 0) return false;
        most = std::max(most, n);
    }
    const int R = most;
    if (!(dense_ns(p->L, padded(R)) < 0.85 * dense_ns(p->L, whole.SP))) return false;
    const size_t LR = (size_t)p->L * R;
    const size_t off_mem = align_up(4 * LR, 256), off_intra = off_mem + align_up(4 * LR, 256), off_inter = off_intra + align_up(8 * LR, 256),
                 bytes = off_inter + 8 * LR * (size_t)R;
    if (bytes > KEPT_BYTES) return false;
    int32_t *kept = reinterpret_cast<int32_t *>(g_kept), *mem = reinterpret_cast<int32_t *>(g_kept + off_mem);
    double *intra = reinterpret_cast<double *>(g_kept + off_intra), *inter = reinterpret_cast<double *>(g_kept + off_inter);
    std::fill(intra, intra + LR, INFINITY);
    std::fill(inter, inter + LR * (size_t)R, 0.0);
    bounds::fill_kept(p, g_keep, R, [&](int l) { return p->inter + (size_t)(p->inter_index ? p->inter_index[l] : l) * p->S * p->S; }, nullptr, kept,
                      mem, intra, inter);
    *small = *p;
    small->S = R;
    small->mem = mem;
    small->intra = intra;
    small->inter = inter;
    small->inter_index = nullptr;
    small->n_inter = p->L;
    lay_out(small, y);
    return y->variant >= 0 && y->total_bytes <= (size_t)GDP_STATIC_SCRATCH_BYTES && y->small_bytes <= STAGE_BYTES && y->back_bytes <= STAGE_BYTES;
}

// The dense recurrence.  kept: what to say for a strategy of a layer ([L][S] of p), null: itself.
int solve_dense(const gdp_problem *p, const Layout &y, unsigned char *base, bool f0_live, const int32_t *kept, gdp_result *r)
{
    build(p, y, base);
    hipStream_t stream = nullptr;  // the null stream: nothing is created
    hipError_t e = hipMemcpy(base, g_stage, y.small_bytes, hipMemcpyHostToDevice);
    if (e != hipSuccess) return gdp_fail_hip(e, "gdp_solve_static: upload");
    const GdpDevInst *d_inst = reinterpret_cast<const GdpDevInst *>(base + y.off_inst);
    const GdpDevLayer *d_lay = reinterpret_cast<const GdpDevLayer *>(base + y.off_lay);
    // +inf pads and +inf row of both cost buffers, zeros in the first one (the caller's initial f): whatever
    // the last call left there is overwritten before anything reads it
    e = gdp_launch_init(d_inst, 1, y.ld, y.S, d_lay, y.L, 64, GDP_INIT_PADS | GDP_INIT_ZERO, stream);
    if (e == hipSuccess && f0_live) {
        // The caller's initial costs [V][S] into buffer 0, one row per strategy: turned round in the host
        // array a slice of budget rows at a time (the tables it held are on the device by now; the copies
        // are synchronous and follow the launch above in stream order).
        double *stage = reinterpret_cast<double *>(g_stage);
        double *h0 = reinterpret_cast<double *>(base + y.off_H) + y.P;
        const int slice = (int)std::max<size_t>(1, STAGE_BYTES / (sizeof(double) * (size_t)y.S));
        for (int v0 = 0; v0 < y.V && e == hipSuccess; v0 += slice) {
            const int nv = std::min(slice, y.V - v0);
            for (int v = 0; v < nv; ++v)
                for (int s = 0; s < y.S; ++s) stage[(size_t)s * nv + v] = p->f0[(size_t)(v0 + v) * y.S + s];
            e = hipMemcpy2D(h0 + v0, sizeof(double) * (size_t)y.ld, stage, sizeof(double) * (size_t)nv,
                            sizeof(double) * (size_t)nv, (size_t)y.S, hipMemcpyHostToDevice);
        }
    }
    for (int l = 0; l < y.L && e == hipSuccess; ++l) {
        e = gdp_launch_relax(y.variant, true, 0, d_lay, y.L, 1, y.ntile, y.SP, l, stream);
        if (e == hipSuccess && y.has_zero) e = gdp_launch_zero_pass(true, d_inst, d_lay, y.L, 64, 1, y.V, l, stream);
    }
    if (e == hipSuccess)
        e = gdp_launch_epilogue(true, d_inst, reinterpret_cast<const GdpDevKey *>(base + y.off_keys), y.n_key,
                                reinterpret_cast<GdpDevOut *>(base + y.off_out),
                                reinterpret_cast<int32_t *>(base + y.off_res), nullptr, nullptr, stream);
    if (e != hipSuccess) {
        (void)hipDeviceSynchronize();
        return gdp_fail_hip(e, "gdp_solve_static: kernel launch");
    }
    e = hipMemcpy(g_stage, base + y.off_out, y.back_bytes, hipMemcpyDeviceToHost);  // after the kernels, in stream order
    if (e != hipSuccess) return gdp_fail_hip(e, "gdp_solve_static: download");
    const GdpDevOut *out = reinterpret_cast<const GdpDevOut *>(g_stage);
    const int32_t *res = reinterpret_cast<const int32_t *>(g_stage + (y.off_res - y.off_out));
    for (int k = 0; k < y.n_key; ++k) {
        r->total[k] = out[k].total;
        r->remaining[k] = out[k].remaining;
        if (!out[k].feasible) continue;
        memcpy(r->res + (size_t)k * y.L, res + (size_t)k * y.L, sizeof(int32_t) * (size_t)y.L);
        for (int l = 0; kept && l < y.L; ++l) {
            int32_t &strategy = r->res[(size_t)k * y.L + l];
            strategy = kept[(size_t)l * y.S + strategy];
        }
    }
    return GDP_OK;
}

}  // namespace

extern "C" int gdp_solve_static(const gdp_problem *p, gdp_result *r)
{
    gdp_clear_error();
    if (!p || !r) return gdp_fail(GDP_E_BADARG, "null problem or result");
    bool f0_live = false;
    double magnitude = 0;
    int rc = gdp_validate(p, 0, &magnitude);
    if (rc == GDP_OK) rc = gdp_validate_f0(p, 0, &f0_live);
    if (rc != GDP_OK) return rc;
    if (p->flags & (GDP_EXPORT_F | GDP_EXPORT_MARK))
        return gdp_fail(GDP_E_BADARG, "gdp_solve_static does not export f / mark");
    if (p->S > GDP_MAX_S_MARKS) return gdp_fail(GDP_E_BADARG, "gdp_solve_static: S exceeds GDP_MAX_S_MARKS");
    if (p->n_key > 0 && (!r->total || !r->remaining || !r->res)) return gdp_fail(GDP_E_BADARG, "null result array");
    Layout y;
    lay_out(p, &y);
    if (y.variant < 0) return gdp_fail(GDP_E_HIP, "gdp_solve_static: register tile not built");
    if (y.total_bytes > (size_t)GDP_STATIC_SCRATCH_BYTES || y.small_bytes > STAGE_BYTES || y.back_bytes > STAGE_BYTES) {
        char buf[256];
        snprintf(buf, sizeof buf,
                 "gdp_solve_static: this instance needs %zu bytes of device working memory (tables %zu, results %zu); "
                 "the static array holds %zu (tables and results up to %zu each): use gdp_solve",
                 y.total_bytes, y.small_bytes, y.back_bytes, (size_t)GDP_STATIC_SCRATCH_BYTES, STAGE_BYTES);
        return gdp_fail(GDP_E_NOMEM, buf);
    }
    std::lock_guard<std::mutex> lk(g_mu);
    unsigned char *base = nullptr;
    const int rs = scratch_of_device(&base);
    if (rs != GDP_OK) return rs;
    bool marked = false;
    if (!f0_live) {
        bool done = false;
        const int rb = solve_by_bounds(p, magnitude, base, r, &done, &marked);
        if (rb != GDP_OK || done) return rb;
    }
    gdp_problem small;
    Layout ys;
    const bool less = marked && lay_out_kept(p, y, &small, &ys);
    rc = less ? solve_dense(&small, ys, base, false, reinterpret_cast<const int32_t *>(g_kept), r) : solve_dense(p, y, base, f0_live, nullptr, r);
    if (rc == GDP_OK) stats::count(work(p), work(less ? &small : p));
    return rc;
}
