// What the kernels of the DP over labels share: gdp_frontier.hip, gdp_key_labels.hip.
#pragma once
#include "gdp_bounds.h"

namespace {

typedef GdpFrontierLabel Label;

typedef const __attribute__((address_space(1))) double *gdouble;
typedef const __attribute__((address_space(1))) int32_t *gint;
typedef const __attribute__((address_space(1))) uint8_t *gbyte;
typedef __attribute__((address_space(1))) double *gout;
typedef __attribute__((address_space(1))) int32_t *giout;
typedef int int4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) int4v *glabel;
#define GLOBAL(type, p) ((type)(uintptr_t)(p))

typedef int int2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ double min_f64(double a, double b)
{
    double r;   // the bare instruction: no operand is a NaN
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

__device__ __forceinline__ double max_f64(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// x of the lane that CTRL names, `other` where there is none.
template <int CTRL, int ROWS>
__device__ __forceinline__ double moved(double other, double x)
{
    const int2v o = __builtin_bit_cast(int2v, other), w = __builtin_bit_cast(int2v, x);
    const int2v m = {__builtin_amdgcn_update_dpp(o.x, w.x, CTRL, ROWS, 0xf, false), __builtin_amdgcn_update_dpp(o.y, w.y, CTRL, ROWS, 0xf, false)};
    return __builtin_bit_cast(double, m);
}

// Minimum over the lanes up to this one, of the first `lanes`.
__device__ __forceinline__ double prefix_min(double x, int lanes = 64)
{
    if (lanes <= 1) return x;
    x = min_f64(x, moved<0x111, 0xf>(x, x));   // row_shr:1, 2, 4, 8; a lane without a source keeps its own
    x = min_f64(x, moved<0x112, 0xf>(x, x));
    x = min_f64(x, moved<0x114, 0xf>(x, x));
    x = min_f64(x, moved<0x118, 0xf>(x, x));
    if (lanes <= 16) return x;
    x = min_f64(x, moved<0x142, 0xa>(x, x));   // row_bcast:15 into rows 1 and 3
    x = min_f64(x, moved<0x143, 0xc>(x, x));   // row_bcast:31 into rows 2 and 3
    return x;
}

__device__ __forceinline__ double lane_of(double x, int lane)
{
    const int2v w = __builtin_bit_cast(int2v, x);
    const int2v r = {__builtin_amdgcn_readlane(w.x, lane), __builtin_amdgcn_readlane(w.y, lane)};
    return __builtin_bit_cast(double, r);
}

__device__ __forceinline__ int lanes_min(int x)
{
    x = min(x, __builtin_amdgcn_update_dpp(x, x, 0x111, 0xf, 0xf, false));
    x = min(x, __builtin_amdgcn_update_dpp(x, x, 0x112, 0xf, 0xf, false));
    x = min(x, __builtin_amdgcn_update_dpp(x, x, 0x114, 0xf, 0xf, false));
    x = min(x, __builtin_amdgcn_update_dpp(x, x, 0x118, 0xf, 0xf, false));
    x = min(x, __builtin_amdgcn_update_dpp(x, x, 0x142, 0xa, 0xf, false));
    x = min(x, __builtin_amdgcn_update_dpp(x, x, 0x143, 0xc, 0xf, false));
    return __builtin_amdgcn_readlane(x, 63);
}

// The lowest (value, strategy) of a wave's first `lanes`, +inf in the others: the cheapest, of those the lowest strategy.
__device__ __forceinline__ void cheapest(double &c, int &s, int lanes)
{
    const double least = lane_of(prefix_min(c, lanes), min(lanes, 64) - 1);
    const unsigned long long at = __builtin_amdgcn_ballot_w64(c == least);
    s = (at & (at - 1)) == 0 ? __builtin_amdgcn_readlane(s, __builtin_ctzll(at)) : lanes_min(c == least ? s : INT32_MAX);
    c = least;
}

// old = *p, *p += n, in LDS, by one lane.
__device__ __forceinline__ int draw(int32_t *p, int n)
{
    int old;
    asm volatile("ds_add_rtn_u32 %0, %1, %2\n\ts_waitcnt lgkmcnt(0)" : "=&v"(old)
                 : "v"((uint32_t)(uintptr_t)(__attribute__((address_space(3))) int32_t *)p), "v"(n) : "memory");
    return old;
}

// All of a label at a time.
__device__ __forceinline__ int4v words(const Label &x) { return __builtin_bit_cast(int4v, x); }
__device__ __forceinline__ Label label_at(const Label *p) { return __builtin_bit_cast(Label, *reinterpret_cast<const int4v *>(p)); }
__device__ __forceinline__ void put(Label *p, const Label &x) { *reinterpret_cast<int4v *>(p) = words(x); }

// The same in every lane, said so.
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ double uniform(double x) { return lane_of(x, 0); }

}  // namespace
