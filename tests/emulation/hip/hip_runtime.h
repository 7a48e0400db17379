// One workgroup of a HIP kernel on the CPU: what the kernel's source uses of the device, for an x86-64 host compiler.  512 threads are
// coroutines; a wave goes on until all its lanes stand at an instruction between lanes or at the barrier, then another one.
// LDS holds garbage at first.  A wave that has ended while another stands at the barrier is an error: on the device the others
// would go on without it.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#define __HIPCC__ 1
#define __host__
#define __device__
#define __global__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(x) alignas(x)
using std::max;
using std::min;
typedef int hipError_t;
typedef void *hipStream_t;
struct int2 { int x, y; };
struct int4 { int x, y, z, w; };
struct double2 { double x, y; };
struct Index { unsigned x, y, z; };
inline int2 make_int2(int a, int b) { return {a, b}; }
inline int4 make_int4(int a, int b, int c, int d) { return {a, b, c, d}; }
inline double2 make_double2(double a, double b) { return {a, b}; }

namespace emu {

constexpr int WAVES = 8, THREADS = 64 * WAVES;
struct Thread {
    void *stack;
    bool done;
    const long *waits_for;   // goes on when that is `until` at least
    long until;
};
inline Thread thread[THREADS];
inline int now;              // the thread that runs
inline Index block;
inline void *scheduler;
inline long wave_turn[WAVES], barrier_turn;
inline int wave_there[WAVES], barrier_there;
inline int64_t between[WAVES][2][64];
inline long group_turn[3][THREADS];
inline int group_there[3][THREADS], group_between[3][THREADS][2];

extern "C" void emu_switch(void **from, void *to);

inline void wait(const long *what, long until)
{
    thread[now].waits_for = what;
    thread[now].until = until;
    emu_switch(&thread[now].stack, scheduler);
}

// What all 64 lanes of the wave bring.
inline const int64_t *exchange(int64_t own)
{
    const int w = now >> 6;
    const long turn = wave_turn[w];
    int64_t *const all = between[w][turn & 1];
    all[now & 63] = own;
    if (++wave_there[w] == 64) {
        wave_there[w] = 0;
        ++wave_turn[w];
    } else {
        wait(&wave_turn[w], turn + 1);
    }
    return all;
}

// The same of groups of 2, 4 or 8 lanes (kind 0, 1, 2), the others of the wave need not be there.
inline int exchange_within(int kind, int own, int with)
{
    const int group = now & ~((2 << kind) - 1), parity = (int)(group_turn[kind][group] & 1);
    const long turn = group_turn[kind][group];
    group_between[kind][now][parity] = own;
    if (++group_there[kind][group] == 2 << kind) {
        group_there[kind][group] = 0;
        ++group_turn[kind][group];
    } else {
        wait(&group_turn[kind][group], turn + 1);
    }
    return group_between[kind][with][parity];
}

inline int update_dpp(int old, int x, int control, int rows, int, bool zero)
{
    const int64_t *const all = exchange(x);
    const int lane = now & 63, row = lane >> 4;
    int source = -1;
    if (control > 0x110 && control < 0x120) source = (lane & 15) >= control - 0x110 ? lane - (control - 0x110) : -1;   // row_shr
    else if (control == 0x130) source = lane < 63 ? lane + 1 : -1;   // wave_shl:1
    else if (control == 0x138) source = lane - 1;                    // wave_shr:1
    else if (control == 0x142) source = 16 * row - 1;                // row_bcast:15
    else if (control == 0x143) source = lane >= 32 ? 31 : -1;        // row_bcast:31
    else abort();
    if (!(rows >> row & 1)) return old;
    return source < 0 ? (zero ? 0 : old) : (int)all[source];
}

inline int mov_dpp(int x, int control)
{
    if (control == 0xb1) return exchange_within(0, x, now ^ 1);
    if (control == 0x4e) return exchange_within(1, x, now ^ 2);
    if (control == 0x141) return exchange_within(2, x, now ^ 7);   // row_half_mirror
    abort();
}

inline unsigned long long ballot(bool x)
{
    const int64_t *const all = exchange(x);
    unsigned long long m = 0;
    for (int lane = 0; lane < 64; ++lane) m |= (unsigned long long)(all[lane] != 0) << lane;
    return m;
}

struct Position {
    int x;
    Position() : x(now) {}
};

}  // namespace emu

#define threadIdx (emu::Position())
#define blockIdx emu::block
#define __builtin_amdgcn_ballot_w64 emu::ballot
#define __builtin_amdgcn_readlane(x, lane) ((int)emu::exchange(x)[(lane) & 63])
#define __builtin_amdgcn_readfirstlane(x) ((int)emu::exchange(x)[0])
#define __builtin_amdgcn_update_dpp emu::update_dpp
#define __builtin_amdgcn_mov_dpp(x, control, rows, banks, zero) emu::mov_dpp(x, control)
#define __builtin_amdgcn_ds_bpermute(at, x) ((int)emu::exchange(x)[(at) >> 2 & 63])
#define __builtin_amdgcn_wave_barrier() ((void)emu::exchange(0))
#define __builtin_amdgcn_alignbit(hi, lo, n) ((uint32_t)(((uint64_t)(hi) << 32 | (lo)) >> ((n) & 31)))
#define __builtin_amdgcn_mbcnt_lo(m, n) ((n) + __builtin_popcountll((uint32_t)(m) & ((1ull << (emu::now & 63)) - 1)))
#define __builtin_amdgcn_mbcnt_hi(m, n) ((n) + __builtin_popcountll((uint64_t)(uint32_t)(m) << 32 & ((1ull << (emu::now & 63)) - 1)))
#define __hip_atomic_load(p, order, scope) (*(p))
#define __hip_atomic_store(p, x, order, scope) (void)(*(p) = (x))

inline void __syncthreads()
{
    const long turn = emu::barrier_turn;
    if (++emu::barrier_there == emu::THREADS) {
        emu::barrier_there = 0;
        ++emu::barrier_turn;
    } else {
        emu::wait(&emu::barrier_turn, turn + 1);
    }
}
inline int atomicAdd(int *p, int n)
{
    const int old = *p;
    *p += n;
    return old;
}
inline int __popc(unsigned x) { return __builtin_popcount(x); }
inline int __popcll(unsigned long long x) { return __builtin_popcountll(x); }
inline double __longlong_as_double(long long x) { return __builtin_bit_cast(double, x); }
