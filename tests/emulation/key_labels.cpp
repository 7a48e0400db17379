// gdp_key_labels_kernel on the CPU: KERNEL is its source as test_key_labels_on_cpu.py prepares it.
#include <hip/hip_runtime.h>

alignas(256) static char emulated_lds[160 * 1024];
#include KERNEL

asm(R"(
.text
.globl emu_switch
emu_switch:
    pushq %rbp
    pushq %rbx
    pushq %r12
    pushq %r13
    pushq %r14
    pushq %r15
    movq %rsp, (%rdi)
    movq %rsi, %rsp
    popq %r15
    popq %r14
    popq %r13
    popq %r12
    popq %rbx
    popq %rbp
    ret
)");

static_assert(emu::THREADS == THREADS && emu::WAVES == WAVES, "a workgroup");

namespace {

using emu::thread;
using emu::now;
using emu::scheduler;
using emu::emu_switch;
constexpr size_t STACK = 64 * 1024;
const GdpBoundInst *instance;

void begin()
{
    gdp_key_labels_kernel(instance);
    thread[now].done = true;
    for (;;) emu_switch(&thread[now].stack, scheduler);
}

}  // namespace

extern "C" {

size_t instance_size() { return sizeof(GdpBoundInst); }
size_t result_size() { return sizeof(GdpFrontierOut); }
int labels_a_layer() { return GDP_KEY_LABELS; }

// Of the workgroup that ran last: the most labels of a layer, strategies that stay, transitions between them.
void seen(int layers, int *most_labels, int *kept, int *transitions)
{
    const Shared &sh = *reinterpret_cast<const Shared *>(emulated_lds);
    *most_labels = *std::max_element(sh.labels_of, sh.labels_of + layers);
    *kept = sh.layer[layers].y;
    *transitions = sh.layer[layers].z;
}

// The workgroup of a key.  order: waves first to last, last to first, or (seed) at random.  From the moment on that `told_at` waves
// have begun another key of the instance says in this one's upper bound that it has been given up (-1: none does).  0: all
// threads have ended; 1: some never would; 2: a wave had left when others met at a barrier.
int run_key(const GdpBoundInst *inst, int key, int order, unsigned seed, int told_at)
{
    static char *const stacks = static_cast<char *>(malloc(STACK * THREADS));
    memset(emulated_lds, 0xa5, sizeof emulated_lds);
    instance = inst;
    emu::block = {(unsigned)key, 0, 0};
    emu::barrier_turn = emu::barrier_there = 0;
    memset(emu::wave_turn, 0, sizeof emu::wave_turn);
    memset(emu::wave_there, 0, sizeof emu::wave_there);
    memset(emu::group_turn, 0, sizeof emu::group_turn);
    memset(emu::group_there, 0, sizeof emu::group_there);
    for (int i = 0; i < THREADS; ++i) {
        void **top = reinterpret_cast<void **>(stacks + STACK * (i + 1));
        *--top = nullptr;
        *--top = reinterpret_cast<void *>(begin);
        for (int k = 0; k < 6; ++k) *--top = nullptr;
        thread[i] = {top, false, nullptr, 0};
    }
    int begun = 0;
    bool has_begun[WAVES] = {};
    for (;;) {
        bool any = false;
        int turn[WAVES], ended = 0, at_barrier = 0;
        for (int w = 0; w < WAVES; ++w) turn[w] = order == 1 ? WAVES - 1 - w : w;
        if (order == 2)
            for (int w = WAVES - 1; w > 0; --w) std::swap(turn[w], turn[rand_r(&seed) % (w + 1)]);
        for (int w : turn) {
            if (!has_begun[w]) {
                has_begun[w] = true;
                if (begun++ == told_at) inst->ub[key] = GIVEN_UP;
            }
            for (bool ran = true; ran;) {
                ran = false;
                for (int i = 64 * w; i < 64 * (w + 1); ++i) {
                    emu::Thread &t = thread[i];
                    if (t.done || (t.waits_for && *t.waits_for < t.until)) continue;
                    t.waits_for = nullptr;
                    now = i;
                    emu_switch(&scheduler, t.stack);
                    ran = any = true;
                }
            }
        }
        for (const emu::Thread &t : thread) {
            ended += t.done;
            at_barrier += !t.done && t.waits_for == &emu::barrier_turn && t.until > emu::barrier_turn;
        }
        if (ended == THREADS) return 0;
        if (ended > 0 && at_barrier > 0) return 2;
        if (!any) return 1;
    }
}

}  // extern "C"
