// Runtime of the serial CPU emulation of the kernels: the lanes of a workgroup
// are fibers of one thread, one workgroup at a time; __syncthreads is a barrier
// over the workgroup's lanes and a ballot a rendezvous of the wave's lanes.
// Lanes run from one rendezvous to the next in an order that changes each time,
// so that what one leaves to another without a rendezvous is met in either
// order.  At the end of every workgroup each lane must have passed the same
// number of barriers (and each wave's lanes the same number of ballots), and
// lanes that wait for each other in a circle end the run: both abort naming the
// sub-task (ticket) that was running.
#include "hip/hip_runtime.h"
#include <chrono>
#include <cstdio>
#include <deque>
#include <sanitizer/common_interface_defs.h>
#include <sys/mman.h>
#include <vector>

thread_local dim3 threadIdx, blockIdx;
dim3 blockDim, gridDim;

constexpr size_t STACK = 1 << 20;
struct Lane {
    void *sp = nullptr;      // saved stack pointer while switched out
    char *stack = nullptr;
    void *fake = nullptr;
    dim3 idx;
    uint64_t barriers = 0, ballots = 0;
};
static Lane g_lane[1024];
static int g_made = 0, g_nl = 0, g_live = 0, t_lane = -1;
static std::deque<int> g_ready;
static void *g_main_sp, *g_main_fake;
static const void *g_main_bottom;
static size_t g_main_size;
static const std::function<void()> *g_body = nullptr;
static dim3 g_bid;
static unsigned char *g_smem = nullptr;
volatile uint64_t emu_ticket = ~0ull;

// saves the callee's registers on this stack and goes on from another
extern "C" void emu_switch(void **from, void *to);
asm(".text\n.globl emu_switch\nemu_switch:\n"
    "  push %rbp\n  push %rbx\n  push %r12\n  push %r13\n  push %r14\n  push %r15\n"
    "  mov %rsp, (%rdi)\n  mov %rsi, %rsp\n"
    "  pop %r15\n  pop %r14\n  pop %r13\n  pop %r12\n  pop %rbx\n  pop %rbp\n  ret\n");

// from lane `me` (-1: the launching thread) to lane `to`
static void go(int me, int to) {
    if (me == to) return;
    void **fake = me < 0 ? &g_main_fake : &g_lane[me].fake;
    if (to < 0) __sanitizer_start_switch_fiber(fake, g_main_bottom, g_main_size);
    else __sanitizer_start_switch_fiber(fake, g_lane[to].stack, STACK);
    t_lane = to;
    if (to >= 0) {
        threadIdx = g_lane[to].idx;
        blockIdx = g_bid;
    }
    emu_switch(me < 0 ? &g_main_sp : &g_lane[me].sp, to < 0 ? g_main_sp : g_lane[to].sp);
    __sanitizer_finish_switch_fiber(*fake, nullptr, nullptr);
}

// the next lane that can run, or the launching thread once none is left
static void next_lane() {
    const int me = t_lane;
    if (g_ready.empty()) {
        if (g_live) {
            fprintf(stderr, "EMU: lanes wait for each other in block (%u,%u) (ticket %llu)\n",
                    g_bid.x, g_bid.y, (unsigned long long)emu_ticket);
            abort();
        }
        go(me, -1);
        return;
    }
    const int to = g_ready.front();
    g_ready.pop_front();
    go(me, to);
}

// a rendezvous of the lanes [first, first + size)
struct Bar {
    int first = 0, size = 0, expected = 0, arrived = 0;
    uint32_t turn = 0;
    uint64_t acc = 0, result = 0;
    bool waits[1024] = {};
    void reset(int at, int n) {
        first = at;
        size = expected = n;
        arrived = 0;
        acc = 0;
    }
    void release() {
        result = acc;
        acc = 0;
        arrived = 0;
        turn = turn * 1664525u + 1013904223u;
        const int mask = (int)(turn >> 22);
        for (int i = 0; i < 1024; i++) {
            const int l = i ^ mask;
            if (l < size && waits[l]) {
                waits[l] = false;
                g_ready.push_back(first + l);
            }
        }
    }
    uint64_t arrive(uint64_t bits) {
        acc |= bits;
        waits[t_lane - first] = true;
        if (++arrived == expected) release();
        next_lane();
        return result;
    }
    void drop() {
        expected--;
        if (expected > 0 && arrived == expected) release();
    }
};
static Bar g_block, g_wave[16];

void emu_syncthreads() {
    g_lane[t_lane].barriers++;
    g_block.arrive(0);
}
uint64_t emu_ballot(bool p) {
    g_lane[t_lane].ballots++;
    return g_wave[t_lane / 64].arrive(p ? (1ull << (t_lane % 64)) : 0ull);
}
// every lane of a wave posts its value, then reads the lane d below it
static int g_shfl[1024];
int emu_shfl_up(int v, unsigned d) {
    const unsigned l = (unsigned)t_lane % 64;
    g_shfl[t_lane] = v;
    emu_ballot(true);
    const int r = l >= d ? g_shfl[t_lane - d] : v;
    emu_ballot(true);
    return r;
}
int emu_shfl_xor(int v, int m) {
    g_shfl[t_lane] = v;
    emu_ballot(true);
    const int r = g_shfl[t_lane / 64 * 64 + ((t_lane % 64) ^ m)];
    emu_ballot(true);
    return r;
}
// every lane of the wave calls it
int emu_readlane(int v, int lane) {
    g_shfl[t_lane] = v;
    emu_ballot(true);
    const int r = g_shfl[t_lane / 64 * 64 + lane];
    emu_ballot(true);
    return r;
}
void emu_sleep() {
    g_ready.push_back(t_lane);
    next_lane();
}
uint64_t emu_clock() {
    return (uint64_t)std::chrono::duration_cast<std::chrono::nanoseconds>(
               std::chrono::steady_clock::now().time_since_epoch()).count() / 10;
}
unsigned char *emu_smem() { return g_smem; }

static void lane_main() {
    const void *from;
    size_t size;
    __sanitizer_finish_switch_fiber(nullptr, &from, &size);
    if (!g_main_bottom) {   // the first lane of all
        g_main_bottom = from;
        g_main_size = size;
    }
    for (;;) {
        (*g_body)();
        g_wave[t_lane / 64].drop();
        g_block.drop();
        g_live--;
        next_lane();
    }
}

void emu_run_block(dim3 grid, dim3 block, dim3 bid, size_t smem, const std::function<void()> &body) {
    const int nl = (int)(block.x * block.y * block.z);
    if (nl > 1024) { fprintf(stderr, "EMU: block of %d lanes\n", nl); abort(); }
    g_smem = (unsigned char *)malloc(smem ? smem : 1);
    memset(g_smem, 0x5A, smem);
    g_block.reset(0, nl);
    for (int w = 0; w < (nl + 63) / 64; w++) g_wave[w].reset(64 * w, std::min(64, nl - 64 * w));
    for (int l = 0; l < nl; l++) {
        Lane &f = g_lane[l];
        f.idx = dim3(l % block.x, (l / block.x) % block.y, l / (block.x * block.y));
        f.barriers = f.ballots = 0;
    }
    g_bid = bid;
    g_body = &body;
    g_nl = g_live = nl;
    g_ready.clear();
    for (int l = 0; l < nl; l++) g_ready.push_back(l);
    for (; g_made < nl; g_made++) {
        Lane &f = g_lane[g_made];
        f.stack = (char *)mmap(nullptr, STACK, PROT_READ | PROT_WRITE,
                               MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
        if (f.stack == (char *)MAP_FAILED) { fprintf(stderr, "EMU: no stack\n"); abort(); }
        void **top = (void **)(f.stack + STACK) - 1;   // lane_main starts as if called
        *--top = (void *)lane_main;
        for (int r = 0; r < 6; r++) *--top = nullptr;
        f.sp = top;
    }
    next_lane();
    for (int l = 1; l < nl; l++)
        if (g_lane[l].barriers != g_lane[0].barriers) {
            fprintf(stderr, "EMU: barrier count mismatch in block (%u,%u): lane %d %llu vs lane 0 %llu (ticket %llu)\n",
                    bid.x, bid.y, l, (unsigned long long)g_lane[l].barriers,
                    (unsigned long long)g_lane[0].barriers, (unsigned long long)emu_ticket);
            abort();
        }
    for (int l = 0; l < nl; l++)
        if (g_lane[l].ballots != g_lane[(l / 64) * 64].ballots) {
            fprintf(stderr, "EMU: ballot count mismatch in wave %d (ticket %llu)\n", l / 64,
                    (unsigned long long)emu_ticket);
            abort();
        }
    free(g_smem);
    g_smem = nullptr;
}
