// The workgroups of hip/hip_runtime.h, one after the other.  A thread is
// started by makecontext and from then on switched by _setjmp / _longjmp,
// which make no system call.
#include <setjmp.h>
#include <sys/mman.h>
#include <ucontext.h>

#include <vector>

#include "hip/hip_runtime.h"

namespace cpu {
dim3 thread_idx, block_idx, block_dim, grid_dim;
char *dynamic_lds;
uint64_t exchange[1024];
std::function<void()> on_yield;

namespace {
enum State { kRuns, kAtBlock, kAtWave, kEnded };
struct Fiber {
    jmp_buf at;
    ucontext_t start;
    bool started;
    State state;
};
constexpr size_t kStack = 128 << 10, kPage = 4096, kGuard = 1 << 20;
std::vector<Fiber> fibers(1024);
char *stacks = nullptr;
jmp_buf scheduler;
unsigned current;
const std::function<void()> *body_now;

void entry() {
    (*body_now)();
    fibers[current].state = kEnded;
    _longjmp(scheduler, 1);
}
void wait_as(State s) {
    Fiber &f = fibers[current];
    f.state = s;
    if (_setjmp(f.at) == 0) _longjmp(scheduler, 1);
}
void run(unsigned t) {
    Fiber &f = fibers[t];
    current = t;
    thread_idx = dim3(t);
    if (_setjmp(scheduler) == 0) {
        if (f.started) _longjmp(f.at, 1);
        f.started = true;
        setcontext(&f.start);
    }
}
// Lets the threads [a, b) go on once all of them that have not ended wait in
// state s; says whether any did.
bool release(unsigned a, unsigned b, State s) {
    bool any = false;
    for (unsigned t = a; t < b; t++) {
        if (fibers[t].state == kEnded) continue;
        if (fibers[t].state != s) return false;
        any = true;
    }
    for (unsigned t = a; any && t < b; t++)
        if (fibers[t].state == s) fibers[t].state = kRuns;
    return any;
}
}  // namespace

void block_wait() { wait_as(kAtBlock); }
void wave_wait() { wait_as(kAtWave); }

void launch(unsigned grid, unsigned block, size_t lds, const std::function<void()> &body) {
    if (!stacks) stacks = static_cast<char *>(std::malloc(kStack * fibers.size()));
    body_now = &body;
    grid_dim = dim3(grid);
    block_dim = dim3(block);
    // Dynamic LDS ends at an inaccessible page and begins after one.
    const size_t size = (lds + kPage - 1) / kPage * kPage;
    char *m = nullptr;
    if (lds) {
        m = static_cast<char *>(mmap(nullptr, size + 2 * kGuard, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
        mprotect(m + kGuard, size, PROT_READ | PROT_WRITE);
        dynamic_lds = m + kGuard + (size - lds);
    }
    for (unsigned b = 0; b < grid; b++) {
        block_idx = dim3(b);
        for (unsigned t = 0; t < block; t++) {
            Fiber &f = fibers[t];
            getcontext(&f.start);
            f.start.uc_stack.ss_sp = stacks + kStack * t;
            f.start.uc_stack.ss_size = kStack;
            f.start.uc_link = nullptr;
            makecontext(&f.start, entry, 0);
            f.started = false;
            f.state = kRuns;
        }
        for (;;) {
            bool moved = false, left = false;
            for (unsigned t = 0; t < block; t++) {
                if (fibers[t].state != kRuns) continue;
                run(t);
                moved = true;
                if (on_yield) on_yield();
            }
            for (unsigned w = 0; w < block; w += 64) moved |= release(w, std::min(w + 64, block), kAtWave);
            moved |= release(0, block, kAtBlock);
            for (unsigned t = 0; t < block; t++) left |= fibers[t].state != kEnded;
            if (!left) break;
            if (!moved) {
                std::fprintf(stderr, "workgroup %u: threads wait for each other\n", b);
                std::abort();
            }
        }
    }
    if (m) munmap(m, size + 2 * kGuard);
}
}  // namespace cpu
