// Runs a kernel compiled for the CPU (hip/hip_runtime.h beside this file) over a grid.  The fibers of a
// block run one after another up to their next barrier; a block whose threads do not all meet every
// barrier ends the program.  The LDS array is poisoned past the size of the launch.
#pragma once
#include <sanitizer/asan_interface.h>
#include <sanitizer/common_interface_defs.h>
#include <ucontext.h>

#include <cstdio>
#include <cstdlib>
#include <functional>
#include <vector>

#include "hip/hip_runtime.h"

dim3 threadIdx, blockIdx, blockDim, gridDim;

namespace emulate {

constexpr size_t kStack = 64 * 1024;
struct fiber {
    ucontext_t ctx;
    std::vector<char> stack;
    bool done;
    void *fake;
};
std::vector<fiber> fibers;
ucontext_t main_ctx;
void *main_fake;
const void *main_bottom;
size_t main_size;
int current;
const std::function<void()> *body;

void to_main(bool ending) {
    fiber &f = fibers[current];
    __sanitizer_start_switch_fiber(ending ? nullptr : &f.fake, main_bottom, main_size);
    swapcontext(&f.ctx, &main_ctx);
    __sanitizer_finish_switch_fiber(f.fake, nullptr, nullptr);
}
void entry() {
    __sanitizer_finish_switch_fiber(nullptr, &main_bottom, &main_size);
    (*body)();
    fibers[current].done = true;
    to_main(true);
}

// One thread at a time up to its next barrier, until all have ended.
inline void run_block(int threads, const std::function<void()> &fn) {
    body = &fn;
    if ((int)fibers.size() < threads) fibers.resize(threads);
    for (int t = 0; t < threads; t++) {
        fiber &f = fibers[t];
        if (f.stack.empty()) f.stack.resize(kStack);
        f.done = false;
        f.fake = nullptr;
        getcontext(&f.ctx);
        f.ctx.uc_stack.ss_sp = f.stack.data();
        f.ctx.uc_stack.ss_size = kStack;
        f.ctx.uc_link = nullptr;
        makecontext(&f.ctx, entry, 0);
    }
    for (int left = threads; left > 0;) {
        int ended = 0;
        for (int t = 0; t < threads; t++) {
            current = t;
            threadIdx = dim3(t);
            __sanitizer_start_switch_fiber(&main_fake, fibers[t].stack.data(), kStack);
            swapcontext(&main_ctx, &fibers[t].ctx);
            __sanitizer_finish_switch_fiber(main_fake, nullptr, nullptr);
            ended += fibers[t].done ? 1 : 0;
        }
        if (ended && ended != threads) {
            std::printf("threads of one block ended at different barriers\n");
            std::exit(2);
        }
        left -= ended;
    }
}

// kernel() for every block and thread; lds: the dynamic LDS array, lds_bytes of it usable.
inline void run_blocks(long long nblocks, int threads, unsigned char *lds, size_t lds_size, size_t lds_bytes,
                       const std::function<void()> &fn) {
    const size_t used = (lds_bytes + 7) / 8 * 8;
    if (used < lds_size) ASAN_POISON_MEMORY_REGION(lds + used, lds_size - used);
    blockDim = dim3(threads);
    gridDim = dim3((unsigned)nblocks);
    for (long long b = 0; b < nblocks; b++) {
        blockIdx = dim3((unsigned)b);
        run_block(threads, fn);
    }
    ASAN_UNPOISON_MEMORY_REGION(lds, lds_size);
}

}  // namespace emulate

void emulate_yield() { emulate::to_main(false); }
