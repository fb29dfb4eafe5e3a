// Lanes as fibers, and memory behind guard pages (see hip/hip_runtime.h).
#include <dlfcn.h>
#include <hip/hip_runtime.h>
#include <signal.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <map>
#include <string>

dim3 blockIdx, blockDim, gridDim;

// Saves the callee-saved registers and the stack pointer in *save, and goes on
// where `to` was saved.
extern "C" void emulation_switch(void **save, void *to);
asm(R"(
.text
.globl emulation_switch
emulation_switch:
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

namespace emulation {

std::recursive_mutex mu;
Lane *cur = nullptr;

namespace {

enum State { kRun, kDone, kAtWave, kAtBlock };
struct Fiber : Lane {
    void *sp;
    char *stack;
    State state;
    int line;
    uint64_t word;
};
constexpr int kFibers = 1024, kPage = 4096;
constexpr size_t kStack = 256 << 10;

Fiber fibers[kFibers];
uint64_t wave_words[kFibers / 64][64], wave_live[kFibers / 64];
void *scheduler;  // its stack while a fiber runs
const void *kernel_fn;
void (*lane_fn)(void *);
void *lane_arg;
int error = hipSuccess;
std::string fail_kernel;  // emulation_fail_launch
int fail_after = -1;
bool backwards = false;  // emulation_backwards
struct Range {
    char *map, *user;
    size_t mapped, bytes;
};
std::map<void *, Range> ranges;

void to_scheduler() {
    Fiber *const f = static_cast<Fiber *>(cur);
    emulation_switch(&f->sp, scheduler);
}
void fiber_main() {
    for (;;) {
        lane_fn(lane_arg);
        static_cast<Fiber *>(cur)->state = kDone;
        to_scheduler();
    }
}
void new_stacks() {
    for (int i = 0; i < kFibers; ++i) {
        Fiber &f = fibers[i];
        if (!f.stack) {
            f.stack = (char *)mmap(nullptr, kStack, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
            mprotect(f.stack, kPage, PROT_NONE);
        }
        f.tid = (uint32_t)i;
        uint64_t *sp = (uint64_t *)(f.stack + kStack - 64);
        *--sp = 0;  // the stack is at 8 mod 16 in fiber_main, as after a call
        *--sp = (uint64_t)fiber_main;
        for (int k = 0; k < 6; ++k) *--sp = 0;
        f.sp = sp;
    }
}
const char *kernel_name() {
    Dl_info i{};
    return dladdr(kernel_fn, &i) && i.dli_sname ? i.dli_sname : "?";
}
void report(const char *what, int line) {
    fprintf(stderr, "emulation: %s: kernel %s, block %u of %u, thread %d, line %d\n", what, kernel_name(), blockIdx.x, gridDim.x,
            cur ? (int)cur->tid : -1, line);
    error = hipErrorIllegalAddress;
}
// An access that the device would not survive: the launch ends here.
void on_fault(int sig, siginfo_t *, void *) {
    if (!cur) {  // not in a kernel
        signal(sig, SIG_DFL);
        return;
    }
    report("access out of bounds", -1);
    void *gone;
    emulation_switch(&gone, scheduler);
}
void setup() {
    static bool done = false;
    if (done) return;
    done = true;
    new_stacks();
    stack_t alt{};
    alt.ss_size = 1 << 16;
    alt.ss_sp = malloc(alt.ss_size);
    sigaltstack(&alt, nullptr);
    struct sigaction sa {};
    sa.sa_sigaction = on_fault;
    sa.sa_flags = SA_SIGINFO | SA_ONSTACK | SA_NODEFER;
    sigaction(SIGSEGV, &sa, nullptr);
    sigaction(SIGBUS, &sa, nullptr);
}

// Lanes [lo, hi) up to their end or the block's next barrier.
void run_wave(int lo, int hi) {
    for (;;) {
        for (int i = lo; i < hi; ++i) {
            if (fibers[i].state != kRun) continue;
            cur = &fibers[i];
            emulation_switch(&scheduler, fibers[i].sp);
            if (error) return;
        }
        uint64_t live = 0, at = 0;
        int line = -1;
        for (int i = lo; i < hi; ++i) {
            if (fibers[i].state == kDone) continue;
            live |= 1ull << (i - lo);
            if (fibers[i].state != kAtWave) continue;
            at |= 1ull << (i - lo);
            if (line >= 0 && line != fibers[i].line) return report("lanes at different wave operations", fibers[i].line);
            line = fibers[i].line;
        }
        if (!at) return;
        if (at != live) return report("a wave operation that not all lanes come to", line);
        for (int i = lo; i < hi; ++i) {
            wave_words[lo / 64][i - lo] = fibers[i].state == kAtWave ? fibers[i].word : 0;
            if (fibers[i].state == kAtWave) fibers[i].state = kRun;
        }
        wave_live[lo / 64] = live;
    }
}
void run_block(int threads) {
    for (int i = 0; i < threads; ++i) fibers[i].state = kRun;
    for (;;) {
        for (int lo = 0; lo < threads; lo += 64) {
            run_wave(lo, std::min(threads, lo + 64));
            if (error) return;
        }
        int line = -1;
        for (int i = 0; i < threads; ++i) {
            if (fibers[i].state == kDone) continue;
            if (line >= 0 && line != fibers[i].line) return report("threads at different barriers", line);
            line = fibers[i].line;
            fibers[i].state = kRun;
        }
        if (line < 0) return;
    }
}

}  // namespace

uint64_t wave_sync(uint64_t word, int line) {
    Fiber *const f = static_cast<Fiber *>(cur);
    f->word = word;
    f->line = line;
    f->state = kAtWave;
    to_scheduler();
    return wave_live[cur->tid / 64];
}
const uint64_t *snap() { return wave_words[cur->tid / 64]; }
void block_sync(int line) {
    Fiber *const f = static_cast<Fiber *>(cur);
    f->line = line;
    f->state = kAtBlock;
    to_scheduler();
}
void lane_error(const char *what, int line) {
    report(what, line);
    for (;;) to_scheduler();
}
int status() { return error; }

void run(const void *kernel, dim3 grid, dim3 block, void (*fn)(void *), void *arg) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    if (error) return;
    kernel_fn = kernel;
    if (fail_after >= 0 && strstr(kernel_name(), fail_kernel.c_str()) && fail_after-- == 0) {
        error = hipErrorIllegalAddress;
        return;
    }
    setup();
    gridDim = grid;
    blockDim = block;
    lane_fn = fn;
    lane_arg = arg;
    for (uint32_t b = 0; b < grid.x && !error; ++b) {
        blockIdx.x = backwards ? grid.x - 1 - b : b;
        run_block((int)block.x);
    }
    cur = nullptr;
    if (error) new_stacks();
}
// Ends at a page boundary (to 16 bytes), between pages that cannot be touched;
// filled with a pattern no valid id, count or pointer has.
void *alloc(size_t bytes) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    setup();
    const size_t body = (bytes + kPage - 1) / kPage * kPage;
    char *const map = (char *)mmap(nullptr, body + 2 * kPage, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (map == MAP_FAILED) return nullptr;
    mprotect(map + kPage, body, PROT_READ | PROT_WRITE);
    memset(map + kPage, 0xCD, body);
    char *const user = map + kPage + ((body - bytes) & ~(size_t)15);
    ranges[user] = Range{map, user, body + 2 * kPage, bytes};
    return user;
}
void release(void *p) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    const auto it = ranges.find(p);
    if (it == ranges.end()) return;
    madvise(it->second.map, it->second.mapped, MADV_DONTNEED);  // the addresses stay taken: a later access faults
    mprotect(it->second.map, it->second.mapped, PROT_NONE);
    ranges.erase(it);
}

}  // namespace emulation

extern "C" {
// The device works again (0), or fails at the launch after `after` more ones of
// kernels whose name holds `kernel`.
void emulation_reset() {
    emulation::error = hipSuccess;
    emulation::fail_after = -1;
    emulation::backwards = false;
}
// Blocks run from the last to the first.
void emulation_backwards() { emulation::backwards = true; }
void emulation_fail_launch(const char *kernel, int after) {
    emulation::fail_kernel = kernel;
    emulation::fail_after = after;
}
// Every word `from` of the memory in use becomes `to`; how many there were.
uint64_t emulation_replace(uint32_t from, uint32_t to) {
    std::lock_guard<std::recursive_mutex> lock(emulation::mu);
    uint64_t n = 0;
    for (auto &r : emulation::ranges) {
        uint32_t *const w = (uint32_t *)r.second.user;
        for (size_t i = 0; i < r.second.bytes / 4; ++i)
            if (w[i] == from) {
                w[i] = to;
                ++n;
            }
    }
    return n;
}
}
