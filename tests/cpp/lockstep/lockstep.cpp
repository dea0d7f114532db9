// The scheduler of the CPU stand-in (hip/hip_runtime.h): fibers, wave-wide operations, barriers, and the
// device memory, as host memory.
#include <hip/hip_runtime.h>

#include <stdio.h>
#include <stdlib.h>
#include <sys/mman.h>

#include <string>
#include <vector>

namespace ahead_dev {
thread_local char s_op[160 * 1024] __attribute__((aligned(16)));  // dynamic LDS of k_stream
}

namespace lockstep {
namespace {

constexpr size_t kStack = 256 * 1024;
constexpr uint32_t kMost = 1024;

struct Lane {
    ucontext_t ctx;
    Op op;
    int line;
    uint64_t v;
    bool done;
};
struct Wave {
    uint64_t out[64], on;
};

Lane lanes[kMost];
Wave waves[kMost / 64];
ucontext_t sched;
char *stacks;
const std::function<void()> *body;
uint32_t cur, bid, bdim, gdim;
bool bar_any, bar_out;
uint64_t swaps;  // compare-and-swaps of the launch
uint64_t steps;  // wave-wide operations and barriers, summed over the waves, of the launch
int descending, dry, device;
int cus[2] = {256, 4};  // device 0 is a large card, device 1 a small one
std::string log_;
std::vector<std::string> attrs;

[[noreturn]] void bad(const char *what) {
    fprintf(stderr, "lockstep: %s (workgroup %u)\n", what, bid);
    fflush(stderr);
    abort();
}

void entry() {
    (*body)();
    lanes[cur].done = true;
    lanes[cur].op = kNone;
    swapcontext(&lanes[cur].ctx, &sched);
}

void yield() { swapcontext(&lanes[cur].ctx, &sched); }

// Runs a wave until its lanes wait at a barrier or are done; false: done.
bool run_wave(uint32_t w) {
    const uint32_t b = w * 64, e = b + 64 < bdim ? b + 64 : bdim;
    for (;;) {
        for (uint32_t i = b; i < e; ++i) {
            if (lanes[i].done) continue;
            cur = i;
            swapcontext(&sched, &lanes[i].ctx);
        }
        Op op = kNone;
        uint64_t on = 0;
        ++steps;
        for (uint32_t i = b; i < e; ++i) {
            if (lanes[i].done) continue;
            if (op == kNone) op = lanes[i].op;
            if (lanes[i].op != op) bad("the lanes of a wave stand at different operations");
            on |= 1ull << (i - b);
        }
        if (op == kNone) return false;
        if (op == kBarrier) return true;
        for (uint32_t i = b; i < e; ++i) waves[w].out[i - b] = lanes[i].v;
        waves[w].on = on;
    }
}

void run_block() {
    for (uint32_t i = 0; i < bdim; ++i) {
        lanes[i].done = false;
        getcontext(&lanes[i].ctx);
        lanes[i].ctx.uc_stack.ss_sp = stacks + i * kStack;
        lanes[i].ctx.uc_stack.ss_size = kStack;
        lanes[i].ctx.uc_link = nullptr;
        makecontext(&lanes[i].ctx, entry, 0);
    }
    const uint32_t nw = (bdim + 63) / 64;
    std::vector<bool> live(nw, true);
    for (;;) {
        bool any = false;
        bar_any = false;
        for (uint32_t k = 0; k < nw; ++k) {
            const uint32_t w = descending ? nw - 1 - k : k;
            if (live[w]) live[w] = run_wave(w);
            any = any || live[w];
        }
        if (!any) return;
        int line = 0;
        for (uint32_t i = 0; i < bdim; ++i) {
            if (lanes[i].done) continue;
            if (line == 0) line = lanes[i].line;
            if (lanes[i].line != line) bad("the waves of a workgroup stand at different barriers");
        }
        bar_out = bar_any;
    }
}

}  // namespace

uint32_t thread_id() { return cur; }
void count_cas() { ++swaps; }
uint32_t block_id() { return bid; }
uint32_t block_size() { return bdim; }
uint32_t grid_size() { return gdim; }

bool barrier(int line, bool any) {
    lanes[cur].op = kBarrier;
    lanes[cur].line = line;
    bar_any = bar_any || any;
    yield();
    return bar_out;
}

const uint64_t *wave_op(Op op, uint64_t v, uint64_t *on) {
    lanes[cur].op = op;
    lanes[cur].v = v;
    yield();
    *on = waves[cur / 64].on;
    return waves[cur / 64].out;
}

void launch(const char *name, dim3 grid, dim3 block, const std::function<void()> &kernel) {
    struct Log {
        std::string head;
        ~Log() { log_ += head + std::to_string(steps) + " " + std::to_string(swaps) + "\n"; }
    } log{std::string(name) + " " + std::to_string(grid.x) + " " + std::to_string(block.x) + " "};
    steps = swaps = 0;
    if (dry) return;
    if (block.x > kMost) bad("workgroup too large");
    if (stacks == nullptr) {
        stacks = static_cast<char *>(mmap(nullptr, kMost * kStack, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
        if (stacks == MAP_FAILED) bad("no memory for the stacks");
    }
    body = &kernel;
    bdim = block.x;
    gdim = grid.x;
    for (bid = 0; bid < gdim; ++bid) run_block();
}

}  // namespace lockstep

hipError_t hipMalloc(void **p, size_t bytes) {
    *p = aligned_alloc(256, (bytes + 255) / 256 * 256);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
    free(p);
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t bytes) {
    memset(p, v, bytes);
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, int, int dev) {
    *v = lockstep::cus[dev];
    return hipSuccess;
}
hipError_t hipGetDevice(int *dev) {
    *dev = lockstep::device;
    return hipSuccess;
}
hipError_t hipSetDevice(int dev) {
    lockstep::device = dev;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, int, int) {
    lockstep::log_ += "attribute " + std::to_string(lockstep::device) + "\n";
    return hipSuccess;
}

extern "C" {
// Waves in descending order; kernels recorded but not run; the current device.
void lockstep_set(int descending, int dry, int device) {
    lockstep::descending = descending;
    lockstep::dry = dry;
    lockstep::device = device;
}
// The launches since the last call, one line each: kernel, workgroups, threads, steps run,
// compare-and-swaps.
const char *lockstep_launches(void) {
    static std::string out;
    out.swap(lockstep::log_);
    lockstep::log_.clear();
    return out.c_str();
}
}
