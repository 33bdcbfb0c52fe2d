// The scheduler of simt.hpp's fibres.
#include "simt.hpp"

#include <sys/mman.h>
#include <vector>

#if defined(__SANITIZE_ADDRESS__)
#define SIMT_ASAN 1
#elif defined(__has_feature)
#if __has_feature(address_sanitizer)
#define SIMT_ASAN 1
#endif
#endif
#ifdef SIMT_ASAN
extern "C" {
void __sanitizer_start_switch_fiber(void **save, const void *bottom, size_t size);
void __sanitizer_finish_switch_fiber(void *save, const void **bottom, size_t *size);
}
#endif
#undef asm

extern "C" {
extern char __start_simt_lds[] __attribute__((weak));
extern char __stop_simt_lds[] __attribute__((weak));
// Saves the callee-saved registers on the stack, its top in *from, and goes on at `to`.
void simt_switch(void **from, void *to);
void simt_entry();
}
__asm__(
    ".text\n.globl simt_switch\nsimt_switch:\n"
    "pushq %rbp\npushq %rbx\npushq %r12\npushq %r13\npushq %r14\npushq %r15\n"
    "movq %rsp, (%rdi)\nmovq %rsi, %rsp\n"
    "popq %r15\npopq %r14\npopq %r13\npopq %r12\npopq %rbx\npopq %rbp\nret\n"
    ".globl simt_entry\nsimt_entry:\ncall simt_main\n");

namespace simt {

enum State { kReady, kMeet, kBarrier, kDone };
constexpr size_t kStack = 256 << 10;
struct Thread : Fibre {
    State state = kDone;
    void *sp = nullptr, *fake = nullptr;
    char *stack = nullptr;
    const char *file = nullptr;
    int line = 0;
};
struct Wave {
    uint64_t words[2][64];
    int turn = 0;  // the words of the last meeting stay valid during the next
    uint64_t live = 0;
};

Fibre *cur = nullptr;
static std::vector<Thread> threads;
static std::vector<Wave> waves;
static void *main_sp = nullptr, *main_fake = nullptr;
static const void *main_bottom = nullptr;
static size_t main_size = 0;
static const std::function<void()> *body = nullptr;

static void to_main(bool last) {
    Thread *t = static_cast<Thread *>(cur);
#ifdef SIMT_ASAN
    __sanitizer_start_switch_fiber(last ? nullptr : &t->fake, main_bottom, main_size);
#endif
    simt_switch(&t->sp, main_sp);
#ifdef SIMT_ASAN
    __sanitizer_finish_switch_fiber(t->fake, nullptr, nullptr);
#endif
    (void)last;
}

extern "C" void simt_main() {
#ifdef SIMT_ASAN
    __sanitizer_finish_switch_fiber(nullptr, &main_bottom, &main_size);
#endif
    (*body)();
    static_cast<Thread *>(cur)->state = kDone;
    to_main(true);
    std::abort();
}

static void resume(Thread &t) {
    cur = &t;
#ifdef SIMT_ASAN
    __sanitizer_start_switch_fiber(&main_fake, t.stack, kStack);
#endif
    simt_switch(&main_sp, t.sp);
#ifdef SIMT_ASAN
    __sanitizer_finish_switch_fiber(main_fake, nullptr, nullptr);
#endif
}

const uint64_t *meet(uint64_t word, uint64_t *live, const char *file, int line) {
    Thread *t = static_cast<Thread *>(cur);
    Wave &w = waves[t->wave];
    const int turn = w.turn;
    w.words[turn][t->lane] = word;
    t->file = file;
    t->line = line;
    t->state = kMeet;
    to_main(false);
    *live = w.live;
    return w.words[turn];
}

void barrier() {
    static_cast<Thread *>(cur)->state = kBarrier;
    to_main(false);
}

// Runs wave w as far as a barrier lets it.
static void run_wave(int w, int n) {
    const int lo = 64 * w, hi = lo + 64 < n ? lo + 64 : n;
    for (;;) {
        for (int i = lo; i < hi; ++i)
            if (threads[i].state == kReady) resume(threads[i]);
        // lanes at one meeting go on together; where a branch has some of
        // them elsewhere, those in the innermost file and line first
        const Thread *at = nullptr;
        for (int i = lo; i < hi; ++i) {
            const Thread &t = threads[i];
            if (t.state == kMeet && (!at || std::strcmp(t.file, at->file) < 0 ||
                                     (!std::strcmp(t.file, at->file) && t.line < at->line)))
                at = &t;
        }
        if (!at) return;
        uint64_t live = 0;
        const char *file = at->file;
        const int line = at->line;
        for (int i = lo; i < hi; ++i) {
            Thread &t = threads[i];
            if (t.state == kDone) continue;
            const bool same = t.state == kMeet && t.line == line && !std::strcmp(t.file, file);
            if (same) live |= 1ull << (i - lo);
            // only the branch for odd denominators (device.hpp), whose ballot
            // chooses between equal results, is met by a part of the wave
            else if (!std::strstr(file, "device.hpp")) {
                std::fprintf(stderr, "simt: lanes of a wave at %s:%d and %s:%d\n", file, line,
                             t.state == kBarrier ? "a barrier" : t.file, t.line);
                std::exit(70);
            }
        }
        Wave &W = waves[w];
        W.live = live;
        W.turn ^= 1;
        std::memcpy(W.words[W.turn], W.words[W.turn ^ 1], sizeof W.words[0]);
        for (int i = lo; i < hi; ++i)
            if (live >> (i - lo) & 1) threads[i].state = kReady;
    }
}

void launch(dim3 grid, dim3 block, const std::function<void()> &fn) {
    const int n = (int)block.x, nw = (n + 63) / 64;
    static uint64_t rng = 0;
    static int order = -1;
    if (order < 0) {
        const char *e = std::getenv("NBG_SIMT_ORDER");
        order = e ? std::atoi(e) : 0;
        rng = (uint64_t)order * 0x9E3779B97F4A7C15ull + 1;
    }
    if (threads.empty()) {
        threads.resize(1024);
        for (auto &t : threads)
            t.stack = (char *)mmap(nullptr, kStack, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
        waves.resize(16);
    }
    body = &fn;
    std::vector<int> seq(nw);
    for (unsigned b = 0; b < grid.x; ++b) {
        if (__start_simt_lds) std::memset(__start_simt_lds, 0xA5, __stop_simt_lds - __start_simt_lds);
        for (int i = 0; i < n; ++i) {
            Thread &t = threads[i];
            t.tid = dim3(i, 0, 0);
            t.bid = dim3(b, 0, 0);
            t.bdim = block;
            t.gdim = grid;
            t.lane = i % 64;
            t.wave = i / 64;
            t.state = kReady;
            void **p = reinterpret_cast<void **>(t.stack + kStack - 16);
            *--p = reinterpret_cast<void *>(&simt_entry);
            for (int r = 0; r < 6; ++r) *--p = nullptr;
            t.sp = p;
        }
        for (;;) {
            for (int w = 0; w < nw; ++w) seq[w] = order == 1 ? nw - 1 - w : w;
            if (order >= 2)
                for (int w = nw - 1; w > 0; --w) {
                    rng = rng * 6364136223846793005ull + 1442695040888963407ull;
                    std::swap(seq[w], seq[(rng >> 33) % (w + 1)]);
                }
            for (int w : seq) run_wave(w, n);
            bool waiting = false;
            for (int i = 0; i < n; ++i)
                if (threads[i].state == kBarrier) {
                    threads[i].state = kReady;
                    waiting = true;
                }
            if (!waiting) break;
        }
    }
    cur = nullptr;
}

}  // namespace simt
