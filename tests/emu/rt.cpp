// Lanes of a wave as coroutines, and a check of what they exchange through LDS.
//
// The lanes of a wave run one after the other, in an order that changes at every
// operation across lanes, each up to its next such operation.  Every access to
// LDS is reported here by the compiler's instrumentation of loads and stores
// (the callbacks below stand in for its runtime).  On the GPU a store of one lane
// and a load of another are in program order only where the compiler keeps them
// so, and it does only across a fence: a word that two lanes touch between two
// fences, one of them storing another value, is reported as unordered.
#include "rt.hpp"

#include <setjmp.h>
#include <stdio.h>
#include <stdlib.h>
#include <ucontext.h>

#include <algorithm>
#include <map>
#include <random>
#include <string>
#include <vector>

namespace emu {

int lane = 0;

namespace {
constexpr int kMax = 64;
constexpr size_t kStackBytes = 512 << 10;
int n_lanes = 0;
bool done[kMax];
ucontext_t ctx[kMax], home;
jmp_buf jb[kMax], jb_home;
bool started[kMax];
char *stacks[kMax];
void (*body)(void *);
void *body_arg;

uint32_t slots[2][kMax];
int parity = 0;
int op_of[kMax], arg_of[kMax];
long meets = 0, meet_limit = 0;
std::mt19937 rng;

// LDS and what the lanes did there since the last fence
char *lds_lo = nullptr, *lds_hi = nullptr;
char *own_lo = nullptr, *own_hi = nullptr;
struct Word {
    uint32_t epoch = 0;
    uint64_t readers = 0, writers = 0;
    bool atomic = false;
};
std::vector<Word> words;
uint32_t epoch = 1;
const char *atomic_lo = nullptr, *atomic_hi = nullptr;
bool quiet = true;
std::map<std::string, long> unordered;
struct Later {
    uint32_t *p;
    uint32_t before;
    const char *what;
};
std::vector<Later> later;

[[noreturn]] void stop(const char *msg) {
    fprintf(stderr, "emulator: %s (lane %d)\n", msg, lane);
    exit(3);
}

// hazards whose store has been carried out since: of no effect if it left the word as it was
void settle() {
    for (const Later &l : later)
        if (*l.p != l.before) {
            char b[96];
            snprintf(b, sizeof b, "%s of LDS byte %ld", l.what, (long)((char *)l.p - lds_lo) & ~3l);
            unordered[b]++;
        }
    later.clear();
}

void access(void *addr, int bytes, bool write) {
    if (quiet) return;
    char *a = (char *)addr;
    if (a < lds_lo || a >= lds_hi) return;
    if (!later.empty()) settle();
    if (a + bytes > lds_hi) stop("access past the end of LDS");
    if (a >= own_lo && a < own_hi) return;
    const bool atomic = (const char *)a >= atomic_lo && (const char *)a < atomic_hi;
    for (char *p = (char *)((uintptr_t)a & ~(uintptr_t)3); p < a + bytes; p += 4) {
        Word &w = words[(p - lds_lo) / 4];
        if (w.epoch != epoch) w = Word{epoch, 0ull, 0ull, false};
        const uint64_t me = 1ull << lane;
        if (write) {
            if ((w.writers & ~me) != 0ull && !(atomic && w.atomic))
                later.push_back({(uint32_t *)p, *(uint32_t *)p, "two stores"});
            else if (!atomic && (w.readers & ~me) != 0ull)
                later.push_back({(uint32_t *)p, *(uint32_t *)p, "load, then store by another lane,"});
            else if (atomic && (w.readers & ~me) != 0ull && !w.atomic)
                later.push_back({(uint32_t *)p, *(uint32_t *)p, "load, then atomic by another lane,"});
            w.writers |= me;
            w.atomic = atomic;
        } else {
            if (!atomic && (w.writers & ~me) != 0ull) {
                char b[96];
                snprintf(b, sizeof b, "store, then load by another lane, of LDS byte %ld", (long)(p - lds_lo));
                unordered[b]++;
            }
            if (!atomic) w.readers |= me;
        }
    }
    if (atomic && write) atomic_lo = atomic_hi = nullptr;  // (its load came before)
}

void to_home() {
    const int me = lane;
    if (_setjmp(jb[me]) == 0) _longjmp(jb_home, 1);
}
void entry() {
    body(body_arg);
    done[lane] = true;
    _longjmp(jb_home, 1);
}
void resume(int l) {
    lane = l;
    if (_setjmp(jb_home) == 0) {
        if (started[l]) _longjmp(jb[l], 1);
        started[l] = true;
        setcontext(&ctx[l]);
    }
}
}  // namespace

int lanes() { return n_lanes; }

const uint32_t *meet(Op op, int arg, uint32_t x) {
    const int me = lane;
    slots[parity][me] = x;
    op_of[me] = op;
    arg_of[me] = arg;
    const int at = parity;
    to_home();
    return slots[at];
}

uint64_t ballot(bool p) {
    const uint32_t *s = meet(kBallot, 0, p ? 1u : 0u);
    uint64_t m = 0;
    for (int l = 0; l < n_lanes; ++l) m |= (uint64_t)s[l] << l;
    return m;
}

uint32_t dpp(uint32_t x, int ctrl) {
    const uint32_t *s = meet(kDpp, ctrl, x);
    const int row = lane & ~15, l = lane & 15;
    if (ctrl < 0x100) return s[(lane & ~3) + ((ctrl >> (2 * (lane & 3))) & 3)];  // quad_perm
    if (ctrl >= 0x111 && ctrl <= 0x11F) return l >= (ctrl & 15) ? s[row + l - (ctrl & 15)] : 0u;  // row_shr
    if (ctrl >= 0x121 && ctrl <= 0x12F) return s[row + ((l - (ctrl & 15)) & 15)];  // row_ror
    if (ctrl == 0x140) return s[row + 15 - l];
    if (ctrl == 0x141) return s[row + (l ^ 7)];
    if (ctrl >= 0x150 && ctrl <= 0x15F) return s[row + (ctrl & 15)];  // row_newbcast
    stop("unknown DPP control");
}

void fence() { meet(kFence, 0, 0u); }

void atomic_at(const void *p, int bytes) {
    if (!later.empty()) settle();
    atomic_lo = (const char *)p;
    atomic_hi = atomic_lo + bytes;
}

void watch(void *lds, size_t bytes) {
    lds_lo = (char *)lds;
    lds_hi = lds_lo + bytes;
    words.assign(bytes / 4 + 1, Word{});
}
void leave_out(void *p, size_t bytes) {
    own_lo = (char *)p;
    own_hi = own_lo + bytes;
}

void run(int n, unsigned seed, long limit, void (*f)(void *), void *arg) {
    n_lanes = n;
    body = f;
    body_arg = arg;
    meets = 0;
    meet_limit = limit;
    rng.seed(seed);
    ++epoch;
    int order[kMax];
    for (int l = 0; l < n; ++l) {
        done[l] = started[l] = false;
        order[l] = l;
        if (!stacks[l]) stacks[l] = (char *)malloc(kStackBytes);
        getcontext(&ctx[l]);
        ctx[l].uc_stack.ss_sp = stacks[l];
        ctx[l].uc_stack.ss_size = kStackBytes;
        ctx[l].uc_link = &home;
        makecontext(&ctx[l], entry, 0);
    }
    quiet = false;
    while (true) {
        std::shuffle(order, order + n, rng);
        for (int t = 0; t < n; ++t) {
            resume(order[t]);
            if (!later.empty()) settle();
            atomic_lo = atomic_hi = nullptr;
        }
        int ended = 0;
        for (int l = 0; l < n; ++l) ended += done[l];
        if (ended == n) break;
        if (ended) stop("some lanes ended while others wait for them");
        for (int l = 1; l < n; ++l)
            if (op_of[l] != op_of[0] || arg_of[l] != arg_of[0]) {
                fprintf(stderr, "lane 0 at operation %d (%d), lane %d at %d (%d)\n", op_of[0], arg_of[0], l, op_of[l], arg_of[l]);
                stop("lanes wait at different operations");
            }
        if (op_of[0] == kFence) ++epoch;
        parity ^= 1;
        if (++meets > meet_limit) stop("no end in sight: more operations across lanes than allowed");
    }
    quiet = true;
}

int report(FILE *f) {
    for (const auto &u : unordered) fprintf(f, "unordered: %s (%ld times)\n", u.first.c_str(), u.second);
    return (int)unordered.size();
}

}  // namespace emu

extern "C" {
void __tsan_init() {}
void __tsan_func_entry(void *) {}
void __tsan_func_exit() {}
#define HOOKS(n)                                                                      \
    void __tsan_read##n(void *p) { emu::access(p, n, false); }                    \
    void __tsan_write##n(void *p) { emu::access(p, n, true); }                    \
    void __tsan_unaligned_read##n(void *p) { emu::access(p, n, false); }          \
    void __tsan_unaligned_write##n(void *p) { emu::access(p, n, true); }          \
    void __tsan_volatile_read##n(void *p) { emu::access(p, n, false); }           \
    void __tsan_volatile_write##n(void *p) { emu::access(p, n, true); }
HOOKS(1)
HOOKS(2)
HOOKS(4)
HOOKS(8)
HOOKS(16)
void __tsan_read_range(void *p, size_t n) { emu::access(p, (int)n, false); }
void __tsan_write_range(void *p, size_t n) { emu::access(p, (int)n, true); }
void __tsan_vptr_update(void **, void *) {}
void __tsan_vptr_read(void **) {}
}
