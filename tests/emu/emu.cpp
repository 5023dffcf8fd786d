// Lanes as fibers, and the log of the runtime's calls.
#include "hip/hip_runtime.h"
#include <string>
#include <vector>

// Saves the callee-saved registers and the stack pointer in *save and goes on at `to` (x86-64).
// swapcontext would do, but its system call per switch is most of a run's time.
extern "C" __attribute__((naked, noinline)) void emu_switch(void **save, void *to)
{
    asm("push %rbx; push %rbp; push %r12; push %r13; push %r14; push %r15;"
        "mov %rsp, (%rdi); mov %rsi, %rsp;"
        "pop %r15; pop %r14; pop %r13; pop %r12; pop %rbp; pop %rbx; ret");
}

namespace emu {
dim3 tIdx, bIdx, bDim, gDim;
unsigned char *dyn_lds;
namespace {
struct Fiber {
    void *sp;
    bool done;
    char *stack;
    long turn[64];          // exchanges done per distance
    uint64_t sent[64][2];
};
constexpr size_t kStack = 1 << 20;
std::vector<Fiber *> fibers;
void *scheduler;
int cur, n_lanes;
const std::function<void()> *body_fn;
long wave_gen[16], wave_cnt[16], block_gen, block_cnt;
uint64_t slot[1024];
bool vote[1024];

void body()
{
    (*body_fn)();
    fibers[cur]->done = true;
    emu_switch(&fibers[cur]->sp, scheduler);
}
void yield()
{
    const int me = cur;
    emu_switch(&fibers[me]->sp, scheduler);
}
int alive(int a, int b)
{
    int k = 0;
    for (int i = a; i < b; ++i) k += !fibers[i]->done;
    return k;
}
struct Entry {
    std::string name;
    long long v[6];  // stream, object (launches: threads), grid x, grid y, block, LDS bytes
};
std::vector<Entry> log;
std::string fail_name;
int fail_after = -1, n_objects = 1;
bool execute = true;
hipError_t last = hipSuccess;
}  // namespace

int lane() { return cur & 63; }

void wave_barrier()
{
    const int w = cur / 64;
    const long g = wave_gen[w];
    ++wave_cnt[w];
    while (wave_gen[w] == g) {
        if (wave_cnt[w] >= alive(w * 64, std::min(n_lanes, w * 64 + 64))) {
            wave_cnt[w] = 0;
            ++wave_gen[w];
            return;
        }
        yield();
    }
}

void block_barrier()
{
    const long g = block_gen;
    ++block_cnt;
    while (block_gen == g) {
        if (block_cnt >= alive(0, n_lanes)) {
            block_cnt = 0;
            ++block_gen;
            return;
        }
        yield();
    }
}

// with the lane at distance off, which may be apart from the rest of its wavefront
uint64_t exchange(uint64_t v, int off)
{
    Fiber *const f = fibers[cur], *const o = fibers[(cur & ~63) + (lane() ^ off)];
    const long k = ++f->turn[off];
    f->sent[off][k & 1] = v;
    while (o->turn[off] < k) yield();
    return o->sent[off][k & 1];
}

uint64_t broadcast(uint64_t v, int src)
{
    slot[cur] = v;
    wave_barrier();
    const uint64_t r = slot[(cur & ~63) + src];
    wave_barrier();
    return r;
}

unsigned long long ballot(bool p)
{
    vote[cur] = p;
    wave_barrier();
    unsigned long long m = 0;
    for (int i = 0; i < 64 && (cur & ~63) + i < n_lanes; ++i)
        if (vote[(cur & ~63) + i]) m |= 1ull << i;
    wave_barrier();
    return m;
}

hipError_t call(const char *name, int stream, int object)
{
    log.push_back(Entry{name, {stream, object, 0, 0, 0, 0}});
    if (fail_after >= 0 && fail_name == name && fail_after-- == 0)
        return last = fail_name == "hipMalloc" ? hipErrorOutOfMemory : hipErrorUnknown;
    return hipSuccess;
}

void launch(const char *name, dim3 g, dim3 b, size_t lds, hipStream_t s, const std::function<void()> &fn)
{
    const long long threads = (long long)g.x * b.x;
    log.push_back(Entry{name, {stream_id(s), threads, (long long)g.x, (long long)g.y, (long long)b.x, (long long)lds}});
    if (fail_after >= 0 && fail_name == "launch" && fail_after-- == 0) {
        last = hipErrorUnknown;
        return;
    }
    if (!execute) return;
    n_lanes = b.x;
    bDim = b;
    gDim = g;
    body_fn = &fn;
    while ((int)fibers.size() < n_lanes) {
        auto *f = new Fiber();
        f->stack = (char *)malloc(kStack);
        fibers.push_back(f);
    }
    for (unsigned by = 0; by < g.y; ++by)
        for (unsigned bx = 0; bx < g.x; ++bx) {
            dyn_lds = lds ? (unsigned char *)malloc(lds) : nullptr;
            if (lds) memset(dyn_lds, 0x7f, lds);
            for (int i = 0; i < n_lanes; ++i) {
                Fiber *f = fibers[i];
                f->done = false;
                memset(f->turn, 0, sizeof f->turn);
                // the switch pops six registers and returns into body(), which never returns
                void **top = reinterpret_cast<void **>(f->stack + kStack) - 1;  // 8 mod 16, as after a call
                top[-1] = reinterpret_cast<void *>(&body);
                f->sp = top - 7;
            }
            memset(wave_cnt, 0, sizeof wave_cnt);
            block_cnt = 0;
            for (int left = n_lanes; left;) {
                left = 0;
                for (int i = 0; i < n_lanes; ++i) {
                    if (fibers[i]->done) continue;
                    cur = i;
                    tIdx = dim3(i, 0, 0);
                    bIdx = dim3(bx, by, 0);
                    emu_switch(&scheduler, fibers[i]->sp);
                    left += !fibers[i]->done;
                }
            }
            free(dyn_lds);
        }
}
}  // namespace emu

hipError_t hipGetLastError()
{
    const hipError_t e = emu::last;
    emu::last = hipSuccess;
    return e;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = nullptr;
    if (hipError_t r = emu::call("hipEventCreate")) return r;
    *e = new EmuEvent{emu::n_objects++};
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = nullptr;
    if (hipError_t r = emu::call("hipStreamCreate")) return r;
    *s = new EmuStream{emu::n_objects++, 0};
    return hipSuccess;
}

// ---- for the tests
extern "C" {
void emu_execute(int on) { emu::execute = on; }
// the (n + 1)-th call of that name from now on fails once ("launch": the launch; n < 0: none)
void emu_fail(const char *name, int n)
{
    emu::fail_name = name;
    emu::fail_after = n;
}
void emu_clear() { emu::log.clear(); }
void emu_clear_error() { emu::last = hipSuccess; }
int emu_size() { return (int)emu::log.size(); }
const char *emu_entry(int i, long long *v)
{
    memcpy(v, emu::log[i].v, sizeof emu::log[i].v);
    return emu::log[i].name.c_str();
}
void *emu_stream()
{
    hipStream_t s;
    return hipStreamCreateWithFlags(&s, 0) ? nullptr : s;
}
}
