// The CPU side of include/hip/hip_runtime.h.
//
// * Memory: every hipMalloc lies against an inaccessible page, at its end
//   (default) or, with emu_alloc_low(1), at its start; a kernel's dynamic LDS
//   likewise.  An access out of range stops the process.  New memory is filled
//   with 0xA5.
// * Threads: the lanes of a block are fibers.  A lane that reaches a wavefront
//   operation waits until every lane of its wavefront waits or has ended; the
//   lanes at the operation then exchange their values.  A block barrier waits for
//   the block.
// * Streams: launches run at once; vector clocks keep what each stream is
//   ordered after, so that emu_unjoined() can tell how many streams hold work
//   that the null stream does not wait for.
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <dlfcn.h>
#include <map>
#include <string>
#include <vector>

// ---- memory
namespace {
constexpr size_t kPage = 4096;
bool g_low = false;
struct Block { char* base; size_t len; };
std::map<void*, Block> g_mem;

void* guarded(size_t n, Block* out) {
    const size_t body = (std::max<size_t>(n, 1) + kPage - 1) / kPage * kPage;
    char* b = (char*)mmap(nullptr, body + 2 * kPage, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (b == MAP_FAILED || mprotect(b + kPage, body, PROT_READ | PROT_WRITE)) return nullptr;
    *out = {b, body + 2 * kPage};
    char* p = g_low ? b + kPage : b + kPage + body - n;
    std::memset(p, 0xA5, n);
    return p;
}
}  // namespace
extern "C" void emu_alloc_low(int low) { g_low = low != 0; }
hipError_t hipMalloc(void** p, size_t n) {
    Block b;
    *p = guarded(n, &b);
    if (!*p) return hipErrorOutOfMemory;
    g_mem[*p] = b;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    const auto it = g_mem.find(p);
    if (it == g_mem.end()) return p ? hipErrorInvalidValue : hipSuccess;
    munmap(it->second.base, it->second.len);
    g_mem.erase(it);
    return hipSuccess;
}

// ---- streams and events
struct EmuStream { std::map<EmuStream*, long long> seen; long long work = 0; };
struct EmuEvent { std::map<EmuStream*, long long> seen; };
namespace {
EmuStream g_null;
std::vector<EmuStream*> g_streams;
EmuStream* of(hipStream_t s) { return s ? s : &g_null; }
void merge(std::map<EmuStream*, long long>& a, const std::map<EmuStream*, long long>& b) {
    for (const auto& kv : b) a[kv.first] = std::max(a[kv.first], kv.second);
}
void enqueue(hipStream_t s) { of(s)->seen[of(s)] = ++of(s)->work; }
// the next hipGetLastError answers after `left` good ones (-1: never)
long long g_fail_in = -1;
}  // namespace
extern "C" void emu_fail_in(long long n) { g_fail_in = n; }
extern "C" int emu_unjoined() {
    int n = 0;
    for (EmuStream* s : g_streams) n += g_null.seen[s] < s->work;
    return n;
}
hipError_t hipGetLastError() {
    if (g_fail_in < 0 || g_fail_in-- > 0) return hipSuccess;
    return hipErrorLaunchFailure;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "emulated error"; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
    enqueue(st);
    return hipMemcpy(d, s, n, k);
}
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) { *p = {}; return hipSuccess; }
hipError_t hipDeviceSynchronize() {
    for (EmuStream* s : g_streams) merge(g_null.seen, s->seen);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    g_streams.push_back(*s = new EmuStream);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    g_streams.erase(std::find(g_streams.begin(), g_streams.end(), s));
    return hipSuccess;   // kept: the clocks hold its address
}
hipError_t hipStreamSynchronize(hipStream_t s) { merge(g_null.seen, of(s)->seen); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    merge(of(s)->seen, e->seen);
    if (s) enqueue(s);   // a forked stream is joined whether or not it then works
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { *e = new EmuEvent; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { e->seen = of(s)->seen; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }

// ---- kernels
namespace {
std::map<std::string, long long> g_scratch;   // per lane, by mangled name
std::string g_record;                         // "name grid block lds stream\n" of each launch
const char* kernel_name(const void* f) {
    Dl_info i;
    return dladdr(f, &i) && i.dli_sname ? i.dli_sname : "?";
}
}  // namespace
extern "C" void emu_set_scratch(const char* name, long long bytes) { g_scratch[name] = bytes; }
extern "C" const char* emu_record() { return g_record.c_str(); }
extern "C" void emu_clear_record() { g_record.clear(); }
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void* f) {
    *a = {};
    const auto it = g_scratch.find(kernel_name(f));
    if (it != g_scratch.end()) a->localSizeBytes = it->second;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t lds) {
    *n = lds ? std::max<int>(1, std::min<int>(8, 160 * 1024 / lds)) : 8;
    return hipSuccess;
}

// saves the callee's registers and stack pointer, continues on another stack
extern "C" void emu_switch(void** save, void* next);
__asm__(R"(
.text
.globl emu_switch
emu_switch:
    push %rbp
    push %rbx
    push %r12
    push %r13
    push %r14
    push %r15
    mov %rsp, (%rdi)
    mov %rsi, %rsp
    pop %r15
    pop %r14
    pop %r13
    pop %r12
    pop %rbx
    pop %rbp
    ret
)");

namespace emu {
Idx g_block, g_thread, g_block_dim, g_grid_dim;
namespace {
constexpr size_t kStack = 512 * 1024;
enum State { kReady, kWave, kBlock, kDone };
struct Fiber {
    void* sp = nullptr;
    char* stack = nullptr;
    State st = kDone;
    uint64_t val = 0;
    const char* what = nullptr;
    Idx tid;
};
std::vector<Fiber> g_fib;
std::vector<Wave> g_wave;
void* g_main;
int g_cur = -1;
void* g_lds = nullptr;
const std::function<void()>* g_body;

void entry() {
    (*g_body)();
    g_fib[g_cur].st = kDone;
    emu_switch(&g_fib[g_cur].sp, g_main);
}
void wait(State s) {
    Fiber& f = g_fib[g_cur];
    f.st = s;
    emu_switch(&f.sp, g_main);
}
void run(int k) {
    g_cur = k;
    g_thread = g_fib[k].tid;
    g_fib[k].st = kReady;
    emu_switch(&g_main, g_fib[k].sp);
}
// runs the wavefront's lanes until each has ended or waits for the block
void run_wave(int w, int n) {
    const int l0 = 64 * w, l1 = std::min(n, l0 + 64);
    for (;;) {
        bool any = false;
        for (int k = l0; k < l1; ++k)
            if (g_fib[k].st == kReady) run(k);
        Wave& W = g_wave[w];
        W.active = 0;
        const char* what = nullptr;
        for (int k = l0; k < l1; ++k)
            if (g_fib[k].st == kWave) {
                if (what && std::strcmp(what, g_fib[k].what)) {
                    std::fprintf(stderr, "emulator: lanes of one wavefront wait at %s and %s\n", what, g_fib[k].what);
                    std::abort();
                }
                what = g_fib[k].what;
                W.active |= 1ull << (k - l0);
                W.v[k - l0] = g_fib[k].val;
                any = true;
            }
        if (!any) return;
        for (int k = l0; k < l1; ++k)
            if (g_fib[k].st == kWave) g_fib[k].st = kReady;
    }
}
}  // namespace

void* dynamic_lds() { return g_lds; }
unsigned lane() { return (unsigned)(g_cur & 63); }
const Wave& wave_op(uint64_t mine, const char* what) {
    g_fib[g_cur].val = mine;
    g_fib[g_cur].what = what;
    const int w = g_cur >> 6;
    wait(kWave);
    // the values stay until this lane's next operation: no lane passes one before all have left this one
    return g_wave[w];
}
void block_barrier() { wait(kBlock); }

void launch(const void* kernel, dim3 grid, dim3 block, size_t lds, hipStream_t s, const std::function<void()>& body) {
    char line[512];
    std::snprintf(line, sizeof line, "%s %u %u %zu %d\n", kernel_name(kernel), grid.x * grid.y * grid.z, block.x, lds,
                  s ? 1 + int(std::find(g_streams.begin(), g_streams.end(), s) - g_streams.begin()) : 0);
    g_record += line;
    enqueue(s);
    const int n = (int)block.x;
    if ((int)g_fib.size() < n) g_fib.resize(n);
    g_wave.resize((n + 63) / 64);
    Block lb{nullptr, 0};
    g_lds = lds ? guarded(lds, &lb) : nullptr;
    g_body = &body;
    g_block_dim = {block.x, 1, 1};
    g_grid_dim = {grid.x, grid.y, grid.z};
    for (unsigned by = 0; by < grid.y; ++by)
        for (unsigned bx = 0; bx < grid.x; ++bx) {
            g_block = {bx, by, 0};
            for (int k = 0; k < n; ++k) {
                Fiber& f = g_fib[k];
                if (!f.stack)
                    f.stack = (char*)mmap(nullptr, kStack, PROT_READ | PROT_WRITE,
                                          MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
                void** top = (void**)(f.stack + kStack) - 2;   // entry() starts with the stack 8 off 16
                *top = (void*)entry;
                f.sp = top - 6;
                f.tid = {(unsigned)k, 0, 0};
                f.st = kReady;
            }
            for (;;) {
                for (size_t w = 0; w < g_wave.size(); ++w) run_wave((int)w, n);
                bool again = false;
                for (int k = 0; k < n; ++k)
                    if (g_fib[k].st == kBlock) { g_fib[k].st = kReady; again = true; }
                if (!again) break;
            }
        }
    if (lb.base) munmap(lb.base, lb.len);
    g_cur = -1;
}
}  // namespace emu
