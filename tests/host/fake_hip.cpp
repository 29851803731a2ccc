// fake_hip.cpp -- the HIP runtime calls that libsjf makes, on the CPU and without a device: memory
// comes from one reserved range that is never handed out twice, copies are plain copies, kernels do
// not run but are recorded.  Loaded before libsjf it lets a test fail a chosen allocation and see
// what the host code then launches: a launch whose argument table names freed memory, or whose grid
// HIP refuses, is recorded as such.
#include <cxxabi.h>
#include <sys/mman.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

struct dim3 {
    uint32_t x, y, z;
};

namespace {
constexpr int kOk = 0, kInvalidValue = 1, kOutOfMemory = 2, kInvalidConfiguration = 9;
constexpr size_t kRange = size_t(1) << 42;

struct Launch {
    std::string kernel;
    dim3 grid, block;
    bool refused;
    int stale;  // words of its argument table that name freed memory
    std::string table;
};

struct State {
    char* base = nullptr;
    size_t used = 0, live_bytes = 0;
    std::map<uintptr_t, size_t> live;
    std::map<void*, size_t> host;  // pinned
    size_t host_bytes = 0;
    std::map<const void*, std::string> kernels;
    std::map<const void*, std::pair<void*, size_t>> vars;
    long countdown = -1;  // allocations until one fails; -1: none does
    long allocations = 0;
    int bad_copies = 0;  // copies from, to, or word passes over memory that is not live
    Launch last_step;
    long steps = 0, launches = 0, refused = 0, entries = 0, shared = 0;
    std::string log, words;
    dim3 grid, block;
    size_t shmem = 0;
    void* stream = nullptr;
    int error = kOk;
};
State& st() {
    static State* s = new State();
    return *s;
}

bool in_range(uintptr_t p) {
    const State& s = st();
    return s.base && p >= (uintptr_t)s.base && p < (uintptr_t)s.base + kRange;
}
// [p, p + n) within one live allocation
bool is_live(uintptr_t p, size_t n) {
    const auto& m = st().live;
    auto it = m.upper_bound(p);
    if (it == m.begin()) return false;
    --it;
    return p + n <= it->first + it->second;
}
bool fine(const void* p, size_t n) { return !in_range((uintptr_t)p) || is_live((uintptr_t)p, n); }

void* take(size_t n) {
    State& s = st();
    if (!s.base) {
        s.base = (char*)mmap(nullptr, kRange, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
        if (s.base == MAP_FAILED) abort();
    }
    n = (n + 4095) & ~size_t(4095);
    if (s.used + n > kRange) abort();
    char* p = s.base + s.used;
    s.used += n;
    return p;
}
void clear(void* p, int v, size_t n) {
    const uintptr_t lo = ((uintptr_t)p + 4095) & ~uintptr_t(4095), hi = ((uintptr_t)p + n) & ~uintptr_t(4095);
    if (v != 0 || n < 1 << 20 || !in_range((uintptr_t)p)) {
        memset(p, v, n);
        return;
    }
    memset(p, 0, lo - (uintptr_t)p);
    madvise((void*)lo, hi - lo, MADV_DONTNEED);
    memset((void*)hi, 0, (uintptr_t)p + n - hi);
}
int copy(void* d, const void* f, size_t n) {
    if (!fine(d, n) || !fine(f, n)) {
        st().bad_copies++;
        return kInvalidValue;
    }
    memcpy(d, f, n);
    return kOk;
}
int result(int rc) {
    if (rc != kOk) st().error = rc;
    return rc;
}
}  // namespace

extern "C" {
// ---- what tests ask and set
void fake_fail_at(long n) { st().countdown = n; }          // the n-th allocation from now (0: the next)
long fake_allocations() { return st().allocations; }
double fake_live_bytes() { return (double)st().live_bytes; }
double fake_host_bytes() { return (double)st().host_bytes; }  // pinned host memory
long fake_steps() { return st().steps; }                   // fused steps launched
int fake_last_stale() { return st().last_step.stale; }
const char* fake_last_kernel() { return st().last_step.kernel.c_str(); }
int fake_last_block() { return (int)st().last_step.block.x; }
int fake_last_grid() { return (int)st().last_step.grid.x; }
size_t fake_last_table(char* out, size_t cap) {            // the argument table of the last fused step
    const std::string& t = st().last_step.table;
    memcpy(out, t.data(), t.size() < cap ? t.size() : cap);
    return t.size();
}
long fake_source_entries() { return st().entries; }  // entries of all source launches (of one engine each)
long fake_source_shared() { return st().shared; }    // of these, on a value that another entry of the launch writes
long fake_refused() { return st().refused; }
int fake_bad_copies() { return st().bad_copies; }
int fake_first_word() {                                    // first given material word of the last k_words launch
    int w = -1;
    if (st().words.size() >= 4) memcpy(&w, st().words.data(), 4);
    return w;
}
const char* fake_log() { return st().log.c_str(); }        // one line per launch since the last clear
void fake_clear_log() { st().log.clear(); }

// ---- memory
int hipMalloc(void** p, size_t n) {
    State& s = st();
    s.allocations++;
    if (s.countdown >= 0 && s.countdown-- == 0) return result(kOutOfMemory);
    *p = take(n);
    s.live[(uintptr_t)*p] = n;
    s.live_bytes += n;
    return kOk;
}
int hipFree(void* p) {
    if (!p) return kOk;
    State& s = st();
    auto it = s.live.find((uintptr_t)p);
    if (it == s.live.end()) return result(kInvalidValue);
    s.live_bytes -= it->second;
    madvise(p, (it->second + 4095) & ~size_t(4095), MADV_DONTNEED);
    s.live.erase(it);
    return kOk;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
    *p = malloc(n);
    if (!*p) return result(kOutOfMemory);
    st().host[*p] = n;
    st().host_bytes += n;
    return kOk;
}
int hipHostFree(void* p) {
    const auto it = st().host.find(p);
    if (it == st().host.end()) return result(kInvalidValue);
    st().host_bytes -= it->second;
    st().host.erase(it);
    free(p);
    return kOk;
}
int hipMemGetInfo(size_t* f, size_t* t) {
    *f = *t = size_t(200) << 30;
    return kOk;
}
int hipMemset(void* p, int v, size_t n) {
    if (!fine(p, n)) return result(kInvalidValue);
    clear(p, v, n);
    return kOk;
}
int hipMemsetAsync(void* p, int v, size_t n, void*) { return hipMemset(p, v, n); }
int hipMemcpyAsync(void* d, const void* f, size_t n, int, void*) { return result(copy(d, f, n)); }
int hipMemcpy2DAsync(void* d, size_t dp, const void* f, size_t fp, size_t w, size_t h, int, void*) {
    for (size_t r = 0; r < h; ++r)
        if (int rc = copy((char*)d + r * dp, (const char*)f + r * fp, w)) return result(rc);
    return kOk;
}

// ---- modules and launches
void** __hipRegisterFatBinary(const void*) {
    static void* m;
    return &m;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    int rc = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &rc);
    st().kernels[host] = rc == 0 ? d : name;
    free(d);
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) { st().vars[var] = {nullptr, size}; }
int hipGetSymbolAddress(void** p, const void* var) {
    auto it = st().vars.find(var);
    if (it == st().vars.end()) return result(kInvalidValue);
    if (!it->second.first) hipMalloc(&it->second.first, it->second.second);
    *p = it->second.first;
    return kOk;
}
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, void* stream) {
    State& s = st();
    s.grid = grid, s.block = block, s.shmem = shmem, s.stream = stream;
    return kOk;
}
int __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, void** stream) {
    State& s = st();
    *grid = s.grid, *block = s.block, *shmem = s.shmem, *stream = s.stream;
    return kOk;
}
int hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t shmem, void*) {
    State& s = st();
    Launch l{s.kernels[f], grid, block, false, 0, ""};
    s.launches++;
    const uint64_t most = uint64_t(1) << 32;
    l.refused = grid.x == 0 || grid.y == 0 || grid.z == 0 || (uint64_t)grid.x * block.x >= most ||
                (uint64_t)grid.y * block.y >= most || (uint64_t)grid.z * block.z >= most ||
                (uint64_t)block.x * block.y * block.z > 1024 || shmem > 160 * 1024;
    char line[64];
    snprintf(line, sizeof line, " %u %u %u x %u%s\n", grid.x, grid.y, grid.z, block.x, l.refused ? " refused" : "");
    s.log += l.kernel + line;
    if (l.refused) {
        s.refused++;
        return result(kInvalidConfiguration);
    }
    if (l.kernel.find("::k_source") != std::string::npos) {
        // SrcTables: sources, and per workgroup its source and entries first .. end - 1; per entry a value's index
        const void* const* t = (const void* const*)args[0];
        const long *first = (const long*)t[2], *end = (const long*)t[3], *idx = (const long*)t[4];
        const int blocks = l.kernel.find("k_source_dft") != std::string::npos ? *(const int*)args[1] : (int)grid.x;
        std::map<long, int> seen;
        for (int b = 0; b < blocks; ++b)
            for (long q = first[b]; q < end[b]; ++q) {
                s.entries++;
                if (seen[idx[q]]++) s.shared++;
            }
    }
    if (l.kernel.find("::k_words<") != std::string::npos) {  // given, matw, seg, lut: all have to be there
        for (int q = 0; q < 4; ++q)
            if (!is_live(*(uintptr_t*)args[q], 1)) s.bad_copies++;
        const auto it = s.live.find(*(uintptr_t*)args[0]);
        if (it != s.live.end()) s.words.assign((const char*)it->first, it->second);
    }
    if (l.kernel.find("k_step") != std::string::npos) {
        s.steps++;
        const auto it = s.live.find(*(uintptr_t*)args[0]);
        if (it == s.live.end()) {
            l.stale = -1;  // the table itself is gone
        } else {
            l.table.assign((const char*)it->first, it->second);
            for (size_t q = 0; q + 8 <= it->second; q += 8) {
                uintptr_t w;
                memcpy(&w, l.table.data() + q, 8);
                if (in_range(w) && !is_live(w, 1)) l.stale++;
            }
        }
        s.last_step = l;
    }
    return kOk;
}

// ---- devices, streams, events, graphs
int hipGetDeviceCount(int* n) {
    *n = 1;
    return kOk;
}
int hipSetDevice(int) { return kOk; }
int hipGetLastError() {
    const int e = st().error;
    st().error = kOk;
    return e;
}
const char* hipGetErrorString(int e) { return e == kOk ? "no error" : e == kOutOfMemory ? "out of memory" : "error"; }
int hipStreamCreateWithFlags(void** s, unsigned) {
    *s = malloc(1);
    return kOk;
}
int hipStreamDestroy(void* s) {
    free(s);
    return kOk;
}
int hipStreamSynchronize(void*) { return kOk; }
int hipStreamBeginCapture(void*, int) { return kOk; }
int hipStreamEndCapture(void*, void** g) {
    *g = malloc(1);
    return kOk;
}
int hipGraphInstantiate(void** x, void*, void*, char*, size_t) {
    *x = malloc(1);
    return kOk;
}
int hipGraphLaunch(void*, void*) { return kOk; }
int hipGraphDestroy(void* g) {
    free(g);
    return kOk;
}
int hipGraphExecDestroy(void* x) {
    free(x);
    return kOk;
}
int hipEventCreate(void** e) {
    *e = malloc(1);
    return kOk;
}
int hipEventDestroy(void* e) {
    free(e);
    return kOk;
}
int hipEventRecord(void*, void*) { return kOk; }
int hipEventSynchronize(void*) { return kOk; }
int hipEventElapsedTime(float* ms, void*, void*) {
    *ms = 1.0f;
    return kOk;
}
}
