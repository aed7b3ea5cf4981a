// A HIP runtime without a device, for tests of the library's host side: it is
// loaded ahead of the real runtime, so that libpicchio_hip.so's calls land
// here. Device memory is host memory under a budget; an address is never
// given out twice, so a use after the free is seen. Kernels do nothing; their
// names, grids and the pointers that they are passed (also inside structures
// passed by value) are kept, per launch and per captured graph. A launch or a
// graph replay that passes a pointer into freed memory counts as stale.
#include <hip/hip_runtime.h>

#include <cxxabi.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#include <map>
#include <string>
#include <vector>

#include "pk_engine.h"

namespace {

struct range { uintptr_t end; bool live; };
struct kernel { std::string name; std::vector<int> words; };      // 8-byte words per argument (0: no pointers)
struct launch { std::string name; dim3 grid; std::vector<uintptr_t> ptrs; };
struct graph { std::vector<launch> nodes; };

std::map<uintptr_t, range> mem;
std::map<const void *, kernel> kernels;
std::vector<launch> log_;
int64_t in_use, peak, budget = -1;
int stale, replays, instantiated, execs;
graph *capture;
dim3 cfg_grid, cfg_block;
size_t cfg_shmem;
hipStream_t cfg_stream;
hipError_t last = hipSuccess;

hipError_t fail(hipError_t e) { return last = e; }

// the range that holds p, or none
std::map<uintptr_t, range>::iterator find(uintptr_t p) {
    auto it = mem.upper_bound(p);
    if (it == mem.begin()) return mem.end();
    --it;
    return p < it->second.end ? it : mem.end();
}
void touch(uintptr_t p) {
    auto it = find(p);
    if (it != mem.end() && !it->second.live) ++stale;
}

// 8-byte words of an argument that may hold pointers
int words_of(const std::string &t) {
    if (t.find('*') != std::string::npos) return 1;
    if (t == "pk_i4_items") return sizeof(pk_i4_items) / 8;
    if (t == "pk_i4_tiles") return sizeof(pk_i4_tiles) / 8;
    if (t == "pk_mfma_args") return sizeof(pk_mfma_args) / 8;
    if (t == "pk_combine_args") return sizeof(pk_combine_args) / 8;
    if (t == "pk_route_args") return sizeof(pk_route_args) / 8;
    if (t == "pk_moe_ffn_args") return sizeof(pk_moe_ffn_args) / 8;
    return 0;
}

}  // namespace

extern "C" {

// ── the tests' side ──
void hh_budget(int64_t bytes) { budget = bytes; }
int64_t hh_in_use() { return in_use; }
int64_t hh_peak(int reset) { const int64_t p = peak; if (reset) peak = in_use; return p; }
int hh_buffers() { int n = 0; for (auto &m : mem) n += m.second.live; return n; }
int hh_stale() { return stale; }
int hh_execs() { return execs; }
int hh_instantiated() { return instantiated; }
int hh_launches() { return (int)log_.size(); }
int64_t hh_groups(int i) { return (int64_t)log_[i].grid.x * log_[i].grid.y * log_[i].grid.z; }
const char *hh_name(int i) { return log_[i].name.c_str(); }
void hh_clear() { log_.clear(); }

// ── the runtime's side ──
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    kernel k;
    int st = 0;
    char *d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    std::string s = d ? d : name;
    free(d);
    // the parameter list: the last top-level parenthesis
    const size_t e = s.rfind(')');
    size_t b = e;
    for (int depth = 0; b != std::string::npos && b > 0; --b) {
        if (s[b] == ')') ++depth;
        if (s[b] == '(' && --depth == 0) break;
    }
    int depth = 0;
    std::string arg;
    for (size_t i = b + 1; i <= e && e != std::string::npos; ++i) {
        if (s[i] == '<' || s[i] == '(') ++depth;
        if (depth == 0 && (s[i] == ',' || i == e)) {
            k.words.push_back(words_of(arg.substr(arg.find_first_not_of(' ') == std::string::npos ? 0 : arg.find_first_not_of(' '))));
            arg.clear();
            continue;
        }
        if (s[i] == '>' || s[i] == ')') --depth;
        arg += s[i];
    }
    std::string n = s.substr(0, b);
    const size_t ns = n.find("(anonymous namespace)::");
    if (ns != std::string::npos) n.erase(ns, 23);
    if (n.compare(0, 5, "void ") == 0) n.erase(0, 5);
    k.name = n;
    kernels[f] = k;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
    cfg_grid = g; cfg_block = b; cfg_shmem = sh; cfg_stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *st) {
    *g = cfg_grid; *b = cfg_block; *sh = cfg_shmem; *st = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t sh, hipStream_t) {
    if (!g.x || !g.y || !g.z || g.y > 65535 || g.z > 65535 || b.x * b.y * b.z > 1024 || sh > 160 * 1024)
        return fail(hipErrorInvalidConfiguration);
    const kernel &k = kernels[f];
    launch l{k.name, g, {}};
    for (size_t i = 0; i < k.words.size(); ++i)
        for (int w = 0; w < k.words[i]; ++w) {
            uintptr_t p;
            memcpy(&p, (const char *)args[i] + 8 * w, 8);
            if (find(p) != mem.end()) l.ptrs.push_back(p);
        }
    if (capture) {
        capture->nodes.push_back(l);
        return hipSuccess;
    }
    for (uintptr_t p : l.ptrs) touch(p);
    log_.push_back(l);
    return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t n) {
    *p = nullptr;
    if (budget >= 0 && in_use + (int64_t)n > budget) return fail(hipErrorOutOfMemory);
    const size_t len = (n + 4095) & ~(size_t)4095;
    // low halves of the addresses: none that a small int (beside 32 bits of
    // padding in a structure) could be taken for
    constexpr uintptr_t LO = 0x10000000, HI = 0xf0000000;
    if (len > HI - LO) return fail(hipErrorOutOfMemory);
    static uintptr_t next = 0x5a0000000000ull + LO;
    if ((next & 0xffffffffu) + len > HI) next = (next & ~(uintptr_t)0xffffffffu) + 0x100000000ull + LO;
    void *m = mmap((void *)next, len, PROT_READ | PROT_WRITE,
                   MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE | MAP_FIXED_NOREPLACE, -1, 0);
    next += len;
    if (m == MAP_FAILED) return fail(hipErrorOutOfMemory);
    mem[(uintptr_t)m] = {(uintptr_t)m + n, true};
    in_use += (int64_t)n;
    if (in_use > peak) peak = in_use;
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    auto it = mem.find((uintptr_t)p);
    if (it == mem.end() || !it->second.live) return fail(hipErrorInvalidValue);
    it->second.live = false;
    const size_t n = it->second.end - it->first;
    in_use -= (int64_t)n;
    madvise(p, (n + 4095) & ~(size_t)4095, MADV_DONTNEED);        // (the address stays taken)
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = calloc(1, n)) ? hipSuccess : fail(hipErrorOutOfMemory); }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    touch((uintptr_t)d);
    touch((uintptr_t)s);
    memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
    if (capture) {
        launch l{"memcpy", dim3(1), {}};
        for (uintptr_t p : {(uintptr_t)d, (uintptr_t)s})
            if (find(p) != mem.end()) l.ptrs.push_back(p);
        capture->nodes.push_back(l);
        return hipSuccess;
    }
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    touch((uintptr_t)d);
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *a = nullptr;
    if (!a) a = mmap(nullptr, 64 << 20, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    *p = a;
    return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { capture = new graph(); return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    *g = (hipGraph_t)capture;
    capture = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
    *e = (hipGraphExec_t) new graph(*(graph *)g);
    ++execs;
    ++instantiated;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    for (const launch &l : ((graph *)e)->nodes) {
        for (uintptr_t p : l.ptrs) touch(p);
        log_.push_back(l);
    }
    ++replays;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete (graph *)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete (graph *)e; --execs; return hipSuccess; }

hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *t, hipEvent_t, hipEvent_t) { *t = 0.0f; return hipSuccess; }

}  // extern "C"
