// A HIP runtime of host memory and kernels that do not run, for tests of the
// library's host logic without a device (tests/test_host_cpu.py): loaded before
// libparm_hip.so, its functions take the runtime's place.  Allocations can be
// refused, a freed block's address is given out again, a launch can be refused, and what a
// launch reports to the host (skin flags, build reports, sums) is scripted.
// A launch that would go through a null list, or one smaller than the launch
// takes it for, is counted (hh_bad) instead of made.  Compiled for the host only.
#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <string>
#include <vector>

#include "../parm_amd/csrc/kernels.hpp"

using namespace parm;

namespace {

constexpr size_t kSlot = size_t(1) << 28;  // address space per small allocation
size_t g_limit = ~size_t(0);
std::map<void *, size_t> g_live;      // allocation -> its size
std::vector<void *> g_free;           // slots, the last one freed first
std::map<const void *, std::string> g_name;
std::string g_log, g_refuse;
int g_graphs = 0, g_bad = 0, g_overflows = 0, g_fail_in = 0;
bool g_capturing = false;
hipError_t g_last = hipSuccess;
std::deque<uint32_t> g_flags;         // of the next skin tests
std::deque<unsigned long long> g_max; // fullest rows of the next list builds
unsigned long long g_entries = 2;     // entries of every list built

struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
std::vector<Config> g_config;

hipError_t err(hipError_t e) {
    if (e != hipSuccess) g_last = e;
    return e;
}

size_t room(const void *p) {
    auto it = g_live.find(const_cast<void *>(p));
    return it == g_live.end() ? 0 : it->second;
}

void list_used(const void *nbr, size_t words) {
    if (room(nbr) < words * sizeof(uint32_t)) g_bad++;
}

void used(const void *p) {
    if (room(p) == 0) g_bad++;
}

template <typename T>
T arg(void **a, int k) {
    return *static_cast<T *>(a[k]);
}

uint32_t next_flag() {
    if (g_flags.empty()) return 0;
    const uint32_t f = g_flags.front();
    g_flags.pop_front();
    return f;
}

// What a step launch's reduction of the test before it tells the host.
void step_flag(const ReduceBuf &R) {
    if (R.g.nprev <= 0) return;
    const uint32_t stop = kFlagRebuild | kFlagNonFinite | kFlagStopped;
    if (R.g.gate && (*R.g.gate & stop)) {
        *R.g.flag = kFlagStopped;
        return;
    }
    const uint32_t fl = next_flag();
    *R.g.flag = fl;
    *R.g.hflag = (R.g.seq << kFlagBits) | fl;
}

void run(const std::string &name, void **a) {
    auto is = [&](const char *s) { return name.find(s) != std::string::npos; };
    if (is("k_build_stats")) {
        auto *r = arg<BuildReport *>(a, 6);
        const int cap = arg<int>(a, 8);
        unsigned long long mx = 4;
        if (!g_max.empty()) {
            mx = g_max.front();
            g_max.pop_front();
        }
        if (r) {
            r->sum = g_entries;
            r->max = mx;
            r->flag = 0;
            r->ntiles = arg<const int *>(a, 5) ? 1 : 0;
            r->smax = r->ntiles ? 8 : 0;
            r->bad = 0;
            r->ok = r->ntiles && mx <= (unsigned long long)cap;
            r->seq = arg<uint32_t>(a, 7);
        }
        if (auto *v = arg<uint32_t *>(a, 9))
            *v = mx <= (unsigned long long)cap ? 0u : (uint32_t)kFlagStopped;
    } else if (is("k_tile_extremes")) {
        int *info = arg<int *>(a, 1);
        info[0] = 1;
        info[1] = 8;
        info[2] = 0;
    } else if (is("k_finalize_sums")) {
        const ReduceBuf R = arg<ReduceBuf>(a, 1);
        for (int k = 0; R.rec && k < kRedWidth; k++) R.rec[k].seq = R.rseq;
    } else if (is("k_finalize")) {
        const ReduceBuf R = arg<ReduceBuf>(a, 1);
        *R.hflag = (R.g.seq << kFlagBits) | next_flag();
    } else if (is("k_force_tiled") || is("7k_force")) {
        const AtomArrays A = arg<AtomArrays>(a, 0);
        const ListView Lv = arg<ListView>(a, 1);
        if (Lv.built) list_used(Lv.nbr, (size_t)Lv.wcap * Lv.tpa * Lv.npad);
        used(A.pos_in);
        step_flag(arg<ReduceBuf>(a, 5));
    } else if (is("k_batch_force")) {
        const ListView Lv = arg<ListView>(a, 1);
        if (Lv.built) list_used(Lv.nbr, (size_t)Lv.wcap * Lv.tpa * Lv.npad);
    } else if (is("k_batch_build")) {
        list_used(arg<uint32_t *>(a, 7), (size_t)arg<int>(a, 5) * arg<int>(a, 6));
        if (g_overflows > 0 && !g_capturing) {
            g_overflows--;
            *arg<uint32_t *>(a, 15) |= kFlagOverflow;
        }
    } else if (is("k_build_list")) {
        list_used(arg<uint32_t *>(a, 16), (size_t)arg<int>(a, 14) * arg<int>(a, 15));
        for (int k : {7, 17, 18}) used(arg<void *>(a, k));
    } else if (is("k_build_tiled")) {
        list_used(arg<void *>(a, 19), (size_t)arg<int>(a, 16) * arg<int>(a, 17) / 2);
        for (int k : {0, 1, 10, 20, 21}) used(arg<void *>(a, k));
    } else if (is("k_cell_scan")) {
        for (int k : {2, 4}) used(arg<void *>(a, k));
    } else if (is("k_tile_plan")) {
        for (int k : {5, 7, 8}) used(arg<void *>(a, k));
    }
}

}  // namespace

extern "C" {

// ------------------------------------------------------- the test's controls
void hh_reset() {
    g_limit = ~size_t(0);
    g_log.clear();
    g_refuse.clear();
    g_graphs = g_bad = g_overflows = g_fail_in = 0;
    g_last = hipSuccess;
    g_entries = 2;
    g_flags.clear();
    g_max.clear();
}
void hh_alloc_limit(size_t bytes) { g_limit = bytes; }
void hh_fail_at(int k) { g_fail_in = k; }  // the k-th allocation from here
void hh_refuse(const char *kernel) { g_refuse = kernel; }
void hh_flag(uint32_t f) { g_flags.push_back(f); }
void hh_row(unsigned long long m) { g_max.push_back(m); }
void hh_entries(unsigned long long m) { g_entries = m; }
void hh_overflows(int n) { g_overflows = n; }
int hh_graphs() { return g_graphs; }
int hh_bad() { return g_bad; }
const char *hh_log() { return g_log.c_str(); }
void hh_clear_log() { g_log.clear(); }

// ------------------------------------------------------------- registration
void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
    g_name[fn] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    g_config.push_back({g, b, lds, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
    const Config c = g_config.back();
    g_config.pop_back();
    *g = c.grid;
    *b = c.block;
    *lds = c.lds;
    *s = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3, dim3, void **a, size_t, hipStream_t) {
    const std::string &name = g_name[fn];
    if (!g_refuse.empty() && name.find(g_refuse) != std::string::npos)
        return err(hipErrorInvalidConfiguration);
    g_log += name + "\n";
    run(name, a);
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "refused"; }

// ------------------------------------------------------------------- memory
hipError_t hipMalloc(void **p, size_t n) {
    *p = nullptr;
    if (n > g_limit || (g_fail_in > 0 && --g_fail_in == 0)) return err(hipErrorOutOfMemory);
    if (n <= kSlot && !g_free.empty()) {
        *p = g_free.back();
        g_free.pop_back();
    } else {
        *p = mmap(nullptr, n > kSlot ? n : kSlot, PROT_READ | PROT_WRITE,
                  MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
        if (*p == MAP_FAILED) return err(hipErrorOutOfMemory);
    }
    g_live[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    const size_t n = room(p);
    g_live.erase(p);
    if (n <= kSlot)
        g_free.push_back(p);
    else
        munmap(p, n);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) {
    *d = h;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    if (!d || !s) return err(hipErrorInvalidValue);
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    if (!d) return err(hipErrorInvalidValue);
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static std::vector<double> scratch(1 << 21);
    *p = scratch.data();
    return hipSuccess;
}

// ------------------------------------------------- device, streams, events
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
// (hipGetDeviceProperties is a macro for this name)
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    p->sharedMemPerBlock = 64 * 1024;
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = reinterpret_cast<hipEvent_t>(1);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}

// ------------------------------------------------------------------- graphs
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    g_capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    g_capturing = false;
    *g = reinterpret_cast<hipGraph_t>(1);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    g_graphs++;
    *e = reinterpret_cast<hipGraphExec_t>(1);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }

}  // extern "C"
