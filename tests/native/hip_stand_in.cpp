// A stand-in for the HIP runtime on host memory, for CPU tests of the library's host code
// (tests/test_host_faults.py loads it before libpixelflow.so, whose HIP calls then come here).
// Device memory is host memory; kernels do nothing, except that k_clear_u64 clears, k_pack fills
// the rows with its source's first value that is not 0, and a resident sweep's launch counts its
// blocks in (or leaves the give-up bit).  Any call can be
// made to fail, and what the host reads back can be set.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace {

std::mutex g_mu;
thread_local hipError_t t_last = hipSuccess;
struct Fault { int skip, times; hipError_t err; };
std::map<std::string, Fault> g_faults;
std::map<std::string, int> g_calls;
std::map<const void *, std::string> g_kernels;
std::vector<std::string> g_log;
std::map<size_t, std::deque<std::vector<char>>> g_reads;   // by size: what later device-to-host copies deliver
// pending: a resident launch not yet waited for
struct Stream { int pending = 0; unsigned blocks = 0; bool capturing = false; };
int g_give_up = 0, g_good = 0, g_hold_ms = 0;
unsigned g_blocks = 0, g_most_blocks = 0;
int g_inflight = 0, g_most = 0;
size_t g_allocated = 0;
std::map<void *, size_t> g_sizes;

hipError_t done(hipError_t e) {
    if (e != hipSuccess) t_last = e;
    return e;
}
// The scripted error of a call, if it is its turn.
hipError_t scripted(const char *fn) {
    ++g_calls[fn];
    auto it = g_faults.find(fn);
    if (it == g_faults.end()) return hipSuccess;
    Fault &f = it->second;
    if (f.skip > 0) { --f.skip; return hipSuccess; }
    if (f.times == 0) return hipSuccess;
    --f.times;
    return f.err;
}
#define CALL(name)                                   \
    std::lock_guard<std::mutex> lk(g_mu);            \
    const hipError_t e_ = scripted(name);            \
    if (e_ != hipSuccess) return done(e_)

struct Config { dim3 grid, block; size_t shared; hipStream_t st; };
thread_local Config t_config;
constexpr unsigned long long GONE = 1ull << 63;

}  // namespace

extern "C" {

// ---- the script ----
void fake_reset() {
    std::lock_guard<std::mutex> lk(g_mu);
    g_faults.clear();
    g_calls.clear();
    g_log.clear();
    g_reads.clear();
    g_give_up = g_good = g_hold_ms = g_most = 0;
    g_most_blocks = 0;
    t_last = hipSuccess;
}
// Calls of fn fail with err: `times` of them (-1: all) after the first `skip`.
void fake_fail(const char *fn, int skip, int times, int err) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_faults[fn] = Fault{skip, times, (hipError_t)err};
}
// The next `n` resident launches give up.
void fake_give_up(int n) { g_give_up = n; g_good = 0; }
// The `n` after the next `good` do.
void fake_give_up_after(int good, int n) { g_good = good; g_give_up = n; }
// A wait for an event, or for a stream that holds a resident launch, takes this long.
void fake_hold(int ms) { g_hold_ms = ms; }
// The next device-to-host copy of `bytes` bytes delivers `data` (a queue per size).
void fake_read(const void *data, size_t bytes) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_reads[bytes].emplace_back((const char *)data, (const char *)data + bytes);
}
// Launches so far whose kernel's name holds `part`.
int fake_launches(const char *part) {
    std::lock_guard<std::mutex> lk(g_mu);
    int n = 0;
    for (const auto &s : g_log) n += s.find(part) != std::string::npos;
    return n;
}
int fake_calls(const char *fn) { return g_calls[fn]; }
int fake_most_resident() { return g_most; }
unsigned fake_most_resident_blocks() { return g_most_blocks; }
size_t fake_allocated() { return g_allocated; }

// ---- registration and launches ----
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *,
                           dim3 *, int *) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
    t_config = Config{g, b, s, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st) {
    *g = t_config.grid;
    *b = t_config.block;
    *s = t_config.shared;
    *st = t_config.st;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t st) {
    CALL("hipLaunchKernel");
    if (st && ((Stream *)st)->capturing) return hipSuccess;
    const std::string &name = g_kernels[f];
    const bool resident = name.find("k_sor_resident") != std::string::npos;
    if (resident) {
        const hipError_t r = scripted("resident launch");
        if (r != hipSuccess) return done(r);
        Stream *s = (Stream *)st;
        s->pending = 1;
        s->blocks = grid.x;
        g_most = std::max(g_most, ++g_inflight);
        g_blocks += grid.x;
        g_most_blocks = std::max(g_most_blocks, g_blocks);
    }
    if (name.find("k_clear_u64") != std::string::npos)
        std::memset(*(void **)args[0], 0, (size_t) * (int *)args[1] * 8);
    if (name.find("k_pack") != std::string::npos) {
        const double *src = *(const double **)args[1];
        while (*src == 0.) ++src;
        std::fill_n(*(double **)args[2], *(unsigned *)args[4], *src);
    }
    g_log.push_back(name);
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { CALL("hipFuncSetAttribute"); return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int threads, size_t lds) {
    CALL("hipOccupancyMaxActiveBlocksPerMultiprocessor");
    const int by_waves = 16 / std::max(1, (threads + 63) / 64), by_lds = lds ? (int)(163840 / lds) : 32;
    *n = std::min(by_waves, by_lds);
    return hipSuccess;
}

// ---- memory ----
hipError_t hipMalloc(void **p, size_t n) {
    CALL("hipMalloc");
    *p = std::calloc(n ? n : 1, 1);
    g_sizes[*p] = n;
    g_allocated += n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    CALL("hipFree");
    if (p) {
        g_allocated -= g_sizes[p];
        g_sizes.erase(p);
    }
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    CALL("hipHostMalloc");
    *p = std::calloc(n ? n : 1, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = (size_t)288 << 30; return hipSuccess; }
static hipError_t copy(void *dst, const void *src, size_t n, hipMemcpyKind kind, Stream *s) {
    if (kind == hipMemcpyDeviceToHost && s && s->pending == 1 && n == 8) {
        unsigned long long *count = (unsigned long long *)src;
        if (g_good > 0) {
            --g_good;
            *count += s->blocks;
        } else if (g_give_up > 0) {
            --g_give_up;
            *count |= GONE;
        } else {
            *count += s->blocks;
        }
        s->pending = 2;
    }
    std::memcpy(dst, src, n);
    if (kind == hipMemcpyDeviceToHost && !(s && s->pending == 2 && n == 8)) {
        auto it = g_reads.find(n);
        if (it != g_reads.end() && !it->second.empty()) {
            std::memcpy(dst, it->second.front().data(), n);
            it->second.pop_front();
        }
    }
    return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind kind) {
    CALL("hipMemcpy");
    return copy(dst, src, n, kind, nullptr);
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t st) {
    CALL("hipMemcpyAsync");
    Stream *s = (Stream *)st;
    if (kind == hipMemcpyDeviceToHost && s && s->pending == 1 && n == 8) {
        const hipError_t r = scripted("count copy");
        if (r != hipSuccess) return done(r);
    }
    return copy(dst, src, n, kind, s);
}
hipError_t hipMemset(void *p, int v, size_t n) { CALL("hipMemset"); std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) {
    CALL("hipMemsetAsync");
    std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    CALL("hipGetSymbolAddress");
    static char space[1 << 20];
    *p = space;
    return hipSuccess;
}

// ---- devices, streams, events, graphs ----
hipError_t hipGetDevice(int *d) { CALL("hipGetDevice"); *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { CALL("hipSetDevice"); return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
    CALL("hipDeviceGetAttribute");
    *v = 256;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    CALL("hipStreamCreateWithFlags");
    *s = (hipStream_t) new Stream();
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { delete (Stream *)s; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d) { *d = 0; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t st) {
    Stream *s = (Stream *)st;
    int hold = 0;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (s && s->pending) hold = g_hold_ms;
    }
    if (hold) std::this_thread::sleep_for(std::chrono::milliseconds(hold));
    std::lock_guard<std::mutex> lk(g_mu);
    const bool was = s && s->pending;
    if (was) {
        s->pending = 0;
        --g_inflight;
        g_blocks -= s->blocks;
        const hipError_t r = scripted("resident wait");
        if (r != hipSuccess) return done(r);
    }
    return done(scripted("hipStreamSynchronize"));
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { CALL("hipStreamWaitEvent"); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { CALL("hipEventCreate"); *e = (hipEvent_t) new int(0); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    CALL("hipEventCreateWithFlags");
    *e = (hipEvent_t) new int(0);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { delete (int *)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { CALL("hipEventRecord"); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
    if (g_hold_ms) std::this_thread::sleep_for(std::chrono::milliseconds(g_hold_ms));
    CALL("hipEventSynchronize");
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t st, hipStreamCaptureMode) {
    CALL("hipStreamBeginCapture");
    ((Stream *)st)->capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t st, hipGraph_t *g) {
    ((Stream *)st)->capturing = false;
    CALL("hipStreamEndCapture");
    *g = (hipGraph_t) new int(0);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    CALL("hipGraphInstantiate");
    *x = (hipGraphExec_t) new int(0);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { delete (int *)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { delete (int *)x; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    CALL("hipGraphLaunch");
    g_log.push_back("graph");
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipGetLastError() {
    const hipError_t e = t_last;
    t_last = hipSuccess;
    return e;
}

}  // extern "C"
