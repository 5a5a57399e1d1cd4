// pf_download.hip -- a field from its device layout into the caller's array.
//
// A kernel writes the field in the host's order (ghosts included, Fortran order) straight
// into pinned host memory, a chunk of rows at a time, and host threads copy each chunk into
// the caller's array while the next one crosses the bus.  The device layout never reaches
// the host.  Measured, ms a field, copying the padded device layout through the runtime's
// staging and a host loop over its cells / this: 97x65x49 0.5-1.0 / 0.2, 256x128x128 11.2 /
// 1.5, 512x256x256 85-92 / 8.5-9.2 (31 GB/s).  The bus bounds it (0.6 ms for 35 MB), with
// the first touch of the caller's pages beside it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <functional>
#include <sched.h>
#include <thread>
#include <vector>

#include "pf_download.h"

namespace pf {

namespace {

// Rows [row0, row0 + rows) of the ghosted field, two values per thread (16-byte stores: the
// bus carries whole 64-byte lines).
template <bool SPLIT>
__global__ __launch_bounds__(256) void k_pack(PfGeom g, const double *__restrict__ src, double *__restrict__ dst,
                                              int row0, unsigned count) {
    const unsigned W = (unsigned)(g.m + 2), e = 2u * (blockIdx.x * 256u + threadIdx.x);
    if (e >= count) return;
    double v[2] = {0., 0.};
#pragma unroll
    for (unsigned q = 0; q < 2; ++q) {
        if (e + q >= count) break;
        const unsigned r = (e + q) / W;
        const int i = (int)(e + q - r * W), row = row0 + (int)r, k = row / g.Y, j = row - k * g.Y;
        v[q] = src[SPLIT ? pf_soff(g, i, j, k) : pf_off(g, i, j, k)];
    }
    if (e + 1 < count) *(double2 *)(dst + e) = make_double2(v[0], v[1]);
    else dst[e] = v[0];
}

constexpr size_t CHUNK = (size_t)8 << 20;
constexpr size_t PER_THREAD = (size_t)1 << 20;   // below this a further thread costs more than it copies
constexpr int THREADS = 8;

int cpu_share() {
    cpu_set_t set;
    CPU_ZERO(&set);
    if (sched_getaffinity(0, sizeof(set), &set) != 0) return 1;
    return std::max(1, CPU_COUNT(&set));
}

// rows [r0, r1) of a chunk that starts at row0
void copy_rows(const PfGeom &g, const double *from, int row0, int r0, int r1, double *host, int64_t ldi, int64_t ldj) {
    const size_t W = (size_t)g.m + 2;
    if (ldi == (int64_t)W && ldj == g.Y) {
        std::memcpy(host + (size_t)(row0 + r0) * W, from + (size_t)r0 * W, (size_t)(r1 - r0) * W * sizeof(double));
        return;
    }
    for (int r = r0; r < r1; ++r) {
        const int row = row0 + r, k = row / g.Y, j = row - k * g.Y;
        std::memcpy(host + (size_t)ldi * ((size_t)j + (size_t)ldj * (size_t)k), from + (size_t)r * W, W * sizeof(double));
    }
}

void copy_chunk(const PfGeom &g, const double *from, int row0, int rows, double *host, int64_t ldi, int64_t ldj,
                int cpus) {
    const size_t bytes = (size_t)rows * (size_t)(g.m + 2) * sizeof(double);
    const int parts = std::max(1, std::min({THREADS, cpus, rows, (int)(bytes / PER_THREAD)}));
    const auto at = [&](int p) { return (int)((int64_t)rows * p / parts); };
    std::vector<std::thread> th;
    int started = 1;
    try {
        th.reserve((size_t)parts);
        for (; started < parts; ++started)
            th.emplace_back(copy_rows, std::cref(g), from, row0, at(started), at(started + 1), host, ldi, ldj);
    } catch (...) {
        // no further thread: this one copies what is left
    }
    copy_rows(g, from, row0, 0, at(1), host, ldi, ldj);
    if (started < parts) copy_rows(g, from, row0, at(started), rows, host, ldi, ldj);
    for (std::thread &t : th) t.join();
}

}  // namespace

void Downloader::release() {
    for (int b = 0; b < 2; ++b) {
        if (pin[b]) (void)hipHostFree(pin[b]);
        if (done[b]) (void)hipEventDestroy(done[b]);
        pin[b] = nullptr;
        done[b] = nullptr;
    }
    cap = 0;
}

hipError_t Downloader::reserve(size_t bytes, int buffers) {
    if (bytes > cap) release();
    hipError_t e = hipSuccess;
    for (int b = 0; b < buffers && e == hipSuccess; ++b) {
        if (pin[b]) continue;
        e = hipHostMalloc(&pin[b], std::max(bytes, cap), hipHostMallocDefault);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&done[b], hipEventDisableTiming);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        release();
    } else {
        cap = std::max(bytes, cap);
    }
    return e;
}

// Without pinned memory: the device layout as it is, put in order here.
static hipError_t get_staged(hipStream_t st, const PfGeom &g, bool split, const double *src, double *host, int64_t ldi,
                             int64_t ldj) {
    std::vector<double> stage((size_t)(split ? 2 * g.HS : g.NS));
    hipError_t e = hipStreamSynchronize(st);
    if (e == hipSuccess) e = hipMemcpy(stage.data(), src, stage.size() * sizeof(double), hipMemcpyDeviceToHost);
    if (e != hipSuccess) return e;
    for (int k = 0; k < g.Z; ++k)
        for (int j = 0; j < g.Y; ++j)
            for (int i = 0; i < g.m + 2; ++i)
                host[(size_t)i + (size_t)ldi * ((size_t)j + (size_t)ldj * (size_t)k)] =
                    stage[(size_t)(split ? pf_soff(g, i, j, k) : pf_off(g, i, j, k))];
    return hipSuccess;
}

hipError_t Downloader::get(hipStream_t st, const PfGeom &g, bool split, const double *src, double *host, int64_t ldi,
                           int64_t ldj) {
    std::lock_guard<std::mutex> lock(turn);
    // the calling thread's device need not be the stream's
    int now = 0;
    hipDevice_t own = 0;
    hipError_t e = hipGetDevice(&now);
    if (e == hipSuccess) e = hipStreamGetDevice(st, &own);
    if (e == hipSuccess && own != now) e = hipSetDevice(own);
    if (e != hipSuccess) return e;
    e = chunks(st, g, split, src, host, ldi, ldj);
    if (own != now) (void)hipSetDevice(now);
    return e;
}

hipError_t Downloader::chunks(hipStream_t st, const PfGeom &g, bool split, const double *src, double *host,
                              int64_t ldi, int64_t ldj) {
    const size_t row = ((size_t)g.m + 2) * sizeof(double);
    const int rows = g.Y * g.Z;
    const int per = (int)std::max<size_t>(1, std::min<size_t>((size_t)rows, CHUNK / row));
    const int n = (rows + per - 1) / per;
    hipError_t e = reserve(((size_t)per * row + 15) / 16 * 16, n > 1 ? 2 : 1);
    if (e != hipSuccess) return get_staged(st, g, split, src, host, ldi, ldj);
    const int cpus = (size_t)per * row >= 2 * PER_THREAD ? cpu_share() : 1;
    auto send = [&](int c) -> hipError_t {
        const int row0 = c * per;
        const unsigned count = (unsigned)(std::min(per, rows - row0)) * (unsigned)(g.m + 2);
        const dim3 grid((count + 511) / 512);
        double *dst = (double *)pin[c & 1];
        if (split) hipLaunchKernelGGL(k_pack<true>, grid, dim3(256), 0, st, g, src, dst, row0, count);
        else hipLaunchKernelGGL(k_pack<false>, grid, dim3(256), 0, st, g, src, dst, row0, count);
        const hipError_t le = hipGetLastError();
        return le != hipSuccess ? le : hipEventRecord(done[c & 1], st);
    };
    e = send(0);
    for (int c = 0; c < n && e == hipSuccess; ++c) {
        if (c + 1 < n) e = send(c + 1);   // its buffer was copied out in the last turn
        if (e != hipSuccess) break;
        e = hipEventSynchronize(done[c & 1]);
        if (e == hipSuccess)
            copy_chunk(g, (const double *)pin[c & 1], c * per, std::min(per, rows - c * per), host, ldi, ldj, cpus);
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(st);   // nothing in flight into the buffers afterwards
    return e;
}

}  // namespace pf
