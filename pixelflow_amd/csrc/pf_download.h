// pf_download.h -- fields from the device layouts into host arrays (pf_download.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

#include <mutex>

#include "pf_layout.h"

namespace pf {

// Pinned chunk buffers, one for a field of a single chunk, else two, of at most 8 MB (one row
// where a row is longer), kept by their owner from its first download until release.
struct Downloader {
    void *pin[2] = {nullptr, nullptr};
    hipEvent_t done[2] = {nullptr, nullptr};
    size_t cap = 0;
    // The field src (colour-split or natural layout) after all work queued on st, into host
    // storage with leading dimensions ldi >= m + 2 and ldj >= n + 2; returns when it is there.
    // Calls of several threads take turns.
    hipError_t get(hipStream_t st, const PfGeom &g, bool split, const double *src, double *host, int64_t ldi,
                   int64_t ldj);
    void release();

   private:
    std::mutex turn;   // of the buffers
    hipError_t reserve(size_t bytes, int buffers);
    hipError_t chunks(hipStream_t st, const PfGeom &g, bool split, const double *src, double *host, int64_t ldi,
                      int64_t ldj);
};

}  // namespace pf
