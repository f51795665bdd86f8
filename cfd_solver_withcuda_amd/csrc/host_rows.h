// Per-cell results handed to the host (part of the C-ABI translation units).
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>

namespace cfd {

// Rows of a device array in tiled order, handed to a host array in the caller's order: a kernel orders
// them on the device and the copy goes straight to the caller. Bound by that copy: 942k states take
// 2.3 ms on MI355X (the copy 1.7), ordered by the host from a copy of its own 5.9 ms. That is still what
// happens for few cells, and where the device has no room for the ordered rows. Calls from several
// threads take turns. The buffers, up to 68 bytes a cell, stay until the object goes.
class HostRows {
    std::mutex lock_;
    double *buf_ = nullptr;  // ordered rows, as large as the largest so far
    size_t cap_ = 0;
    int *d_iperm_ = nullptr;  // caller cell -> tiled cell
    static hipError_t get_by_host(const std::vector<int> &iperm, int w, const double *d, double *h, hipStream_t st);

  public:
    HostRows() = default;
    HostRows(const HostRows &) = delete;
    HostRows &operator=(const HostRows &) = delete;
    ~HostRows();
    // Cell c's w doubles (1, 4 or 8), h[c w ..] = d[iperm[c] w ..], after the work on `st` so far; done on
    // return. queued: that work has only been launched, so that another launch adds nothing to it.
    hipError_t get(const std::vector<int> &iperm, int w, const double *d, double *h, hipStream_t st, bool queued = false);
};

}  // namespace cfd
