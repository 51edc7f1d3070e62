// kh_transfer.h -- field rows between HBM and the caller's pageable arrays
// (kh_transfer.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <memory>
#include <mutex>

namespace kh {

// One field: `rows` rows of `width` elements, `pitch` elements apart on the
// device (doubles, or floats where fp32 is set); on the host consecutive rows
// of `hwidth` >= width doubles, of which a download sets the last
// hwidth - width to zero and an upload reads none. pitch, width and hwidth
// are even.
struct RowField {
    void     *dev;
    double   *host;
    long long rows;
    int       pitch, width, hwidth;
    bool      fp32;
};

// Pinned staging of one run's transfers: allocated by the first, kept for
// the next ones, given back with the run (release).
struct PinnedRows {
    static constexpr int WORKERS = 8, SLOTS = 2;  // slots per worker
    char      *buf       = nullptr;               // pinned, `slots` slots of slot_bytes
    size_t     slot_bytes = 0;
    int        slots      = 0;
    hipEvent_t done[WORKERS * SLOTS] = {};
    // held by each transfer: threads that read one run at a time share the slots
    std::shared_ptr<std::mutex> lock = std::make_shared<std::mutex>();
    void       release();
};

// Moves nfields fields, ordered after the work on s; returns once the host
// arrays are complete (to_host) or the rows are enqueued and the host arrays
// no longer needed (to the device).
hipError_t move_rows(PinnedRows &st, int device, const RowField *f, int nfields, bool to_host, hipStream_t s);

}  // namespace kh
