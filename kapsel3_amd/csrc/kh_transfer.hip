// kh_transfer.hip -- field rows between HBM and the caller's pageable arrays.
//
// Device rows are padded (spectra) or unpadded (real fields) and in the
// field precision; the host's are the reference's padded doubles. A strided
// copy by the runtime moves such rows one by one (7 us a row here: 0.45 s for
// one 256^3 field of 65536 rows, 7 ms for a 32^3 one). Instead a kernel
// gathers whole chunks of rows straight into pinned host memory over the
// link, converting as it goes, and host threads copy finished chunks into the
// caller's array while the next ones arrive; uploads run the same way back.
// Each worker thread owns every WORKERS-th chunk and two slots, so there is no
// hand-over between threads. The link and the first touch of the caller's pages are
// what bounds it: measured figures at move_rows.
#include "kh_transfer.h"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <new>
#include <thread>
#include <vector>

namespace kh {

namespace {

constexpr int    TR_NT = 256;
constexpr size_t CHUNK = 2u << 20;  // bytes of host rows per slot: 40 us on the link, a launch is 5

struct alignas(16) d2 {
    double x, y;
};
template <typename T>
struct alignas(2 * sizeof(T)) t2 {
    T x, y;
};

// Two elements per lane: consecutive lanes write (read) consecutive 16 bytes
// of the pinned rows.
template <typename T, bool OUT>
__global__ __launch_bounds__(TR_NT) void k_rows(T *__restrict__ dev, d2 *__restrict__ host, int rows, int pitch,
                                                int width, int hwidth) {
    const unsigned w2 = (unsigned)hwidth / 2, n = (unsigned)rows * w2;
    for (unsigned e = blockIdx.x * TR_NT + threadIdx.x; e < n; e += gridDim.x * TR_NT) {
        const unsigned row = e / w2, k = 2 * (e - row * w2);
        t2<T>         *p   = reinterpret_cast<t2<T> *>(dev + (size_t)row * pitch + k);
        if (OUT) {
            d2 v = {0.0, 0.0};
            if (k < (unsigned)width) {
                const t2<T> a = *p;
                v             = {(double)a.x, (double)a.y};
            }
            host[e] = v;
        } else if (k < (unsigned)width) {
            const d2 v = host[e];
            *p         = {(T)v.x, (T)v.y};
        }
    }
}

struct Chunk {
    const RowField *f;
    long long       row;
    int             rows;
    size_t          bytes() const { return (size_t)rows * f->hwidth * sizeof(double); }
    double         *host() const { return f->host + row * f->hwidth; }
};

template <typename T, bool OUT>
hipError_t launch(const Chunk &c, void *slot, hipStream_t s) {
    const size_t   n      = (size_t)c.rows * (c.f->hwidth / 2);
    const unsigned blocks = (unsigned)std::min<size_t>((n + TR_NT - 1) / TR_NT, 1024);
    hipLaunchKernelGGL((k_rows<T, OUT>), dim3(blocks), dim3(TR_NT), 0, s, (T *)c.f->dev + c.row * c.f->pitch, (d2 *)slot,
                       c.rows, c.f->pitch, c.f->width, c.f->hwidth);
    return hipGetLastError();
}
hipError_t launch(const Chunk &c, void *slot, bool out, hipStream_t s) {
    if (c.f->fp32) return out ? launch<float, true>(c, slot, s) : launch<float, false>(c, slot, s);
    return out ? launch<double, true>(c, slot, s) : launch<double, false>(c, slot, s);
}

hipError_t reserve(PinnedRows &st, int slots, size_t slot_bytes) {
    if (st.slots < slots || st.slot_bytes < slot_bytes) {
        st.release();
        hipError_t e = hipHostMalloc((void **)&st.buf, (size_t)slots * slot_bytes, hipHostMallocDefault);
        if (e != hipSuccess) {
            (void)hipGetLastError();  // not the next launch's
            st.buf = nullptr;
            return e;
        }
        st.slots      = slots;
        st.slot_bytes = slot_bytes;
    }
    for (int i = 0; i < slots; i++)
        if (!st.done[i]) {
            hipError_t e = hipEventCreateWithFlags(&st.done[i], hipEventDisableTiming);
            if (e != hipSuccess) {
                (void)hipGetLastError();
                st.done[i] = nullptr;
                return e;
            }
        }
    return hipSuccess;
}

// Without pinned memory: copies by the runtime, row by row where the rows
// have gaps, converted on the host where the device holds floats.
hipError_t move_pageable(const RowField &f, bool out, hipStream_t s) {
    const size_t esz = f.fp32 ? sizeof(float) : sizeof(double), dpitch = esz * f.pitch, w = esz * f.width;
    const size_t hpitch = sizeof(double) * f.hwidth;
    hipError_t   e;
    if (!f.fp32) {
        e = out ? hipMemcpy2DAsync(f.host, hpitch, f.dev, dpitch, w, f.rows, hipMemcpyDeviceToHost, s)
                : hipMemcpy2DAsync(f.dev, dpitch, f.host, hpitch, w, f.rows, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
    } else {
        std::vector<float> tmp((size_t)f.rows * f.width);
        if (!out)
            for (long long r = 0; r < f.rows; r++)
                for (int k = 0; k < f.width; k++) tmp[(size_t)r * f.width + k] = (float)f.host[r * f.hwidth + k];
        e = out ? hipMemcpy2DAsync(tmp.data(), w, f.dev, dpitch, w, f.rows, hipMemcpyDeviceToHost, s)
                : hipMemcpy2DAsync(f.dev, dpitch, tmp.data(), w, w, f.rows, hipMemcpyHostToDevice, s);
        const hipError_t e2 = hipStreamSynchronize(s);  // also after an error: tmp goes
        if (e == hipSuccess) e = e2;
        if (out && e == hipSuccess)
            for (long long r = 0; r < f.rows; r++)
                for (int k = 0; k < f.width; k++) f.host[r * f.hwidth + k] = tmp[(size_t)r * f.width + k];
    }
    if (out && e == hipSuccess)
        for (long long r = 0; r < f.rows; r++) std::fill(f.host + r * f.hwidth + f.width, f.host + (r + 1) * f.hwidth, 0.0);
    return e;
}

// chunks w, w + step, w + 2 step, ... through slots w * SLOTS ..
hipError_t work(PinnedRows &st, const Chunk *c, int n, int w, int step, bool out, hipStream_t s) {
    constexpr int B = PinnedRows::SLOTS;
    hipError_t    e = hipSuccess;
    auto          slot = [&](int k) { return w * B + k % B; };
    auto          buf  = [&](int k) { return st.buf + (size_t)slot(k) * st.slot_bytes; };
    auto          send = [&](int k) {
        if ((e = launch(c[w + k * step], buf(k), out, s)) != hipSuccess) return false;
        return (e = hipEventRecord(st.done[slot(k)], s)) == hipSuccess;
    };
    const int mine = w < n ? (n - w + step - 1) / step : 0;
    if (out) {
        for (int k = 0; k < std::min(B, mine); k++)
            if (!send(k)) return e;
        for (int k = 0; k < mine; k++) {
            if ((e = hipEventSynchronize(st.done[slot(k)])) != hipSuccess) return e;
            memcpy(c[w + k * step].host(), buf(k), c[w + k * step].bytes());
            if (k + B < mine && !send(k + B)) return e;
        }
    } else {
        for (int k = 0; k < mine; k++) {
            // the kernel that last read this slot is done
            if (k >= B && (e = hipEventSynchronize(st.done[slot(k)])) != hipSuccess) return e;
            memcpy(buf(k), c[w + k * step].host(), c[w + k * step].bytes());
            if (!send(k)) return e;
        }
        for (int k = std::max(0, mine - B); k < mine; k++)
            if ((e = hipEventSynchronize(st.done[slot(k)])) != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

void PinnedRows::release() {
    if (buf) (void)hipHostFree(buf);
    buf        = nullptr;
    slot_bytes = 0;
    slots      = 0;
    for (hipEvent_t &e : done) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
}

// Measured on kh_get_fluid (two spectral fields), against the strided copies
// by the runtime: 256^3 FP64 903 -> 6.0 ms (45 GB/s), 128^3 FP64 218 -> 1.5 ms,
// 32^3 FP64 14.2 -> 0.11 ms, 256^3 mixed (which converted on the host) 57 -> 6.1
// ms, 512^3 mixed 422 -> 44 ms. Where the pinned memory is not to be had for
// every worker one worker takes its two slots, and without those the runtime copies.
static hipError_t move_rows_on(PinnedRows &st, int device, const RowField *f, int nfields, bool to_host, hipStream_t s) {
    std::vector<Chunk> c;
    size_t             most = 0;
    for (int i = 0; i < nfields; i++) {
        const size_t    row = (size_t)f[i].hwidth * sizeof(double);
        const long long per = std::max<long long>(1, (long long)(CHUNK / row));
        for (long long r = 0; r < f[i].rows; r += per) {
            c.push_back({&f[i], r, (int)std::min(per, f[i].rows - r)});
            most = std::max(most, c.back().bytes());
        }
    }
    const int n = (int)c.size();
    if (n == 0) return hipSuccess;
    most = (most + 4095) / 4096 * 4096;
    // one worker, the calling thread, while all chunks fit its slots
    int workers = std::max(1, std::min(PinnedRows::WORKERS, n / PinnedRows::SLOTS));
    if (reserve(st, workers * PinnedRows::SLOTS, most) != hipSuccess) {
        workers = 1;
        if (reserve(st, PinnedRows::SLOTS, most) != hipSuccess) {
            hipError_t e = hipSuccess;
            for (int i = 0; i < nfields && e == hipSuccess; i++) e = move_pageable(f[i], to_host, s);
            return e;
        }
    }
    if (workers == 1) return work(st, c.data(), n, 0, 1, to_host, s);
    std::atomic<int> err{(int)hipSuccess};
    auto             run = [&](int w) {
        hipError_t r = hipSetDevice(device);
        if (r == hipSuccess) r = work(st, c.data(), n, w, workers, to_host, s);
        if (r != hipSuccess) err.store((int)r);
    };
    std::vector<std::thread> t;
    std::vector<int>         here;  // the calling thread's share
    t.reserve(workers);
    here.reserve(workers);
    here.push_back(0);
    for (int w = 1; w < workers; w++) {
        try {
            t.emplace_back(run, w);
        } catch (const std::exception &) {  // no thread to be had: the caller does it
            here.push_back(w);
        }
    }
    for (int w : here) run(w);
    for (std::thread &x : t) x.join();
    return (hipError_t)err.load();
}

hipError_t move_rows(PinnedRows &st, int device, const RowField *f, int nfields, bool to_host, hipStream_t s) {
    std::lock_guard<std::mutex> held(*st.lock);
    int                         dev = device;
    hipError_t                  e   = hipGetDevice(&dev);
    if (e == hipSuccess && dev != device) e = hipSetDevice(device);  // the caller's may be another
    if (e != hipSuccess) return e;
    try {
        e = move_rows_on(st, device, f, nfields, to_host, s);
    } catch (const std::bad_alloc &) {  // no exception leaves a C entry
        e = hipErrorOutOfMemory;
    }
    if (dev != device) (void)hipSetDevice(dev);
    return e;
}

}  // namespace kh
