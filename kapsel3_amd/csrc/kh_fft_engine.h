// kh_fft_engine.h -- short DFTs in registers, the butterflies of the FFT
// engines (kh_wave_fft.h, kh_col_fft.h).
#pragma once

#include "kh_common.h"

namespace kh {

// ---------------------------------------------------------------- DFTs
template <typename T, int R, bool FWD>
struct Dft;

template <typename T, bool FWD>
struct Dft<T, 2, FWD> {
    __device__ __forceinline__ static void run(cpx<T> *v) {
        cpx<T> a = v[0], b = v[1];
        v[0]     = cadd(a, b);
        v[1]     = csub(a, b);
    }
};

template <typename T, bool FWD>
struct Dft<T, 3, FWD> {
    __device__ __forceinline__ static void run(cpx<T> *v) {
        const T s3 = (T)0.86602540378443864676372317075294;  // sqrt(3)/2
        cpx<T>  t1 = cadd(v[1], v[2]);
        cpx<T>  t2 = csub(v[0], cscale(t1, (T)0.5));
        cpx<T>  d  = cscale(csub(v[1], v[2]), s3);
        cpx<T>  md = cmul_mi<T, FWD>(d);  // -i*s3*(v1-v2) forward
        v[0]       = cadd(v[0], t1);
        v[1]       = cadd(t2, md);
        v[2]       = csub(t2, md);
    }
};

template <typename T, bool FWD>
struct Dft<T, 4, FWD> {
    __device__ __forceinline__ static void run(cpx<T> *v) {
        cpx<T> a = cadd(v[0], v[2]), b = csub(v[0], v[2]);
        cpx<T> c = cadd(v[1], v[3]), d = cmul_mi<T, FWD>(csub(v[1], v[3]));
        v[0]     = cadd(a, c);
        v[1]     = cadd(b, d);
        v[2]     = csub(a, c);
        v[3]     = csub(b, d);
    }
};

template <typename T, bool FWD>
struct Dft<T, 8, FWD> {
    __device__ __forceinline__ static void run(cpx<T> *v) {
        const T h = (T)0.70710678118654752440084436210485;  // 1/sqrt(2)
        cpx<T>  e[4] = {v[0], v[2], v[4], v[6]};
        cpx<T>  o[4] = {v[1], v[3], v[5], v[7]};
        Dft<T, 4, FWD>::run(e);
        Dft<T, 4, FWD>::run(o);
        // o[k] *= W8^k, W8 = exp(-+ 2 pi i / 8)
        cpx<T> o1 = FWD ? cmk((o[1].x + o[1].y) * h, (o[1].y - o[1].x) * h)
                        : cmk((o[1].x - o[1].y) * h, (o[1].y + o[1].x) * h);
        cpx<T> o2 = cmul_mi<T, FWD>(o[2]);
        cpx<T> o3 = FWD ? cmk((o[3].y - o[3].x) * h, -(o[3].x + o[3].y) * h)
                        : cmk(-(o[3].x + o[3].y) * h, (o[3].x - o[3].y) * h);
        v[0] = cadd(e[0], o[0]);
        v[4] = csub(e[0], o[0]);
        v[1] = cadd(e[1], o1);
        v[5] = csub(e[1], o1);
        v[2] = cadd(e[2], o2);
        v[6] = csub(e[2], o2);
        v[3] = cadd(e[3], o3);
        v[7] = csub(e[3], o3);
    }
};

}  // namespace kh
