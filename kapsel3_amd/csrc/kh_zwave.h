// kh_zwave.h -- z passes on the wavefront-scope FFT engine (kh_zwave.hip).
#pragma once

#include "kh_common.h"
#include "kh_fft.h"

namespace kh {

// rows of L reals -> half spectra (modes kz < kzv, < 0: all L/2+1), ncomp
// components in one launch; spectral rows `pitch` complex apart
template <typename T>
hipError_t zw_r2c(int L, const RIO<T> &io, int ncomp, long long nrows, int pitch, hipStream_t s, int kzv = -1);
// half spectra (modes kz < kzv, rest zero) -> rows of L reals * scale; grid y = component.
// mask (a real field): only 4-point vectors where it is nonzero are written
// (a non-null skip, masked passes only: nothing is done once *skip is nonzero;
// a non-null batch, masked passes only: its batch fields make one launch
// cover the batch's runs)
template <typename T>
hipError_t zw_c2r(int L, const ZIO<T> &io, int ncomp, long long nrows, T scale, int kzv, int pitch,
                  hipStream_t s, const T *mask = nullptr, const int *skip = nullptr, const Grid *batch = nullptr,
                  Occ occ = {});
// sheared advection: inverse z of u and omega (3 + 3) -> u x omega -> forward
// z (3), modes kz < TRN_Z; out may be u
template <typename T>
hipError_t zw_obl_adv(const Grid &g, cpx<T> *const u[3], cpx<T> *const w[3], cpx<T> *const out[3], T scale,
                      hipStream_t s);
// inverse z (3) -> advection products -> forward z (5), modes kz < TRN_Z
template <typename T>
hipError_t zw_adv(const Grid &g, cpx<T> *const s3[3], cpx<T> *const p5[5], T scale, hipStream_t s);
// f = up - min(phi_sum,1) u* -> forward z (3), modes kz < TRN_Z; u* = us +
// us2 when us2 is given, f = up when us is null (then phis may be null: up
// is read at every point instead of where phi_sum != 0); `clear` bit 0 leaves up
// zero, bit 1 phi_sum; a non-null `tick` is incremented once; nothing is
// done once a non-null *skip is nonzero
template <typename T>
struct ZForceIO {
    T       *up[3];
    T       *phis;
    const T *us[3];
    const T *us2[3];
    cpx<T>  *f[3];
    Occ      occ;  // with u* absent: where f may be nonzero (cleared with phi_sum)
};
template <typename T>
hipError_t zw_force(const Grid &g, T *const up[3], T *phis, T *const us[3], cpx<T> *const f[3], int clear,
                    int *tick, hipStream_t s, T *const us2[3] = nullptr, const int *skip = nullptr, Occ occ = {});

}  // namespace kh
