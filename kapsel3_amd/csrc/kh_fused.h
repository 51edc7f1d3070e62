// kh_fused.h -- host launchers of the dealiasing-pruned fused passes
// (kh_fused.hip).
#pragma once

#include "kh_common.h"

namespace kh {

// y passes on columns kz < TRN_Z; x passes on kept (ky,kz) columns (a
// non-null skip: nothing is done once *skip is nonzero)
template <typename T, bool FWD>
hipError_t cols_y(const Grid &g, const Comps<T> &data, int ncomp, int in_mask, int out_mask, hipStream_t s,
                  const int *skip = nullptr);
template <typename T, bool FWD>
hipError_t cols_x(const Grid &g, const Comps<T> &data, int ncomp, int in_mask, int out_mask, hipStream_t s);
// zeta -> u_hat (truncated) -> inverse x pass, 3 components
template <typename T>
hipError_t x_zeta2u_inv(const Grid &g, const cpx<T> *z0, const cpx<T> *z1, cpx<T> *const u[3], const double *ukdc,
                        hipStream_t s);
// inverse z (3) -> products -> forward z (5); p5[2] may be s3[0], p5[1]
// s3[2] and p5[0] s3[1] (and no other aliasing)
template <typename T>
hipError_t z_adv(const Grid &g, cpx<T> *const s3[3], cpx<T> *const p5[5], hipStream_t s);
// f = up - min(phi_sum,1) u* -> forward z (3), see zw_force; clear: bit 0
// leaves up zero for the next step, bit 1 phi_sum; a non-null `tick` is
// incremented once
template <typename T>
hipError_t z_force(const Grid &g, T *const up[3], T *phis, T *const us[3], cpx<T> *const f[3], int clear,
                   int *tick, hipStream_t s, T *const us2[3] = nullptr, const int *skip = nullptr, Occ occ = {});
// the slip iteration's projection on the pruned transform: forward x (3) of
// the slip force field -> truncation + Solenoidal_uk, its curl into (a0, a1)
// at the kept modes and its k = 0 mode into dc -> inverse x (3), in place
template <typename T>
hipError_t x_slip(const Grid &g, cpx<T> *const f[3], cpx<T> *a0, cpx<T> *a1, double *dc, const int *skip,
                  hipStream_t s);
// forward x (5 products) -> Omega + slaved-Euler update of zeta at the kept
// modes -> FIX_CELL, u*_hat -> inverse x, 3 components (u may be product buffers)
template <typename T>
hipError_t x_ns_u(const Grid &g, const Comps<T> &prod, cpx<T> *z0, cpx<T> *z1, cpx<T> *const u[3], double *ukdc,
                  double dmy0, double dmy1, int fixmask, hipStream_t s);
// forward x (3) -> projection + u* + curl -> zeta, uk_dc; next: also the next
// step's x_zeta2u_inv, its three components in f
template <typename T>
hipError_t x_f_zeta(const Grid &g, cpx<T> *const f[3], cpx<T> *z0, cpx<T> *z1, double *ukdc, bool next, hipStream_t s);
// zeta += (a0, a1) at the kept modes, uk_dc += dc
template <typename T>
hipError_t zeta_add(const Grid &g, cpx<T> *z0, cpx<T> *z1, const cpx<T> *a0, const cpx<T> *a1, double *ukdc,
                    const double *dc, hipStream_t s);
template <typename T>
hipError_t zeta_clean(const Grid &g, cpx<T> *z0, cpx<T> *z1, hipStream_t s);

}  // namespace kh
