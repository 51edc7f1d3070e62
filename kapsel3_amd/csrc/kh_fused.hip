// kh_fused.hip -- the dealiasing-pruned, fused FFT passes of the SPM step.
//
// Every spectral field the step transforms is 2/3-truncated on one side of
// the transform (Truncate_two_third_rule, fft_wrapper.h:754-796): inverse
// transforms start from truncated spectra, forward transforms feed consumers
// that only read kept modes. So only the kept part of each pass is touched:
//   y passes : columns kz < TRN_Z only; inverse passes read only kept ky
//              rows (the rest are zero), forward passes write only kept ky
//   x passes : columns (ky, kz) both kept only; forward passes write only
//              kept kx
//   z passes : read/write only kz < TRN_Z
// Pointwise work between two passes on the same axis is fused into one
// kernel: the real-space quadratic products sit between the inverse and the
// forward z pass (k_zw_adv), the construction of u_hat from zeta sits in
// front of the inverse x pass (k_x_zeta2u_inv), -Omega, the slaved-Euler update
// of zeta and u*_hat of the new zeta sit between the products' forward and the
// inverse x pass (k_x_ns_u), and the projection, the addition of u* and the curl
// sit behind the forward x pass (k_x_f_zeta), which in a captured chain of steps
// goes on to the next step's u_hat and inverse x pass.
#include "kh_col_fft.h"
#include "kh_fused.h"
#include "kh_modes.h"
#include "kh_zwave.h"

#include <type_traits>

namespace kh {

// Element e of a spectral field. A field has at most 512 x 512 x 272 complex
// elements, so byte offsets fit 32 bits: one offset register then serves every
// field a lane reads at the same place (the field's base stays scalar), where
// 64-bit addresses took a register pair per access.
template <typename P>
__device__ __forceinline__ P &at(P *field, unsigned e) {
    using C = typename std::conditional<std::is_const<P>::value, const char, char>::type;
    return *reinterpret_cast<P *>(reinterpret_cast<C *>(field) + e * (unsigned)sizeof(P));
}

// ------------------------------------------------------------------------
// Column passes. Y mode: outer block = x, line along y, columns kz < ncols.
// X mode: outer block = kept ky row, line along x, columns kz < ncols.
// in_mask: rows whose wavenumber is truncated are taken as zero (not read).
// out_mask: such rows are not written.
template <typename T, int L, bool FWD, bool XMODE>
__global__ __launch_bounds__((ColGeom<T, L>::NT)) void k_cols(Comps<T> comps, Grid g, int ncols, int in_mask,
                                                            int out_mask, const int *__restrict__ skip) {
    using F = ColFft<T, L, FWD, FWD>;
    if ((skip && *skip) || batch_skip(g)) return;
    cpx<T> *__restrict__ data = brun(comps.p[blockIdx.y], g);  // one component per grid row
    __shared__ cpx<T> s[F::BUF], tw[F::TW];
    const int ntiles = (ncols + F::C - 1) / F::C;
    const int o = blockIdx.x / ntiles, kz0 = (blockIdx.x - o * ntiles) * F::C;
    const int l = threadIdx.x / F::C, c = threadIdx.x - l * F::C;
    unsigned base, lstride;
    int      trn;
    if (XMODE) {
        const int j = kept_index(o, g.ny, g.trn_y);
        base        = (unsigned)j * g.nzp + kz0 + c;
        lstride     = (unsigned)g.ny * g.nzp;
        trn         = g.trn_x;
    } else {
        base    = (unsigned)o * g.ny * g.nzp + kz0 + c;
        lstride = g.nzp;
        trn     = g.trn_y;
    }
    const bool ok = kz0 + c < ncols;
    cpx<T>     v[F::E];
#pragma unroll
    for (int i = 0; i < F::E; i++) {
        const int n = F::in_point(l, i);
        v[i]        = cmk((T)0, (T)0);
        if (ok && (!in_mask || kept1(n > L / 2 ? n - L : n, trn))) v[i] = at(data, base + n * lstride);
    }
    F::fill_tw(tw);  // while the loads are in flight
    F::run(v, s, tw, l, c);
#pragma unroll
    for (int i = 0; i < F::E; i++) {
        const int n = F::out_point(l, i);
        if (ok && (!out_mask || kept1(n > L / 2 ? n - L : n, trn))) at(data, base + n * lstride) = v[i];
    }
}

// The tile of a fused x pass: workgroup -> kept (ky) row and kz columns, lane
// -> column c and its E points of the line along x.
template <typename T, int L>
struct XTile {
    using Geo = ColGeom<T, L>;
    int       l, kz, j, iky;
    bool      ok;
    unsigned  base, lstride;
    __device__ __forceinline__ explicit XTile(const Grid &g) {
        const int ntiles = (g.trn_z + Geo::C - 1) / Geo::C;
        const int o      = blockIdx.x / ntiles;
        l                = threadIdx.x / Geo::C;
        // Lines of 8 and 12 points sit whole in one lane, so l is 0 and every
        // wavenumber a constant, but the compiler finds that out late, when the
        // test for the mean mode has become (ikx | iky | kz) == 0: it then drops an
        // ikx of -1 from the OR instead of making the result -1, and mode
        // (-1, 0, 0) was taken for the mean mode (zeta and uk_dc wrong after a
        // step). With l kept unknown nothing is folded, as at the longer lengths.
        if constexpr (Geo::G == 1) asm volatile("" : "+v"(l));
        kz               = (blockIdx.x - o * ntiles) * Geo::C + (threadIdx.x - l * Geo::C);
        j                = kept_index(o, g.ny, g.trn_y);
        iky              = ky_of(g, j);
        ok               = kz < g.trn_z;
        lstride          = (unsigned)g.ny * g.nzp;
        base             = (unsigned)j * g.nzp + kz;
    }
    __device__ __forceinline__ unsigned elem(int n) const { return base + (unsigned)n * lstride; }
    __device__ __forceinline__ int  c() const { return threadIdx.x - l * Geo::C; }
    __device__ __forceinline__ bool first() const { return blockIdx.x == 0; }  // holds (ky, kz) = (0, 0)
    __device__ __forceinline__ static int ikx(int n) { return n > L / 2 ? n - L : n; }
    __device__ __forceinline__ bool kept(const Grid &g, int n) const { return ok && kept1(ikx(n), g.trn_x); }
};

// ------------------------------------------------------------------------
// u_hat from zeta (Zeta_k2u_k, fft_wrapper.cxx:591-688, on the truncated
// zeta) for one mode; (0,0,0) gives uk_dc.
template <typename T>
__device__ __forceinline__ void zeta_to_uhat(const Grid &g, int ikx, int iky, int kz, cpx<T> d1, cpx<T> d2,
                                             const double *uk, cpx<T> *u) {
    if (ikx == 0 && iky == 0 && kz == 0) {
        u[0] = cmk((T)uk[0], (T)0);
        u[1] = cmk((T)uk[1], (T)0);
        u[2] = cmk((T)uk[2], (T)0);
        return;
    }
    const double kx = g.wave_x * ikx, ky = g.wave_y * iky, kz_ = g.wave_z * kz;
    const double k2 = kx * kx + ky * ky + kz_ * kz_;
    const double ik2 = (k2 > 0.0) ? 1. / k2 : 0.0;
    double       o0r, o0i, o1r, o1i, o2r, o2i;
    if (ikx != 0) {
        o0r = -(1. / kx) * (ky * (double)d1.x + kz_ * (double)d2.x);
        o0i = -(1. / kx) * (ky * (double)d1.y + kz_ * (double)d2.y);
        o1r = d1.x;
        o1i = d1.y;
        o2r = d2.x;
        o2i = d2.y;
    } else if (iky != 0) {
        const double dmy = -(kz_ / ky);
        o0r = d2.x;
        o0i = d2.y;
        o1r = dmy * (double)d1.x;
        o1i = dmy * (double)d1.y;
        o2r = d1.x;
        o2i = d1.y;
    } else {
        o0r = d1.x;
        o0i = d1.y;
        o1r = d2.x;
        o1i = d2.y;
        o2r = 0.0;
        o2i = 0.0;
    }
    const double qx = kx * ik2, qy = ky * ik2, qz = kz_ * ik2;
    u[0] = cmk((T)(-(qy * o2i - qz * o1i)), (T)(qy * o2r - qz * o1r));
    u[1] = cmk((T)(-(qz * o0i - qx * o2i)), (T)(qz * o0r - qx * o2r));
    u[2] = cmk((T)(-(qx * o1i - qy * o0i)), (T)(qx * o1r - qy * o0r));
}

// zeta -> u_hat (3 components) on the kept (ky,kz) columns, then the
// inverse x pass of each component.
template <typename T, int L>
__global__ __launch_bounds__((ColGeom<T, L>::NT)) void k_x_zeta2u_inv(
    Grid g, const cpx<T> *__restrict__ z0, const cpx<T> *__restrict__ z1, cpx<T> *__restrict__ u0,
    cpx<T> *__restrict__ u1, cpx<T> *__restrict__ u2, const double *__restrict__ ukdc) {
    using F = ColFft<T, L, false, false>;
    if (batch_skip(g)) return;
    z0 = brun(z0, g), z1 = brun(z1, g), u0 = brun(u0, g), u1 = brun(u1, g), u2 = brun(u2, g);
    ukdc = brun(ukdc, g);
    __shared__ cpx<T> s[F::BUF], tw[F::TW];
    __shared__ double uk[3];
    const XTile<T, L> t(g);
    cpx<T>            D1[F::E], D2[F::E];
#pragma unroll
    for (int i = 0; i < F::E; i++) {
        const int  n  = F::in_point(t.l, i);
        const bool ok = t.kept(g, n);
        D1[i]         = ok ? at(z0, t.elem(n)) : cmk((T)0, (T)0);
        D2[i]         = ok ? at(z1, t.elem(n)) : cmk((T)0, (T)0);
    }
    F::fill_tw(tw);
    if (threadIdx.x < 3) uk[threadIdx.x] = ukdc[threadIdx.x];
    __syncthreads();
    cpx<T> U[3][F::E];
#pragma unroll
    for (int i = 0; i < F::E; i++) {
        const int n = F::in_point(t.l, i);
        U[0][i] = U[1][i] = U[2][i] = cmk((T)0, (T)0);
        if (t.kept(g, n)) {
            cpx<T> u[3];
            zeta_to_uhat<T>(g, t.ikx(n), t.iky, t.kz, D1[i], D2[i], uk, u);
            U[0][i] = u[0];
            U[1][i] = u[1];
            U[2][i] = u[2];
            __builtin_amdgcn_sched_barrier(0);  // one mode's FP64 temporaries at a time
        }
    }
    cpx<T> *out[3] = {u0, u1, u2};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        F::run(U[d], s, tw, t.l, t.c());
#pragma unroll
        for (int i = 0; i < F::E; i++)
            if (t.ok) at(out[d], t.elem(F::out_point(t.l, i))) = U[d][i];
    }
}

// ------------------------------------------------------------------------
// Forward x pass of the five advection products on the kept (ky,kz)
// columns, per kept mode Omega_k2zeta_k + the slaved-Euler update of zeta
// (NS_solver_slavedEuler, fluid_solver.cxx:348-374), FIX_CELL's zeroing of
// uk_dc (sp_3d_ns.cxx:46-52) and u*_hat of the new zeta, then the inverse x
// pass of its three components: neither the products' spectra nor the new zeta
// are read back from memory. Each product is folded into the two rows of Omega
// its mode stores as soon as it is transformed (8 FP64 registers a mode
// instead of 20), while the next one's loads are in flight. Bound by memory
// latency at two or three workgroups a CU. Against the launches it replaces
// (products' x pass, slaved Euler, zeta -> u_hat): 256^3 mixed 136 -> 103 us
// (3.1 TB/s), 256^3 FP64 199 -> 157 us (4.1 TB/s), 192^3 mixed 61 -> 34 us,
// 512^3 mixed 1320 -> 735 us.
template <typename T, int L, int Q>
__device__ __forceinline__ void adv_products(const Grid &g, const XTile<T, L> &t, const Comps<T> &prod,
                                             cpx<T> (&v)[2][ColGeom<T, L>::E], cpx<double> (&acc)[ColGeom<T, L>::E][2],
                                             cpx<T> *s, const cpx<T> *tw) {
    using F = ColFft<T, L, true, true>;
    if constexpr (Q < 5) {
        if constexpr (Q + 1 < 5) {
            const cpx<T> *src = brun(prod.p[Q + 1], g);
            unsigned      e0  = t.elem(F::in_point(t.l, 0));
            asm volatile("" : "+v"(e0));  // these loads come after the previous product's fold, not all five at once
#pragma unroll
            for (int i = 0; i < F::E; i++)
                v[(Q + 1) & 1][i] =
                    t.ok ? at(src, e0 + (unsigned)(F::in_point(0, i)) * t.lstride) : cmk((T)0, (T)0);
        }
        F::run(v[Q & 1], s, tw, t.l, t.c());
        int l = t.l;
        asm volatile("" : "+v"(l));  // wavenumbers are worked out again for each product, not kept in registers
#pragma unroll
        for (int i = 0; i < F::E; i++) {
            adv_fold<Q, T>(g, XTile<T, L>::ikx(F::out_point(l, i)), t.iky, t.kz, v[Q & 1][i], acc[i]);
            // done here: else the compiler moves the sums to where they are
            // used, below the mode's condition, and keeps all five products
            asm volatile("" : "+v"(acc[i][0].x), "+v"(acc[i][0].y), "+v"(acc[i][1].x), "+v"(acc[i][1].y));
        }
        adv_products<T, L, Q + 1>(g, t, prod, v, acc, s, tw);
    }
}
template <typename T, int L>
__global__ __launch_bounds__((ColGeom<T, L>::NT), (ColGeom<T, L>::WAVES)) void k_x_ns_u(Grid g, Comps<T> prod, cpx<T> *__restrict__ z0,
                                                                cpx<T> *__restrict__ z1, cpx<T> *u0, cpx<T> *u1,
                                                                cpx<T> *u2, double *__restrict__ ukdc, double dmy0,
                                                                double dmy1, int fixmask) {
    using F  = ColFft<T, L, true, true>;
    using Fi = ColFft<T, L, false, false>;
    static_assert(F::RN == Fi::R0, "forward output layout must be the inverse input layout");
    if (batch_skip(g)) return;
    z0 = brun(z0, g), z1 = brun(z1, g), ukdc = brun(ukdc, g);
    __shared__ cpx<T> s[F::BUF], tw[F::TW], twi[Fi::TW];
    __shared__ double uk[3];
    const XTile<T, L> t(g);
    cpx<double>       acc[F::E][2];
    {
        cpx<T>        v[2][F::E];
        const cpx<T> *src = brun(prod.p[0], g);
#pragma unroll
        for (int i = 0; i < F::E; i++) {
            v[0][i]   = t.ok ? at(src, t.elem(F::in_point(t.l, i))) : cmk((T)0, (T)0);
            acc[i][0] = acc[i][1] = {0.0, 0.0};
        }
        F::fill_tw(tw);  // while the loads are in flight
        Fi::fill_tw(twi);
        if (threadIdx.x < 3) {
            const bool fixed = fixmask & (1 << threadIdx.x);
            uk[threadIdx.x]  = fixed ? 0.0 : ukdc[threadIdx.x];
            if (fixed && t.first()) ukdc[threadIdx.x] = 0.0;
        }
        __syncthreads();
        adv_products<T, L, 0>(g, t, prod, v, acc, s, tw);
    }
    cpx<T> U[3][F::E];
#pragma unroll
    for (int i = 0; i < F::E; i++) {
        const int n = F::out_point(t.l, i);
        U[0][i] = U[1][i] = U[2][i] = cmk((T)0, (T)0);
        if (t.kept(g, n)) {
            cpx<T> x0 = at(z0, t.elem(n)), x1 = at(z1, t.elem(n)), u[3];
            slaved_euler_acc<T>(g, t.ikx(n), t.iky, t.kz, acc[i], dmy0, dmy1, x0, x1);
            at(z0, t.elem(n)) = x0;
            at(z1, t.elem(n)) = x1;
            zeta_to_uhat<T>(g, t.ikx(n), t.iky, t.kz, x0, x1, uk, u);
            U[0][i] = u[0];
            U[1][i] = u[1];
            U[2][i] = u[2];
        }
    }
    cpx<T> *out[3] = {brun(u0, g), brun(u1, g), brun(u2, g)};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        Fi::run(U[d], s, twi, t.l, t.c());
#pragma unroll
        for (int i = 0; i < Fi::E; i++)
            if (t.ok) at(out[d], t.elem(Fi::out_point(t.l, i))) = U[d][i];
    }
}

// ------------------------------------------------------------------------
// Forward x pass of the rigidity force on the kept (ky,kz) columns, then per
// kept mode: truncation + Solenoidal_uk (operate_omega.cxx:171-195), the sum
// with u* rebuilt from zeta (the reference's U2zeta_k of u* + f), and
// U_k2zeta_k (fft_wrapper.cxx:407-476). Writes zeta at the kept modes and
// uk_dc += f_hat(0). With the lines in registers 94 to 146 of them instead of
// 220, so two to three workgroups a CU: 512^3 mixed 1104 -> 381 us (3.5 TB/s),
// 256^3 mixed 61 -> 52 us, FP64 83 -> 76 us (4.5 TB/s).
// NEXT: another step follows in the same captured graph, and u_hat of the
// new zeta is formed here and taken through the inverse x pass, in place of
// f, instead of by that step's k_x_zeta2u_inv: the new zeta is not read back,
// and a launch goes (the whole step: 192^3 mixed 324 -> 314 us, 64^3 FP64 88.3 ->
// 86.0, 256^3 mixed 723 -> 712, 256^3 FP64 1272 -> 1257, 512^3 mixed 6.47 -> 6.36 ms).
template <typename T, int L, bool NEXT>
__global__ __launch_bounds__((ColGeom<T, L>::NT)) void k_x_f_zeta(Grid g, cpx<T> *f0, cpx<T> *f1, cpx<T> *f2,
                                                                  cpx<T> *__restrict__ z0, cpx<T> *__restrict__ z1,
                                                                  double *__restrict__ ukdc) {
    using F  = ColFft<T, L, true, true>;
    using Fi = ColFft<T, L, false, false>;
    if (batch_skip(g)) return;
    f0 = brun(f0, g), f1 = brun(f1, g), f2 = brun(f2, g), z0 = brun(z0, g), z1 = brun(z1, g), ukdc = brun(ukdc, g);
    __shared__ cpx<T> s[F::BUF], tw[F::TW], twi[NEXT ? Fi::TW : 1];
    __shared__ double uk[3];
    const XTile<T, L> t(g);
    cpx<T>           *fld[3] = {f0, f1, f2};
    cpx<T>            Fh[3][F::E];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int i = 0; i < F::E; i++)
            Fh[d][i] = t.ok ? at(fld[d], t.elem(F::in_point(t.l, i))) : cmk((T)0, (T)0);
    F::fill_tw(tw);  // while the loads are in flight
    if constexpr (NEXT) Fi::fill_tw(twi);
    if (threadIdx.x < 3) uk[threadIdx.x] = ukdc[threadIdx.x];
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 3; d++) F::run(Fh[d], s, tw, t.l, t.c());
#pragma unroll
    for (int i = 0; i < F::E; i++) {
        const int n = F::out_point(t.l, i), ikx = t.ikx(n), iky = t.iky, kz = t.kz;
        if (!t.kept(g, n)) {
            if constexpr (NEXT) Fh[0][i] = Fh[1][i] = Fh[2][i] = cmk((T)0, (T)0);
            continue;
        }
        const unsigned idx = t.elem(n);
        const double    kx = ikx * g.wave_x, ky = iky * g.wave_y, kzz = kz * g.wave_z;
        const double    K2  = (g.wave_x * ikx) * (g.wave_x * ikx) + (g.wave_y * iky) * (g.wave_y * iky) +
                          (g.wave_z * kz) * (g.wave_z * kz);
        const double IK2 = (K2 > 0.0) ? 1. / K2 : 0.0;
        // Solenoidal_uk on f_hat
        const cpx<T> a = Fh[0][i], b = Fh[1][i], cc = Fh[2][i];
        const double dr = IK2 * ((double)a.x * kx + (double)b.x * ky + (double)cc.x * kzz);
        const double di = IK2 * ((double)a.y * kx + (double)b.y * ky + (double)cc.y * kzz);
        double       fr[3] = {a.x - dr * kx, b.x - dr * ky, cc.x - dr * kzz};
        double       fi[3] = {a.y - di * kx, b.y - di * ky, cc.y - di * kzz};
        // u* rebuilt from the (post-NS, truncated) zeta
        cpx<T> us[3];
        zeta_to_uhat<T>(g, ikx, iky, kz, at(z0, idx), at(z1, idx), uk, us);
        double ur[3], ui[3];
        for (int d = 0; d < 3; d++) {
            ur[d] = (double)us[d].x + fr[d];
            ui[d] = (double)us[d].y + fi[d];
        }
        if (ikx == 0 && iky == 0 && kz == 0) {  // k = 0 stays FP64: uk_dc + sum(f)
            for (int d = 0; d < 3; d++) ukdc[d] = uk[d] + fr[d];
        }
        double ore[3], oim[3];
        ore[0] = -(ky * ui[2] - kzz * ui[1]);
        oim[0] = (ky * ur[2] - kzz * ur[1]);
        ore[1] = -(kzz * ui[0] - kx * ui[2]);
        oim[1] = (kzz * ur[0] - kx * ur[2]);
        ore[2] = -(kx * ui[1] - ky * ui[0]);
        oim[2] = (kx * ur[1] - ky * ur[0]);
        int c0, c1;
        if (ikx != 0) {
            c0 = 1;
            c1 = 2;
        } else if (iky != 0) {
            c0 = 2;
            c1 = 0;
        } else {
            c0 = 0;
            c1 = 1;
        }
        const cpx<T> x0 = cmk((T)ore[c0], (T)oim[c0]), x1 = cmk((T)ore[c1], (T)oim[c1]);
        at(z0, idx) = x0;
        at(z1, idx) = x1;
        if constexpr (NEXT) {
            const double un[3] = {uk[0] + fr[0], uk[1] + fr[1], uk[2] + fr[2]};  // uk_dc, read for k = 0 only
            cpx<T>       u[3];
            zeta_to_uhat<T>(g, ikx, iky, kz, x0, x1, un, u);
            Fh[0][i] = u[0];
            Fh[1][i] = u[1];
            Fh[2][i] = u[2];
        }
        __builtin_amdgcn_sched_barrier(0);  // one mode's FP64 temporaries at a time
    }
    if constexpr (NEXT) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            Fi::run(Fh[d], s, twi, t.l, t.c());
#pragma unroll
            for (int i = 0; i < Fi::E; i++)
                if (t.ok) at(fld[d], t.elem(Fi::out_point(t.l, i))) = Fh[d][i];
        }
    }
}

// The slip iteration's projection (Solenoidal_u, operate_omega.h:105-112,
// which truncates to the 2/3 modes) less its z and y passes: forward x of
// the slip force field's three components on the kept (ky,kz) columns; per
// kept mode truncation + Solenoidal_uk (operate_omega.cxx:171-195) and the
// curl of the projected field (U_k2zeta_k, fft_wrapper.cxx:407-476) into
// (a0, a1), its k = 0 mode into dc; modes beyond the 2/3 rule set to zero;
// then the inverse x pass of each projected component, in place.
template <typename T, int L>
__global__ __launch_bounds__((ColGeom<T, L>::NT)) void k_x_slip(Grid g, cpx<T> *__restrict__ f0, cpx<T> *__restrict__ f1,
                                                              cpx<T> *__restrict__ f2, cpx<T> *__restrict__ a0,
                                                              cpx<T> *__restrict__ a1, double *__restrict__ dc,
                                                              const int *__restrict__ skip) {
    using Ff = ColFft<T, L, true, true>;
    using Fi = ColFft<T, L, false, false>;
    static_assert(Ff::RN == Fi::R0, "forward output layout must be the inverse input layout");
    if (skip && *skip) return;
    __shared__ cpx<T> s[Ff::BUF], twf[Ff::TW], twi[Fi::TW];
    const XTile<T, L> t(g);
    cpx<T>           *F[3] = {f0, f1, f2};
    cpx<T>            Fh[3][Ff::E];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
        for (int i = 0; i < Ff::E; i++)
            Fh[d][i] = t.ok ? at(F[d], t.elem(Ff::in_point(t.l, i))) : cmk((T)0, (T)0);
    Ff::fill_tw(twf);  // while the loads are in flight
    Fi::fill_tw(twi);
#pragma unroll
    for (int d = 0; d < 3; d++) Ff::run(Fh[d], s, twf, t.l, t.c());
#pragma unroll
    for (int i = 0; i < Ff::E; i++) {
        const int n = Ff::out_point(t.l, i), ikx = t.ikx(n), iky = t.iky, kz = t.kz;
        if (!t.kept(g, n)) {
            Fh[0][i] = Fh[1][i] = Fh[2][i] = cmk((T)0, (T)0);
            continue;
        }
        const unsigned idx = t.elem(n);
        const double    kx = ikx * g.wave_x, ky = iky * g.wave_y, kzz = kz * g.wave_z;
        const double    K2  = (g.wave_x * ikx) * (g.wave_x * ikx) + (g.wave_y * iky) * (g.wave_y * iky) +
                          (g.wave_z * kz) * (g.wave_z * kz);
        const double IK2 = (K2 > 0.0) ? 1. / K2 : 0.0;
        // Solenoidal_uk, stored in T as the reference's field is
        const cpx<T> a = Fh[0][i], b = Fh[1][i], cc = Fh[2][i];
        const double dr = IK2 * ((double)a.x * kx + (double)b.x * ky + (double)cc.x * kzz);
        const double di = IK2 * ((double)a.y * kx + (double)b.y * ky + (double)cc.y * kzz);
        const cpx<T> pa = cmk((T)(a.x - dr * kx), (T)(a.y - di * kx));
        const cpx<T> pb = cmk((T)(b.x - dr * ky), (T)(b.y - di * ky));
        const cpx<T> pc = cmk((T)(cc.x - dr * kzz), (T)(cc.y - di * kzz));
        Fh[0][i] = pa;
        Fh[1][i] = pb;
        Fh[2][i] = pc;
        if (ikx == 0 && iky == 0 && kz == 0) {
            dc[0] = pa.x;
            dc[1] = pb.x;
            dc[2] = pc.x;
        }
        double ore[3], oim[3];
        ore[0] = -(ky * (double)pc.y - kzz * (double)pb.y);
        oim[0] = (ky * (double)pc.x - kzz * (double)pb.x);
        ore[1] = -(kzz * (double)pa.y - kx * (double)pc.y);
        oim[1] = (kzz * (double)pa.x - kx * (double)pc.x);
        ore[2] = -(kx * (double)pb.y - ky * (double)pa.y);
        oim[2] = (kx * (double)pb.x - ky * (double)pa.x);
        int c0, c1;
        if (ikx != 0) {
            c0 = 1;
            c1 = 2;
        } else if (iky != 0) {
            c0 = 2;
            c1 = 0;
        } else {
            c0 = 0;
            c1 = 1;
        }
        at(a0, idx) = cmk((T)ore[c0], (T)oim[c0]);
        at(a1, idx) = cmk((T)ore[c1], (T)oim[c1]);
        __builtin_amdgcn_sched_barrier(0);  // one mode's FP64 temporaries at a time
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        Fi::run(Fh[d], s, twi, t.l, t.c());
#pragma unroll
        for (int i = 0; i < Fi::E; i++)
            if (t.ok) at(F[d], t.elem(Fi::out_point(t.l, i))) = Fh[d][i];
    }
}

// zero zeta outside the kept modes (the reference's state there is
// round-off after U2zeta_k; here it is exactly zero)
template <typename T>
__global__ void k_zeta_clean(Grid g, cpx<T> *__restrict__ z0, cpx<T> *__restrict__ z1) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= g.nspec) return;
    const int kz = (int)(idx % g.nzp);
    const long long rest = idx / g.nzp;
    const int j = (int)(rest % g.ny), i = (int)(rest / g.ny);
    if (kz < g.nzh && !kept_mode(g, kx_of(g, i), ky_of(g, j), kz)) {
        z0[idx] = cmk((T)0, (T)0);
        z1[idx] = cmk((T)0, (T)0);
    }
}

// zeta += (a0, a1) and uk_dc += dc: the projected slip field's vorticity
// and mean velocity, added after the slip iteration.
// (a0, a1) hold the 2/3-kept modes only.
template <typename T>
__global__ void k_zeta_add(Grid g, cpx<T> *__restrict__ z0, cpx<T> *__restrict__ z1, const cpx<T> *__restrict__ a0,
                           const cpx<T> *__restrict__ a1, double *__restrict__ ukdc, const double *__restrict__ dc) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx == 0)
        for (int d = 0; d < 3; d++) ukdc[d] += dc[d];
    if (idx >= g.nspec) return;
    const int       kz   = (int)(idx % g.nzp);
    const long long rest = idx / g.nzp;
    const int       j = (int)(rest % g.ny), i = (int)(rest / g.ny);
    if (!kept_mode(g, kx_of(g, i), ky_of(g, j), kz)) return;
    z0[idx] = cadd(z0[idx], a0[idx]);
    z1[idx] = cadd(z1[idx], a1[idx]);
}

// ------------------------------------------------------------ launchers
#define KH_FOR_EACH_L(X) X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512)

static inline int nky(const Grid &g) { return 2 * g.trn_y - 1; }
// kz tiles of a column pass over lines of L points
template <typename T, int L>
static inline int ktiles(const Grid &g) { return (g.trn_z + ColGeom<T, L>::C - 1) / ColGeom<T, L>::C; }

template <typename T, bool FWD>
hipError_t cols_y(const Grid &g, const Comps<T> &data, int ncomp, int in_mask, int out_mask, hipStream_t s,
                  const int *skip) {
    switch (g.ny) {
#define KH_CASE(n)                                                                                                 \
    case n:                                                                                                        \
        hipLaunchKernelGGL((k_cols<T, n, FWD, false>), dim3(g.nx * ktiles<T, n>(g), ncomp, batch_z(g)), dim3(ColGeom<T, n>::NT), 0, s, \
                           data, g, g.trn_z, in_mask, out_mask, skip);                                             \
        return hipGetLastError();
        KH_FOR_EACH_L(KH_CASE)
#undef KH_CASE
        default: return hipErrorInvalidValue;
    }
}

template <typename T, bool FWD>
hipError_t cols_x(const Grid &g, const Comps<T> &data, int ncomp, int in_mask, int out_mask, hipStream_t s) {
    switch (g.nx) {
#define KH_CASE(n)                                                                                                  \
    case n:                                                                                                         \
        hipLaunchKernelGGL((k_cols<T, n, FWD, true>), dim3(nky(g) * ktiles<T, n>(g), ncomp, batch_z(g)), dim3(ColGeom<T, n>::NT), 0, s, \
                           data, g, g.trn_z, in_mask, out_mask, nullptr);                                           \
        return hipGetLastError();
        KH_FOR_EACH_L(KH_CASE)
#undef KH_CASE
        default: return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t x_zeta2u_inv(const Grid &g, const cpx<T> *z0, const cpx<T> *z1, cpx<T> *const u[3], const double *ukdc,
                        hipStream_t s) {
    switch (g.nx) {
#define KH_CASE(n)                                                                                                   \
    case n:                                                                                                          \
        hipLaunchKernelGGL((k_x_zeta2u_inv<T, n>), dim3(nky(g) * ktiles<T, n>(g), 1, batch_z(g)), dim3(ColGeom<T, n>::NT), 0, s, g, z0, z1, u[0], u[1],    \
                           u[2], ukdc);                                                                     \
        return hipGetLastError();
        KH_FOR_EACH_L(KH_CASE)
#undef KH_CASE
        default: return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t z_adv(const Grid &g, cpx<T> *const s3[3], cpx<T> *const p5[5], hipStream_t s) {
    const T scale = (T)(1.0 / ((double)g.nx * (double)g.ny * (double)g.nz));
    return zw_adv<T>(g, s3, p5, scale, s);
}

template <typename T>
hipError_t z_force(const Grid &g, T *const up[3], T *phis, T *const us[3], cpx<T> *const f[3], int clear,
                   int *tick, hipStream_t s, T *const us2[3], const int *skip, Occ occ) {
    return zw_force<T>(g, up, phis, us, f, clear, tick, s, us2, skip, occ);
}

template <typename T>
hipError_t x_ns_u(const Grid &g, const Comps<T> &prod, cpx<T> *z0, cpx<T> *z1, cpx<T> *const u[3], double *ukdc,
                  double dmy0, double dmy1, int fixmask, hipStream_t s) {
    switch (g.nx) {
#define KH_CASE(n)                                                                                                   \
    case n:                                                                                                          \
        hipLaunchKernelGGL((k_x_ns_u<T, n>), dim3(nky(g) * ktiles<T, n>(g), 1, batch_z(g)), dim3(ColGeom<T, n>::NT), 0, s, g, prod, z0, z1, \
                           u[0], u[1], u[2], ukdc, dmy0, dmy1, fixmask);                                             \
        return hipGetLastError();
        KH_FOR_EACH_L(KH_CASE)
#undef KH_CASE
        default: return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t x_f_zeta(const Grid &g, cpx<T> *const f[3], cpx<T> *z0, cpx<T> *z1, double *ukdc, bool next, hipStream_t s) {
    switch (g.nx) {
#define KH_CASE(n)                                                                                                 \
    case n: {                                                                                                      \
        const dim3 grid(nky(g) * ktiles<T, n>(g), 1, batch_z(g)), block(ColGeom<T, n>::NT);                        \
        if (next)                                                                                                  \
            hipLaunchKernelGGL((k_x_f_zeta<T, n, true>), grid, block, 0, s, g, f[0], f[1], f[2], z0, z1, ukdc);    \
        else                                                                                                       \
            hipLaunchKernelGGL((k_x_f_zeta<T, n, false>), grid, block, 0, s, g, f[0], f[1], f[2], z0, z1, ukdc);   \
        return hipGetLastError();                                                                                  \
    }
        KH_FOR_EACH_L(KH_CASE)
#undef KH_CASE
        default: return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t x_slip(const Grid &g, cpx<T> *const f[3], cpx<T> *a0, cpx<T> *a1, double *dc, const int *skip,
                  hipStream_t s) {
    switch (g.nx) {
#define KH_CASE(n)                                                                                                  \
    case n:                                                                                                         \
        hipLaunchKernelGGL((k_x_slip<T, n>), dim3(nky(g) * ktiles<T, n>(g)), dim3(ColGeom<T, n>::NT), 0, s, g, f[0], f[1], f[2], a0, a1, \
                           dc, skip);                                                                               \
        return hipGetLastError();
        KH_FOR_EACH_L(KH_CASE)
#undef KH_CASE
        default: return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t zeta_add(const Grid &g, cpx<T> *z0, cpx<T> *z1, const cpx<T> *a0, const cpx<T> *a1, double *ukdc,
                    const double *dc, hipStream_t s) {
    hipLaunchKernelGGL(k_zeta_add<T>, dim3((unsigned)((g.nspec + 255) / 256)), dim3(256), 0, s, g, z0, z1, a0, a1, ukdc,
                       dc);
    return hipGetLastError();
}

template <typename T>
hipError_t zeta_clean(const Grid &g, cpx<T> *z0, cpx<T> *z1, hipStream_t s) {
    hipLaunchKernelGGL(k_zeta_clean<T>, dim3((unsigned)((g.nspec + 255) / 256)), dim3(256), 0, s, g, z0, z1);
    return hipGetLastError();
}

#define KH_INST(T)                                                                                                  \
    template hipError_t cols_y<T, true>(const Grid &, const Comps<T> &, int, int, int, hipStream_t, const int *);   \
    template hipError_t cols_y<T, false>(const Grid &, const Comps<T> &, int, int, int, hipStream_t, const int *);  \
    template hipError_t cols_x<T, true>(const Grid &, const Comps<T> &, int, int, int, hipStream_t);                \
    template hipError_t cols_x<T, false>(const Grid &, const Comps<T> &, int, int, int, hipStream_t);               \
    template hipError_t x_zeta2u_inv<T>(const Grid &, const cpx<T> *, const cpx<T> *, cpx<T> *const[3],              \
                                        const double *, hipStream_t);                                                          \
    template hipError_t z_adv<T>(const Grid &, cpx<T> *const[3], cpx<T> *const[5], hipStream_t);                   \
    template hipError_t z_force<T>(const Grid &, T *const[3], T *, T *const[3], cpx<T> *const[3], int, int *,          \
                                   hipStream_t, T *const[3], const int *, Occ);                                    \
    template hipError_t x_slip<T>(const Grid &, cpx<T> *const[3], cpx<T> *, cpx<T> *, double *, const int *,          \
                                  hipStream_t);                                                                    \
    template hipError_t x_f_zeta<T>(const Grid &, cpx<T> *const[3], cpx<T> *, cpx<T> *, double *, bool, hipStream_t); \
    template hipError_t x_ns_u<T>(const Grid &, const Comps<T> &, cpx<T> *, cpx<T> *, cpx<T> *const[3], double *,    \
                                  double, double, int, hipStream_t);                                               \
    template hipError_t zeta_clean<T>(const Grid &, cpx<T> *, cpx<T> *, hipStream_t);                               \
    template hipError_t zeta_add<T>(const Grid &, cpx<T> *, cpx<T> *, const cpx<T> *, const cpx<T> *, double *,      \
                                    const double *, hipStream_t);
KH_INST(double)
KH_INST(float)
#undef KH_INST

}  // namespace kh
