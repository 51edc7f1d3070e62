// kh_fft.hip -- 3D real FFT passes on HBM-resident fields (gfx950).
//
// Replaces Ooura's rdft3d/rdft3dsort behind A2a_k / A_k2a
// (fft_wrapper.h:641-681, fftsg3d.c:554-709). Layouts on the device:
//   real     R[x][y][z]   z fastest, NX*NY*NZ values (no padding)
//   spectral S[x][y][kz]  complex, kz = 0..NZ/2 fastest, NX*NY*(NZ/2+1)
// The spectral layout is the reference's ([i][j][2kz] as (re,im)), so host
// transfers of spectral fields are plain copies.
//
// Forward = z-pass (two real rows packed into one complex row, r2c), then
// in-place complex passes along y and along x. Inverse = x, y, then z c2r,
// with the 1/(NX NY NZ) normalisation folded into the last pass. Every pass
// reads and writes each field element once: the z passes on the
// wavefront-scope engine (kh_zwave.hip), the y and x passes a tile of C
// neighbouring columns (C*elem = 128 B per row) in a workgroup's registers
// (kh_col_fft.h).
#include "kh_col_fft.h"
#include "kh_fft.h"
#include "kh_zwave.h"

namespace kh {

// ------------------------------------------------------------ y / x pass
// Lines of L points at stride `lstride`; a tile is C consecutive columns.
// Tile t of outer block o starts at data + o*ostride + t*C; `ncols` columns
// are valid per outer block.
template <typename T, int L, bool FWD>
__global__ __launch_bounds__((ColGeom<T, L>::NT)) void k_fft_strided(Comps<T> data, long long lstride,
                                                                   int ncols, long long ostride, int tiles) {
    using F = ColFft<T, L, FWD, FWD>;
    __shared__ cpx<T> s[F::BUF], tw[F::TW];
    const int  o = blockIdx.x / tiles, t = blockIdx.x - o * tiles;
    const int  g = threadIdx.x / F::C, c = threadIdx.x - g * F::C;
    const bool ok   = t * F::C + c < ncols;
    cpx<T>    *base = data.p[blockIdx.y] + (long long)o * ostride + t * F::C + c;  // one component per grid row
    cpx<T>     v[F::E];
#pragma unroll
    for (int i = 0; i < F::E; i++) v[i] = ok ? base[(long long)F::in_point(g, i) * lstride] : cmk((T)0, (T)0);
    F::fill_tw(tw);  // while the loads are in flight
    F::run(v, s, tw, g, c);
#pragma unroll
    for (int i = 0; i < F::E; i++)
        if (ok) base[(long long)F::out_point(g, i) * lstride] = v[i];
}

// ------------------------------------------------------------ launchers
#define KH_FOR_EACH_L(X) X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512)

bool fft_length_supported(int L) {
    switch (L) {
#define KH_CASE(n) case n:
        KH_FOR_EACH_L(KH_CASE)
        return true;
#undef KH_CASE
        default: return false;
    }
}

template <typename T, bool FWD>
static hipError_t launch_strided(int L, const Comps<T> &data, int ncomp, long long lstride, int ncols,
                                 long long ostride, int nouter, hipStream_t s) {
    switch (L) {
#define KH_CASE(n)                                                                                                 \
    case n: {                                                                                                      \
        using Geo       = ColGeom<T, n>;                                                                           \
        const int tiles = (ncols + Geo::C - 1) / Geo::C;                                                           \
        hipLaunchKernelGGL((k_fft_strided<T, n, FWD>), dim3((unsigned)((long long)tiles * nouter), ncomp), dim3(Geo::NT), \
                           0, s, data, lstride, ncols, ostride, tiles);                                            \
        return hipGetLastError();                                                                                  \
    }
        KH_FOR_EACH_L(KH_CASE)
#undef KH_CASE
        default: return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t fft_z_r2c_multi(const Grid &g, const RIO<T> &io, int ncomp, hipStream_t s, int kzvalid) {
    return zw_r2c<T>(g.nz, io, ncomp, (long long)g.nx * g.ny, g.nzp, s, kzvalid);
}
template <typename T>
hipError_t fft_z_c2r_multi(const Grid &g, const ZIO<T> &io, int ncomp, hipStream_t s, int kzvalid, const T *mask,
                           Occ occ) {
    const T   scale = (T)(1.0 / ((double)g.nx * (double)g.ny * (double)g.nz));
    const int kzv   = kzvalid < 0 ? g.nzh : kzvalid;
    return zw_c2r<T>(g.nz, io, ncomp, (long long)g.nx * g.ny, scale, kzv, g.nzp, s, mask, nullptr, &g, occ);
}
// y: lines along y at stride nzp, columns kz < nzh, one outer block per x
template <typename T, bool FWD>
hipError_t fft_y(const Grid &g, const Comps<T> &data, int ncomp, hipStream_t s) {
    return launch_strided<T, FWD>(g.ny, data, ncomp, g.nzp, g.nzh, (long long)g.ny * g.nzp, g.nx, s);
}
// x: lines along x at stride ny*nzp, columns (y,kz) flattened (the row
// padding columns are transformed too: they hold zeros)
template <typename T, bool FWD>
hipError_t fft_x(const Grid &g, const Comps<T> &data, int ncomp, hipStream_t s) {
    const int M = g.ny * g.nzp;
    return launch_strided<T, FWD>(g.nx, data, ncomp, M, M, 0, 1, s);
}

template <typename T>
hipError_t fft3d_r2c(const Grid &g, const T *real_in, cpx<T> *spec_out, hipStream_t s) {
    hipError_t e;
    if ((e = fft_z_r2c_multi<T>(g, RIO<T>{{real_in}, {spec_out}}, 1, s, -1)) != hipSuccess) return e;
    if ((e = fft_y<T, true>(g, Comps<T>{{spec_out}}, 1, s)) != hipSuccess) return e;
    return fft_x<T, true>(g, Comps<T>{{spec_out}}, 1, s);
}

#define KH_INST(T)                                                                   \
    template hipError_t fft_z_r2c_multi<T>(const Grid &, const RIO<T> &, int, hipStream_t, int); \
    template hipError_t fft_z_c2r_multi<T>(const Grid &, const ZIO<T> &, int, hipStream_t, int, const T *, Occ); \
    template hipError_t fft_y<T, true>(const Grid &, const Comps<T> &, int, hipStream_t);          \
    template hipError_t fft_y<T, false>(const Grid &, const Comps<T> &, int, hipStream_t);         \
    template hipError_t fft_x<T, true>(const Grid &, const Comps<T> &, int, hipStream_t);          \
    template hipError_t fft_x<T, false>(const Grid &, const Comps<T> &, int, hipStream_t);
KH_INST(double)
KH_INST(float)
#undef KH_INST

template hipError_t fft3d_r2c<double>(const Grid &, const double *, cpx<double> *, hipStream_t);

}  // namespace kh
