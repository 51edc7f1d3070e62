// kh_col_fft.h -- column FFT: lines at a stride, held in the registers of a
// workgroup.
//
// A workgroup transforms C neighbouring columns (C * elem = 128 bytes of every
// line element, more for short lines) of L points. Lane g * C + c holds E points
// of column c in the layouts of the wavefront engine (kh_wave_fft.h, the same
// plans): the first stage's butterflies are formed straight from what the
// lane loads, the last stage's results are stored (or used mode by mode)
// where they are, and only the exchanges between stages go through LDS, two
// for 256 points. Staging the tile in LDS first and last and running every stage
// in and out of LDS, as this engine did before, was 8 LDS passes and 7 barriers
// of a 256-point transform against 4 and 4 (measured at the kernels).
#pragma once

#include "kh_wave_fft.h"

namespace kh {

// Points per lane: 8 (radix 8), 12 where 3 divides L.
template <typename T, int L>
struct ColGeom {
    static constexpr int E  = L % 3 == 0 ? 12 : 8;
    static constexpr int G  = L / E;
    static constexpr int C0 = 128 / (int)sizeof(cpx<T>);
    static constexpr int C  = C0 * G >= 64 ? C0 : 64 / G;  // at least one full wavefront
    static constexpr int NT = C * G;
    // wavefronts per SIMD the x_ns_u pass is compiled for: large workgroups of
    // eight or more wavefronts need 128 registers for two of them (or one of
    // sixteen) to fit a CU (256^3 mixed: 131 registers, one workgroup, 134 us;
    // 128 registers, two workgroups, 103 us)
    static constexpr int WAVES = NT >= 512 && L % 3 != 0 ? 4 : 1;
};

template <typename T, int L, bool FWD, bool REV>
struct ColFft {
    using Geo                 = ColGeom<T, L>;
    static constexpr int      E = Geo::E, G = Geo::G, C = Geo::C, NT = Geo::NT;
    static constexpr WavePlan P  = make_wave_plan(L, E, REV);
    static constexpr int      R0 = P.r[0], RN = P.r[P.n - 1];
    static constexpr int      TW  = wave_tw_size(P) > 0 ? wave_tw_size(P) : 1;
    static constexpr int      BS = C + 1, BUF = L * BS;  // LDS row stride, elements of the exchanges

    __device__ __forceinline__ static void fill_tw(cpx<T> *tw) { WaveFft<T, L, E, FWD, REV>::template fill_tw<NT>(tw); }
    __device__ __forceinline__ static int in_point(int g, int i) {
        return (g + G * (i / R0)) + (i % R0) * (L / R0);
    }
    __device__ __forceinline__ static int out_point(int g, int i) {
        return (g + G * (i / RN)) + (i % RN) * (L / RN);
    }
    // LDS slot of point p, column c: rows of C columns (128 bytes, half the
    // banks) padded by one element, so the rows a stage writes R apart spread
    // over the banks while every access of a stage is one address plus a
    // constant (an XOR swizzle needs a register per access: 80 more in the x
    // passes, one wavefront per SIMD instead of two)
    __device__ __forceinline__ static int at(int p, int c) { return p * BS + c; }

    template <int S>
    __device__ __forceinline__ static void stages(cpx<T> *v, cpx<T> *buf, const cpx<T> *tw, int g, int c) {
        constexpr int R = P.r[S], Ns = P.ns[S], NB = E / R, to = wave_tw_off(P, S);
        static_assert(E % R == 0, "radix must divide the points per lane");
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int k = (int)((unsigned)(g + G * b) % (unsigned)Ns);
            if constexpr (Ns > 1) {
#pragma unroll
                for (int r = 1; r < R; r++) {
                    const cpx<T> w = tw[to + (r - 1) * Ns + k];
                    v[b * R + r]   = FWD ? cmul(v[b * R + r], w) : cmulc(v[b * R + r], w);
                }
            }
            Dft<T, R, FWD>::run(v + b * R);
        }
        if constexpr (S + 1 < P.n) {
            __syncthreads();  // the previous exchange is read out
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const int j    = g + G * b;
                const int k    = (int)((unsigned)j % (unsigned)Ns);
                const int base = (j - k) * R + k;
#pragma unroll
                for (int r = 0; r < R; r++) buf[at(base + r * Ns, c)] = v[b * R + r];
            }
            __syncthreads();
            constexpr int R2 = P.r[S + 1], M2 = L / R2, NB2 = E / R2;
#pragma unroll
            for (int b = 0; b < NB2; b++)
#pragma unroll
                for (int r = 0; r < R2; r++) v[b * R2 + r] = buf[at(g + G * b + r * M2, c)];
            stages<S + 1>(v, buf, tw, g, c);
        }
    }
    // v: E points of lane (g, c), input layout -> output layout; every lane of
    // the workgroup takes part, the twiddle table is complete after the first
    // barrier (the one before the first exchange)
    __device__ __forceinline__ static void run(cpx<T> *v, cpx<T> *buf, const cpx<T> *tw, int g, int c) {
        stages<0>(v, buf, tw, g, c);
        // The results are formed here. Without this the compiler moves the last
        // stage below the conditions the results are used under, and keeps its
        // inputs and twiddles of every component alive until then (340
        // registers instead of 160 in the FP64 x_ns_u).
#pragma unroll
        for (int i = 0; i < E; i++) asm volatile("" : "+v"(v[i].x), "+v"(v[i].y));
    }
};

}  // namespace kh
