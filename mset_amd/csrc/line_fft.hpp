// line_fft.hpp -- transforms of a few lines per workgroup with the points in registers in between.
//
// A workgroup holds TL lines of N points, thread t line t % TL and the E points j + r N / E of it (j = t / TL,
// r < E).  The first and the last radix of a plan are E, so these points are both the input of the first
// Stockham stage and the output of the last: between two transforms of the same lines they stay in
// registers, and a transform costs one LDS exchange per stage boundary and one barrier per exchange (two
// exchange buffers alternate).  Twiddles live in registers, loaded once per kernel.
#pragma once
#include <hip/hip_runtime.h>
#include "fft_lds.hpp"

namespace mset {

template <int N> struct LinePlan;
template <> struct LinePlan<16>  { static constexpr int S = 2; static constexpr int R[4] = {4, 4, 1, 1}; };
template <> struct LinePlan<24>  { static constexpr int S = 3; static constexpr int R[4] = {2, 6, 2, 1}; };
template <> struct LinePlan<32>  { static constexpr int S = 3; static constexpr int R[4] = {4, 2, 4, 1}; };
template <> struct LinePlan<48>  { static constexpr int S = 3; static constexpr int R[4] = {4, 3, 4, 1}; };
template <> struct LinePlan<64>  { static constexpr int S = 3; static constexpr int R[4] = {4, 4, 4, 1}; };
template <> struct LinePlan<96>  { static constexpr int S = 3; static constexpr int R[4] = {4, 6, 4, 1}; };
template <> struct LinePlan<128> { static constexpr int S = 3; static constexpr int R[4] = {4, 8, 4, 1}; };
template <> struct LinePlan<256> { static constexpr int S = 4; static constexpr int R[4] = {4, 4, 4, 4}; };

template <int N, int TL> struct Line {
    using P = LinePlan<N>;
    static constexpr int E = P::R[0];          // points per thread
    static constexpr int T = N / E;            // threads per line
    static constexpr int NT = T * TL;          // threads per workgroup
    static constexpr int RM = P::S > 2 ? P::R[1] : 2;   // radix of the second stage
    // LDS slot of a point: TL lines side by side, one pad group after every 4 points.  With 4 lines, 8 lanes of
    // consecutive j (one pass of 64-bit accesses over the banks) then fall on 8 different 32-byte groups in
    // the first stages' writes, and on at most two shared ones otherwise.
    static constexpr int HALF = (N + N / 4) * TL;
    static constexpr int LDS_ELEMS = 2 * HALF;
    static __device__ __forceinline__ int slot(int pos, int line) { return (pos + (pos >> 2)) * TL + line; }
    float2* s;                                 // two exchange buffers
    int buf, line, j;
    float2 w1[RM - 1], w2[3], wl[E - 1];       // twiddles of the second, third (of four) and last stage

    __device__ __forceinline__ void init(float2* lds, const float2* __restrict__ tw) {
        s = lds;
        buf = 0;
        line = threadIdx.x % TL;
        j = threadIdx.x / TL;
        if constexpr (P::S > 2) {
#pragma unroll
            for (int r = 1; r < RM; ++r) w1[r - 1] = tw[(j % E) * r * (N / (E * RM))];
        }
        if constexpr (P::S == 4) {
#pragma unroll
            for (int r = 1; r < 4; ++r) w2[r - 1] = tw[(j % (E * RM)) * r * (N / (E * RM * 4))];
        }
#pragma unroll
        for (int r = 1; r < E; ++r) wl[r - 1] = tw[j * r];
    }

    // a middle stage of radix R and span NS
    template <int R, int NS, bool INV, int NW> __device__ __forceinline__ void mid(const float2 (&w)[NW]) {
        const float2* a = s + buf;
        buf = HALF - buf;
        float2* b = s + buf;
        constexpr int NB = N / R;                       // butterflies per line
        constexpr int CNT = (NB + T - 1) / T;
        static_assert(CNT == 1 || T % NS == 0, "a thread's butterflies share their twiddles");
#pragma unroll
        for (int c = 0; c < CNT; ++c) {
            const int jj = j + c * T;
            if ((c + 1) * T <= NB || jj < NB) {
                float2 u[R];
#pragma unroll
                for (int r = 0; r < R; ++r) u[r] = a[slot(jj + r * NB, line)];
#pragma unroll
                for (int r = 1; r < R; ++r) u[r] = INV ? cmulc(u[r], w[r - 1]) : cmul(u[r], w[r - 1]);
                DFT<R, INV>::run(u);
                const int base = (jj / NS) * NS * R + jj % NS;
#pragma unroll
                for (int r = 0; r < R; ++r) b[slot(base + r * NS, line)] = u[r];
            }
        }
        __syncthreads();
    }

    // N-point transform of the thread's points, in and out (inverse: without the 1/N).  A buffer is written again
    // only after the barrier that follows the reads of it.
    template <bool INV> __device__ __forceinline__ void dft(float2 (&v)[E]) {
        DFT<E, INV>::run(v);
        float2* a = s + buf;
#pragma unroll
        for (int r = 0; r < E; ++r) a[slot(E * j + r, line)] = v[r];
        __syncthreads();
        if constexpr (P::S > 2) mid<RM, E, INV>(w1);
        if constexpr (P::S == 4) mid<4, E * RM, INV>(w2);
        const float2* b = s + buf;
        buf = HALF - buf;
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = b[slot(j + r * T, line)];
#pragma unroll
        for (int r = 1; r < E; ++r) v[r] = INV ? cmulc(v[r], wl[r - 1]) : cmul(v[r], wl[r - 1]);
        DFT<E, INV>::run(v);
    }
};

}  // namespace mset
