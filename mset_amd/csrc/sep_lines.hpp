// sep_lines.hpp -- the separable position routine with the plane on chip (CDNA4, gfx950): forward-only up to
// N = 128, gradients below, the one-position kernel up to 64.
//
// A separable propagator p(kx, ky) = px(kx) py(ky) makes a propagation step two half-steps along one axis
// each, which commute; alternating their order from plane to plane (see process_sep in multislice.hpp) leaves
// one pass along one axis per plane each way, [F, x p, F^-1, plane step, F, x p, F^-1].  Here a workgroup holds
// all N lines of the plane in registers for a pass and turns it over through LDS once per plane, where the
// general routine transforms along both axes twice per plane.
//
// A line of N = R1 R2 points belongs to T lanes of one wave.
//   layout D (along a real-space axis): lane j < R2 holds points j + R2 r, r < R1
//   layout X (along a Fourier axis):    lane j holds k1 + R1 k2, k2 < R2, for k1 = j (and j + T) < R1
// A forward transform runs D -> X: R1-point transform over r, twiddle W_N^(j k1), exchange, R2-point transform
// over j.  An inverse one runs the same steps backwards, X -> D.  So a transform has a single exchange, which
// stays within a wave: LDS operations of a wave execute in order, and no workgroup barrier is needed (a general
// transform of the LDS engine has two stages with two barriers each).  Twiddles live in registers.  The operands
// of a plane step (transmission, saved wave, gradient slab) are requested before its pass begins.
//
// Lanes of a wave cover 8 points along the line times 8 neighbouring lines (4 x 16 at 16), so arrays of either
// orientation are accessed in runs of 8 elements and need no second layout: the orientation of a pass is a
// pair of strides, and the host's buffers are those of the general routine (multislice.hpp).
#pragma once
#include <hip/hip_runtime.h>
#include "fft_lds.hpp"
#include "kernels.hpp"
#include "multislice.hpp"

namespace mset {

template <int N> struct SepPlan;
template <> struct SepPlan<16>  { static constexpr int R1 = 4, R2 = 4, T = 4; };
template <> struct SepPlan<24>  { static constexpr int R1 = 4, R2 = 6, T = 8; };
template <> struct SepPlan<32>  { static constexpr int R1 = 4, R2 = 8, T = 8; };
template <> struct SepPlan<48>  { static constexpr int R1 = 6, R2 = 8, T = 8; };
template <> struct SepPlan<64>  { static constexpr int R1 = 8, R2 = 8, T = 8; };
template <> struct SepPlan<96>  { static constexpr int R1 = 12, R2 = 8, T = 8; };
template <> struct SepPlan<128> { static constexpr int R1 = 16, R2 = 8, T = 8; };

// orders the LDS accesses of a wave's lanes (the hardware runs them in order; this keeps the compiler to it)
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// BUF plane buffers: with two, a turn writes the one that the turn before last was read from, and needs one barrier
// (one-position kernel, 64 x 64, 16 planes: 145 -> 141 us; batches at 48, where it costs a workgroup per CU: 206 -> 259).
template <int N, int BUF> struct SepLines {
    using P = SepPlan<N>;
    static constexpr int R1 = P::R1, R2 = P::R2, T = P::T;
    static constexpr int NT = N * T;
    static constexpr int CX = (R1 + T - 1) / T;            // R2-point transforms per lane in layout X
    static constexpr int EM = R1 > CX * R2 ? R1 : CX * R2;  // registers of a lane
    static constexpr int EXP = R2 + 1, LS = R1 * EXP;      // exchange slots: [line][k1][j], odd pitch
    static constexpr int PITCH = N + 4;                    // plane slots: [y][x]
    // the plane and the exchange slots are apart where both fit beside a second workgroup, else they share
    static constexpr bool APART = N <= 64;
    static constexpr int EX_ELEMS = N * LS, PL_ELEMS = N * PITCH;
    static constexpr int LDS_ELEMS = APART ? EX_ELEMS + BUF * PL_ELEMS : (EX_ELEMS > PL_ELEMS ? EX_ELEMS : PL_ELEMS);
    static_assert(BUF == 1 || APART, "a second buffer beside the exchange slots");
    static_assert(N == R1 * R2 && R2 <= T && 64 % T == 0, "a line's lanes are in one wave");

    float2* lds;
    int line, j, pl;     // pl: the plane buffer of the next turn
    float2 w[R1 - 1];    // W_N^(j k1), k1 = 1 .. R1 - 1
    float2 v[EM];

    __device__ __forceinline__ void init(float2* s, const float2* __restrict__ tw) {
        lds = s;
        line = threadIdx.x / T;
        j = threadIdx.x % T;
        pl = APART ? EX_ELEMS : 0;
#pragma unroll
        for (int k = 1; k < R1; ++k) w[k - 1] = tw[jd() * k % N];
    }
    // Addresses are affine in (line, j); left visible, the compiler hoists them all out of the plane loops and keeps
    // a hundred registers live (see RegEngine::opaque)
    __device__ __forceinline__ void opaque() {
        asm volatile("" : "+v"(line), "+v"(j));
        __builtin_assume(line >= 0 && line < N && j >= 0 && j < T);   // 24-bit multiplies and shifts
    }
    // Where a layout has fewer places than lanes (j >= R2 in D, j + c T >= R1 in X), the lanes beyond the last place
    // duplicate it: same point, same values, same addresses written, so no access needs a mask or a branch.  Sums over
    // the points leave them out (own_x, own_d).
    __device__ __forceinline__ int jd() const { return R2 == T ? j : min(j, R2 - 1); }
    __device__ __forceinline__ int jx(int c) const { return (c + 1) * T <= R1 ? j + c * T : min(j + c * T, R1 - 1); }
    __device__ __forceinline__ bool own_d() const { return R2 == T || j < R2; }
    __device__ __forceinline__ bool own_x(int i) const { return (i / R2 + 1) * T <= R1 || j + i / R2 * T < R1; }

    __device__ __forceinline__ void fwd() {
        opaque();
        float2* ex = lds + line * LS;                       // this line's exchange slots
        DFT<R1, false>::run(v);
#pragma unroll
        for (int k = 1; k < R1; ++k) v[k] = cmul(v[k], w[k - 1]);
#pragma unroll
        for (int k = 0; k < R1; ++k) ex[jd() + k * EXP] = v[k];
        wave_lds_fence();
#pragma unroll
        for (int c = 0; c < CX; ++c) {
            const float2* q = ex + jx(c) * EXP;
#pragma unroll
            for (int i = 0; i < R2; ++i) v[c * R2 + i] = q[i];
        }
        wave_lds_fence();
#pragma unroll
        for (int c = 0; c < CX; ++c) DFT<R2, false>::run(v + c * R2);
    }
    __device__ __forceinline__ void inv() {
        opaque();
        float2* ex = lds + line * LS;
#pragma unroll
        for (int c = 0; c < CX; ++c) DFT<R2, true>::run(v + c * R2);
#pragma unroll
        for (int c = 0; c < CX; ++c) {
            float2* q = ex + jx(c) * EXP;
#pragma unroll
            for (int i = 0; i < R2; ++i) q[i] = v[c * R2 + i];
        }
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < R1; ++k) v[k] = ex[jd() + k * EXP];
        wave_lds_fence();
#pragma unroll
        for (int k = 1; k < R1; ++k) v[k] = cmulc(v[k], w[k - 1]);
        DFT<R1, true>::run(v);
    }

    // the points of layout D / X: f(register, lane's part of the point, the register's part)
    template <class F> __device__ __forceinline__ void each_d(const F& f) const {
        const int p = jd();
#pragma unroll
        for (int r = 0; r < R1; ++r) f(r, p, R2 * r);
    }
    template <class F> __device__ __forceinline__ void each_x(const F& f) const {
#pragma unroll
        for (int c = 0; c < CX; ++c) {
            const int p = jx(c);
#pragma unroll
            for (int i = 0; i < R2; ++i) f(c * R2 + i, p, R1 * i);
        }
    }
    // turns the plane over: layout D or X of lines along one axis -> layout D or X of lines along the other.
    // col: the lines written are columns x (points y).
    template <bool FROM_X, bool TO_X> __device__ __forceinline__ void turn(bool col) {
        if constexpr (BUF == 1) __syncthreads();             // the plane slots were read (and, shared, exchanged in)
        opaque();
        float2* pl = lds + this->pl;
        if constexpr (BUF == 2) this->pl = 2 * EX_ELEMS + PL_ELEMS - this->pl;
        const int wl = col ? 1 : PITCH, wp = col ? PITCH : 1;
        auto put = [&](int i, int p, int q) { (pl + line * wl + p * wp)[q * wp] = v[i]; };
        if constexpr (FROM_X) each_x(put);
        else each_d(put);
        __syncthreads();
        auto get = [&](int i, int p, int q) { v[i] = (pl + line * wp + p * wl)[q * wl]; };
        if constexpr (TO_X) each_x(get);
        else each_d(get);
        if constexpr (!APART) __syncthreads();               // before exchanges write the shared slots
    }
};

// One probe position: K_BATCH (gradient terms into slabs), K_FWD (loss) or K_PLAIN (sequential semantics; gradient
// planes to slab 0, probe and position updated).  Reference pairing, stored waves, multislice operator; passes
// X_0 .. X_(2L+3) and scratch planes as in process_sep, all arrays in the layouts of process_position.
template <int N, int KIND, int BUF> __device__ __forceinline__ void position_sep_lines(const PosArgs& A, int k, int slot, int slab,
                                                                               bool first, SepLines<N, BUF>& E, float2* phx, float2* phy,
                                                                               const float2* px, const float2* py, double* red) {
    using Eng = SepLines<N, BUF>;
    constexpr int N2 = N * N, R1 = Eng::R1, R2 = Eng::R2, EM = Eng::EM, NT = Eng::NT;
    constexpr bool GRAD = KIND != K_FWD;
    const int t = threadIdx.x, L = A.L;
    const float inv_n2 = 1.0f / (float)N2;
    float2* save = A.save + (size_t)slot * (L + 2) * N2;
    const bool want_pos = GRAD && (A.want & WANT_POS) != 0;
    const bool want_probe = GRAD && (A.want & WANT_PROBE) != 0;

    // ---- sub-pixel shift factors (Func_generate_probe_wave_scan_sub_pixel.m:4-27), double-precision phase
    const double row = (double)A.xlist[k], col_ = (double)A.ylist[k];
    __syncthreads();                                         // the previous position's factors were read
    for (int i = t; i < 2 * N; i += NT) {
        const int ii = i < N ? i : i - N;
        const double d = (i < N ? row : col_) - (double)A.cent;
        double sn, cs;
        sincos(-2.0 * M_PI * d * shift_grid<N>(ii) / (double)N, &sn, &cs);
        (i < N ? phx : phy)[ii] = make_float2((float)cs, (float)sn);
    }
    __syncthreads();

    // index of point p + q of the line in a row-major [y][x] array (rm) and in a transposed [x][y] one (tm): the lane's
    // part and the register's (a constant for each orientation)
    auto rm = [&](bool col, int p, int q) {
        return Idx{(unsigned)(E.line * (col ? 1 : N) + p * (col ? N : 1)), (unsigned)(q * (col ? N : 1))};
    };
    auto tm = [&](bool col, int p, int q) { return rm(!col, p, q); };
    auto rm_d = [&](bool col, int r) { return rm(col, E.jd(), r * R2); };
    // propagation half-step factors along the pass axis (px, py hold the 1/N of its inverse transform)
    auto times_p = [&](bool col, bool conj) {
        const float2* f = col ? py : px;
        E.each_x([&](int i, int p, int q) { E.v[i] = conj ? cmulc(E.v[i], (f + p)[q]) : cmul(E.v[i], (f + p)[q]); });
    };
    auto phase = [&](bool col, int p, int q) {
        return cmul(col ? (phy + p)[q] : phy[E.line], col ? phx[E.line] : (phx + p)[q]);
    };
    const BufC probe(KIND == K_PLAIN ? A.probe : const_cast<float2*>(A.probeF), N2);
    const BufF MT(A.sqrtM + (size_t)k * N2, N2);             // [x][y]

    // ---- X0 (columns): fftn(probe) .* Phi, inverse along y
    if constexpr (KIND == K_PLAIN) {
        E.each_d([&](int i, int p, int q) { E.v[i] = probe[rm(false, p, q)]; });
        E.fwd();
        E.template turn<true, false>(false);
        E.fwd();
        E.each_x([&](int i, int p, int q) { E.v[i] = cmul(E.v[i], phase(true, p, q)); });
    } else {
        E.each_x([&](int i, int p, int q) { E.v[i] = cmul(probe[tm(true, p, q)], phase(true, p, q)); });
    }
    E.inv();
    E.template turn<false, true>(true);
    // The operands of a plane step are requested as its pass begins; without a gradient below 128 (where registers
    // allow it) already when the previous plane's step has released theirs, half a pass and a turn earlier (12
    // planes of 700 positions at 96: 353 -> 338 us; with a gradient's stores in between it costs 1 to 8 %).
    constexpr bool EARLY = KIND == K_FWD && N < 128;
    float2 o[R1];
    auto want_t = [&](bool col, int a) {
        const BufC ta(A.trans + (size_t)a * N2, N2);
#pragma unroll
        for (int r = 0; r < R1; ++r) o[r] = ta[rm_d(col, r)];
    };
    want_t(false, 0);
    // ---- X1 (rows): inverse along x -> psi0 (kept), x t_0, half-step along x
    {
        const BufC sv(save, N2);
        E.inv();
        E.each_d([&](int r, int, int) {
            const float2 u = cscale(E.v[r], inv_n2);
            if (GRAD) sv.put(rm_d(false, r), u);
            E.v[r] = cmul(u, o[r]);
        });
        if (EARLY && L > 1) want_t(true, 1);
        E.fwd();
        times_p(false, false);
        E.inv();
        E.template turn<false, false>(false);
    }
    // ---- X_(a+1): finish plane a-1's step, keep psi_a, x t_a, start plane a's step
    auto plane_fwd = [&](bool col, int a) __attribute__((always_inline)) {
        const BufC sv(save + (size_t)a * N2, N2);
        if (!EARLY) want_t(col, a);
        E.fwd();
        times_p(col, false);
        E.inv();
        E.each_d([&](int r, int, int) {
            if (GRAD) sv.put(rm_d(col, r), E.v[r]);
            E.v[r] = cmul(E.v[r], o[r]);
        });
        if (EARLY && a + 1 < L) want_t(!col, a + 1);
        E.fwd();
        times_p(col, false);
        E.inv();
        E.template turn<false, false>(col);
    };
    // a pass of each orientation per round, strides and offsets constants; without a gradient from 96 on one body
    // (fewer spilled registers; 128, 12 planes of 700 positions: 545 us against 560)
    if constexpr (KIND != K_FWD || N < 96) {
        for (int a = 1; a < L; a += 2) {
            plane_fwd(true, a);
            if (a + 1 < L) plane_fwd(false, a + 1);
        }
    } else {
        for (int a = 1; a < L; ++a) plane_fwd(a & 1, a);
    }
    // ---- X_(L+1): finish plane L-1's step, keep psi_L, forward along this axis
    float m[EM];
    {
        const bool col = L & 1;
        const BufC sv(save + (size_t)L * N2, N2);
        if (EARLY) E.each_x([&](int i, int p, int q) { m[i] = MT[tm(!col, p, q)]; });
        E.fwd();
        times_p(col, false);
        E.inv();
        if (GRAD) E.each_d([&](int r, int, int) { sv.put(rm_d(col, r), E.v[r]); });
        E.fwd();
        E.template turn<true, false>(col);
    }
    // ---- X_(L+2): forward along the other axis -> exit wave; intensity, loss, residual (STEP02_FORWARD_4D.m:36-49)
    // times conj(p), inverse along this axis
    double err = 0.0;
    {
        const bool col = !(L & 1);
        float* Iout = A.inten ? A.inten + (size_t)k * N2 : nullptr;
        if (!EARLY) E.each_x([&](int i, int p, int q) { m[i] = MT[tm(col, p, q)]; });
        E.fwd();
        E.each_x([&](int i, int p, int q) {
            const float2 u = E.v[i];
            const float I = u.x * u.x + u.y * u.y;
            const int y = col ? p + q : E.line, x = col ? E.line : p + q;
            if (KIND == K_FWD && Iout) Iout[((y + N / 2) % N) * N + (x + N / 2) % N] = I;
            const float d = m[i] - __builtin_amdgcn_sqrtf(I);
            if (E.own_x(i)) err += (double)(d * d);
            if constexpr (GRAD) {
                const float f = 1.0f - m[i] * __builtin_amdgcn_rsqf(I + 1e-30f);
                E.v[i] = cmulc(make_float2(u.x * f, u.y * f), cmul(px[x], py[y]));
            }
        });
        if constexpr (GRAD) {
            E.inv();
            E.template turn<false, true>(col);
        }
    }
    err = block_sum<NT>(err, red);
    if (t == 0) A.err_pos[k - A.obase] = err;
    if constexpr (KIND == K_FWD) return;

    // ---- adjoint (STEP03_BACK.m:12-24): plane a's step in X_(2L+2-a), columns for even a
    double dr = 0.0, dc = 0.0;
    float2 wv[R1];
    float gi[R1];
    auto plane_back = [&](bool col, int a) __attribute__((always_inline)) {
        const bool head = a == L - 1;
        const BufC ws(save + (size_t)(a + 1) * N2, N2);
        const BufF g(A.gslab + ((size_t)slab * L + a) * N2, N2);
        const BufF gin(A.gslab + ((size_t)slab * L + a) * N2, first ? 0u : N2);   // empty view: reads 0
        want_t(col, a);
#pragma unroll
        for (int r = 0; r < R1; ++r) {
            wv[r] = ws[rm_d(col, r)];
            if (KIND == K_BATCH) gi[r] = gin[rm_d(col, r)];
        }
        if (!head) {
            E.fwd();
            times_p(col, true);
        }
        E.inv();
        E.each_d([&](int r, int, int) {
            const float2 u = E.v[r];
            const float2 tc = cconj(o[r]);
            const float gr = -cmul(tc, cmulc(u, wv[r])).y;   // Re(1i * conj(t) * conj(psi) * b)
            g.put(rm_d(col, r), KIND == K_BATCH ? gi[r] + gr : gr);
            E.v[r] = cmul(u, tc);
        });
        if (a == 0 && want_pos) {
            // position terms (STEP03_BACK.m:35-38): MATLAB gradient() of conj(psi0)
            const float2* p0 = save;
            E.each_d([&](int r, int p, int q) {
                const int x = E.line, y = p + q;
                const int xp = min(x + 1, N - 1), xm = max(x - 1, 0), yp = min(y + 1, N - 1), ym = max(y - 1, 0);
                const float2 gx = cscale(csub(p0[y * N + xp], p0[y * N + xm]), xp - xm == 2 ? 0.5f : 1.0f);
                const float2 gy = cscale(csub(p0[yp * N + x], p0[ym * N + x]), yp - ym == 2 ? 0.5f : 1.0f);
                if (!E.own_d()) return;
                dr += (double)(gx.x * E.v[r].x + gx.y * E.v[r].y);
                dc += (double)(gy.x * E.v[r].x + gy.y * E.v[r].y);
            });
        }
        E.fwd();
        if (a > 0) {
            times_p(col, true);
            E.inv();
            E.template turn<false, false>(col);
        }
    };
    for (int a = (L - 1) | 1; a > 0; a -= 2) {
        if (a < L) plane_back(false, a);
        plane_back(true, a - 1);
    }
    if (want_pos) {
        dr = block_sum<NT>(dr, red);
        dc = block_sum<NT>(dc, red);
        if (t == 0) {
            if constexpr (KIND == K_BATCH) {
                A.dpos[2 * (k - A.obase)] = (float)dr;
                A.dpos[2 * (k - A.obase) + 1] = (float)dc;
            } else {
                A.xlist[k] = (float)(row + (double)A.s3 * dr);
                A.ylist[k] = (float)(col_ + (double)A.s3 * dc);
            }
        }
    }
    // ---- X_(2L+3) (rows): forward along x -> fftn(bw); the probe term, shift(bw, -d) = ifftn(fftn(bw) .* conj(Phi))
    if (want_probe) {
        E.template turn<true, false>(true);
        if constexpr (KIND == K_BATCH) {
            const BufC out(A.pslab + (size_t)slab * N2, N2);
            const BufC in(A.pslab + (size_t)slab * N2, first ? 0u : N2);
            float2 o[EM];
            E.each_x([&](int i, int p, int q) { o[i] = in[tm(false, p, q)]; });
            E.fwd();
            E.each_x([&](int i, int p, int q) { out.put(tm(false, p, q), cadd(o[i], cmulc(E.v[i], phase(false, p, q)))); });
        } else {
            E.fwd();
            E.each_x([&](int i, int p, int q) { E.v[i] = cmulc(E.v[i], phase(false, p, q)); });
            E.inv();
            E.template turn<false, true>(false);
            float2 o[R1];
            E.each_d([&](int r, int p, int q) { o[r] = probe[rm(true, p, q)]; });
            E.inv();
            E.each_d([&](int r, int p, int q) {
                probe.put(rm(true, p, q), csub(o[r], cscale(cscale(E.v[r], inv_n2), A.s2)));
            });
        }
    }
}

// Slab of a launch's position p.  The remainder of a uniform division is computed per lane; made scalar again here,
// or every access through a view of the slab becomes a loop over the lanes' (equal) descriptors.
__device__ __forceinline__ int slab_of(int p, int nslab) { return __builtin_amdgcn_readfirstlane(p % nslab); }

// registers for two workgroups per CU at 64, where LDS holds two, and for one of 1024 threads at 128
template <int N> struct SepCfg {
    static constexpr int NT = SepLines<N, 1>::NT;
    static constexpr int MINB = N == 64 || N == 128 ? 4 : N == 96 ? 3 : 1;
};

#define MSET_SEP_LDS(N, BUF)                                                    \
    using Eng = SepLines<N, BUF>;                                               \
    constexpr int NT = Eng::NT;                                                 \
    __shared__ float2 s[Eng::LDS_ELEMS];                                        \
    __shared__ float2 phx[N], phy[N], px[N], py[N];                             \
    __shared__ double red[(NT + 63) / 64];                                      \
    for (int i = threadIdx.x; i < 2 * N; i += NT) (i < N ? px : py)[i % N] = cscale(A.p1d[i], 1.0f / N); \
    __syncthreads();                                                            \
    Eng E;                                                                      \
    E.init(s, A.tw);

template <int N> __global__ __launch_bounds__((SepCfg<N>::NT), (SepCfg<N>::MINB)) void k_sep_batch(PosArgs A) {
    MSET_SEP_LDS(N, (N <= 32 ? 2 : 1))
    for (int p = blockIdx.x; p < A.count; p += gridDim.x) {
        const int k = A.order ? A.order[A.first + p] : A.first + p;
        position_sep_lines<N, K_BATCH>(A, k, blockIdx.x, slab_of(p, A.nslab), p < A.nslab, E, phx, phy, px, py, red);
    }
}

template <int N> __global__ __launch_bounds__((SepCfg<N>::NT), (SepCfg<N>::MINB)) void k_sep_plain(PosArgs A, int k) {
    MSET_SEP_LDS(N, 2)
    position_sep_lines<N, K_PLAIN>(A, k, 0, 0, true, E, phx, phy, px, py, red);
}

// MT: the work items are positions of several tilts (as k_fwd)
template <int N, bool MT> __global__ __launch_bounds__((SepCfg<N>::NT), (SepCfg<N>::MINB)) void k_sep_fwd(PosArgs A) {
    MSET_SEP_LDS(N, (N <= 32 ? 2 : 1))
    for (int p = blockIdx.x; p < A.count; p += gridDim.x) {
        if constexpr (MT) {
            const int item = A.order[p];
            const TiltArgs& T = A.tilts[item >> ITEM_TILT_SHIFT];
            PosArgs B = A;
            B.trans = const_cast<float2*>(T.trans);
            B.probeF = T.probeF;
            B.sqrtM = T.sqrtM;
            B.xlist = T.xlist;
            B.ylist = T.ylist;
            B.err_pos = T.err_pos;
            B.obase = 0;
            position_sep_lines<N, K_FWD>(B, item & ITEM_POS_MASK, blockIdx.x, 0, true, E, phx, phy, px, py, red);
        } else {
            const int k = A.order ? A.order[A.first + p] : A.first + p;
            position_sep_lines<N, K_FWD>(A, k, blockIdx.x, 0, true, E, phx, phy, px, py, red);
        }
    }
}

}  // namespace mset
