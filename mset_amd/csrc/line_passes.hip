// line_passes.hip -- the sequential path spread over the device: one probe position as a chain of
// one-axis passes, each a launch of N / 4 workgroups of 4 lines.
//
// The sequential semantics (Run_MSET_recon.m:134-158) allow one position at a time, and one workgroup
// that carries it through the forward and adjoint sweep leaves 255 of 256 CUs idle and is bound by the
// VALU issue and the LDS latency of its one CU.  With a separable propagator p(kx, ky) = px(kx) py(ky) a
// propagation step is P = Px Py, two transforms-with-product along one axis each, which commute;
// alternating their order from plane to plane (t0, Px Py, t1, Py Px, t2, ...) leaves one pass along one
// axis per plane each way, [F, x p, F^-1, plane step, F, x p, F^-1], and lines of a pass are independent.
// So a position is 2 L + 6 short launches, and what bounds it is the latency of a launch: the load of a
// line written by another CU, four line transforms, the store.
//
// A workgroup takes 4 lines, thread t line t % 4 and points j + r N / 4 (j = t / 4, r < 4): arrays whose
// lines are contiguous are read in 128-byte runs, arrays of the other orientation in 16- or 32-byte runs
// (the whole plane is at most 512 KB and comes from L2 or the MALL).  Four points per thread keep the
// serial work of a wave short (a line transform is 3 exchanges and about 110 VALU operations at 256; with
// 16 points per thread it would be 1 exchange and 400).  A pass reads its input contiguous and writes its
// output transposed for the next pass; all its global operands are requested before the first transform,
// so a pass waits for memory once.
//
// Per position, passes along x (rows, lines y) and y (columns, lines x); X_1 .. X_(2L+3) as in process_sep
// (multislice.hpp), the forward step of plane a in X_(a+1), its adjoint in X_(2L+2-a):
//   PROBE  rows     probe -> F                                    (also writes the sub-pixel shift factors)
//   SHIFT  columns  F -> fftn(probe), x Phi, F^-1
//   FIRST  rows     F^-1 -> psi_0 (kept), x t_0, half-step
//   FWD    both     half-step -> psi_a (kept), x t_a, half-step      a = 1 .. L-1
//   LAST   both     half-step -> psi_L (kept), F
//   EXIT   both     F -> exit wave: loss, residual, x conj(p), F^-1
//   ADJ    both     half-step back, gradient, V += s1 G, x conj(t_a), half-step back     a = L-1 .. 0
//   BACK   rows     F -> fftn(bw), x conj(Phi), F^-1
//   STEP   columns  F^-1 -> probe -= s2 w, position += s3 d
// V is read in a plane's forward pass, which keeps the transmission for the adjoint one, and updated in its adjoint
// pass, so there are no gradient planes, transmission or update launches.  (Forming the transmission again in the
// adjoint pass: 7.56 instead of 7.28 ms for 36 positions at 128 x 128 x 16 planes; with views instead of pointers and
// no branch around the slices 6.63 ms.)  Waves, loss and
// position sums, rounding order of the transmission and the update as in process_position.
//
// Measured per position, before as one workgroup and now: 576 -> 184 us at 128 x 128 x 16 planes (38 launches),
// 4.5 -> 0.45 ms at 256 x 256 x 32 (70); a pass with four transforms takes about 5 us at 128, about 2 of them the
// launch and the loads.
#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "line_fft.hpp"

namespace mset {

namespace {

constexpr int TL = 4;      // lines per workgroup

// sum of one double per thread over the workgroup, in the first thread
template <int NT> __device__ __forceinline__ double group_sum(double v, double* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double u = __shfl_down(v, o, 64);
        // a partial last wave (96 threads) has no lane to add beyond the workgroup's threads
        if (NT % 64 == 0 || (int)threadIdx.x + o < NT) v += u;
    }
    __syncthreads();
    if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (NT + 63) / 64; ++i) s += red[i];
    return s;
}

enum { PROBE, SHIFT, FIRST, FWD, LAST, EXIT, ADJ, BACK, STEP };

template <int N, int KIND, bool COL> __global__ __launch_bounds__(N) void k_line_pass(LineArgs A) {
    using F_ = Line<N, TL>;
    constexpr int N2 = N * N, E = F_::E, T = F_::T, G = N / TL;
    static_assert(F_::NT == N, "launched with N threads");
    __shared__ float2 s[F_::LDS_ELEMS];
    __shared__ double red[(N + 63) / 64];
    F_ F;
    F.init(s, A.tw);
    const int line = blockIdx.x * TL + F.line, j = F.j;
    // index of point r of the thread in arrays with contiguous lines, and in arrays of the other orientation: the
    // thread's part and a constant, through buffer views (with pointers a pass formed 26 addresses by 64-bit multiplies)
    auto own = [&](int r) { return Idx{(unsigned)(line * N + j), (unsigned)(r * T)}; };
    auto oth = [&](int r) { return Idx{(unsigned)(j * N + line), (unsigned)(r * T * N)}; };
    auto along = [&](int r) { return Idx{(unsigned)j, (unsigned)(r * T)}; };
    const BufC in(A.in, N2), out(A.out, N2), wave(A.wave, N2), trans(A.trans, N2);
    const float inv_n = 1.0f / (float)N, inv_n2 = 1.0f / (float)N2;

    // ---- operands, all requested before the first transform
    float2 v[E];
#pragma unroll
    for (int r = 0; r < E; ++r) v[r] = in[own(r)];
    // propagator factors along the pass
    float2 pf[E];
    if constexpr (KIND == FIRST || KIND == FWD || KIND == LAST || KIND == EXIT || KIND == ADJ) {
        const BufC f(A.p1d + (COL ? N : 0), N);
#pragma unroll
        for (int r = 0; r < E; ++r) pf[r] = f[along(r)];
    }
    // the plane's slices: the first four kept for the update, the sum in slice order.  A slice beyond the bin has an
    // empty view (reads 0, drops writes): with a branch around its loads the compiler moved the first addition up to
    // the load, and the pass waited for memory before its first transform.
    constexpr int KEEP = 4;
    float z[KEEP][E], sum[E];
    // (without an object step the adjoint pass has no slices)
    const int z0 = A.a * A.bin, nzp = KIND == ADJ && A.s1 == 0.f ? 0 : min(A.bin, A.nz - z0);
    float* Vp = A.V + (size_t)z0 * N2;
    auto slice = [&](int i) { return BufF(Vp + (size_t)i * N2, i < nzp ? (unsigned)N2 : 0u); };
    auto vox = [&](int r) { return COL ? oth(r) : own(r); };
    if constexpr (KIND == FIRST || KIND == FWD || KIND == ADJ) {
#pragma unroll
        for (int r = 0; r < E; ++r) sum[r] = 0.f;
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
            const BufF V = slice(i);
#pragma unroll
            for (int r = 0; r < E; ++r) z[i][r] = V[vox(r)];
        }
    }
    float2 wv[E], t[E];
    if constexpr (KIND == ADJ) {
#pragma unroll
        for (int r = 0; r < E; ++r) wv[r] = wave[own(r)];
#pragma unroll
        for (int r = 0; r < E; ++r) t[r] = trans[oth(r)];
    }
    float m[E];
    if constexpr (KIND == EXIT) {
        const BufF M(A.sqrtM, N2);
#pragma unroll
        for (int r = 0; r < E; ++r) m[r] = M[COL ? own(r) : oth(r)];
    }
    float2 pr[E];
    const BufC probe(A.probe, N2);
    if constexpr (KIND == STEP) {
#pragma unroll
        for (int r = 0; r < E; ++r) pr[r] = probe[vox(r)];
    }
    // sub-pixel shift factors: phi[0 .. N) along x, phi[N .. 2N) along y
    float2 ph[E];
    if constexpr (KIND == SHIFT || KIND == BACK) {
        const float2 l = A.phi[(COL ? 0 : N) + line];
        const BufC f(A.phi + (COL ? N : 0), N);
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const float2 q = f[along(r)];
            ph[r] = COL ? cmul(q, l) : cmul(l, q);               // phy * phx
        }
    }
    if constexpr (KIND == PROBE) {
        // this workgroup's 2N / G factors (double-precision phase, Func_generate_probe_wave_scan_sub_pixel.m)
        constexpr int PER = 2 * N / G;
        if (threadIdx.x < PER) {
            const int i = blockIdx.x * PER + threadIdx.x, k = i % N;
            const double d = (double)(i < N ? A.x : A.y)[0] - (double)A.cent;
            const double g = (double)((k + N / 2) % N) - (double)(N / 2);
            double sn, cs;
            sincos(-2.0 * M_PI * d * g / (double)N, &sn, &cs);
            A.phi[i] = make_float2((float)cs, (float)sn);
        }
    }
    // transmission of the plane (STEP02_FORWARD_4D.m:18-19 rounding order), formed where it is applied so
    // that the wait for the slices falls behind the first transforms, and kept for the adjoint pass (which runs along
    // the other axis)
    auto transmission = [&]() {
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
#pragma unroll
            for (int r = 0; r < E; ++r) sum[r] += z[i][r];
        }
        for (int i = KEEP; i < nzp; ++i) {
            const BufF V = slice(i);
#pragma unroll
            for (int r = 0; r < E; ++r) sum[r] += V[vox(r)];
        }
#pragma unroll
        for (int r = 0; r < E; ++r) {
            float sn, cs;
            sincosf(A.sigma * (sum[r] * A.dx), &sn, &cs);
            t[r] = make_float2(cs, sn);
            trans.put(own(r), t[r]);
        }
    };

    auto half = [&](bool conj) {
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = cscale(conj ? cmulc(v[r], pf[r]) : cmul(v[r], pf[r]), inv_n);
    };

    // ---- the pass
    if constexpr (KIND == PROBE) {
        F.template dft<false>(v);
    } else if constexpr (KIND == SHIFT || KIND == BACK) {
        F.template dft<false>(v);
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = KIND == SHIFT ? cmul(v[r], ph[r]) : cmulc(v[r], ph[r]);
        F.template dft<true>(v);
    } else if constexpr (KIND == FIRST || KIND == FWD || KIND == LAST) {
        if constexpr (KIND != FIRST) {
            F.template dft<false>(v);
            half(false);
        }
        F.template dft<true>(v);
#pragma unroll
        for (int r = 0; r < E; ++r) {
            if constexpr (KIND == FIRST) v[r] = cscale(v[r], inv_n2);
            wave.put(own(r), v[r]);
        }
        if constexpr (KIND != LAST) {
            transmission();
#pragma unroll
            for (int r = 0; r < E; ++r) v[r] = cmul(v[r], t[r]);
        }
        F.template dft<false>(v);
        if constexpr (KIND != LAST) {
            half(false);
            F.template dft<true>(v);
        }
    } else if constexpr (KIND == EXIT) {
        F.template dft<false>(v);
        // intensity, loss, residual (STEP02_FORWARD_4D.m:36-49) times conj(p)
        const float2 pl = A.p1d[(COL ? 0 : N) + line];
        double err = 0.0;
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const float I = v[r].x * v[r].x + v[r].y * v[r].y;
            const float d = m[r] - __builtin_amdgcn_sqrtf(I);
            err += (double)(d * d);
            const float f = 1.0f - m[r] * __builtin_amdgcn_rsqf(I + 1e-30f);
            v[r] = cmulc(make_float2(v[r].x * f, v[r].y * f), COL ? cmul(pl, pf[r]) : cmul(pf[r], pl));
        }
        err = group_sum<N>(err, red);
        if (threadIdx.x == 0) A.part[blockIdx.x] = err;
        F.template dft<true>(v);
    } else if constexpr (KIND == ADJ) {
        if (A.head) {
            F.template dft<true>(v);
#pragma unroll
            for (int r = 0; r < E; ++r) v[r] = cscale(v[r], inv_n2);
        } else {
            F.template dft<false>(v);
            half(true);
            F.template dft<true>(v);
        }
        // gradient (STEP03_BACK.m:12-24), the object step of every slice of the bin (:84), x conj(t)
        float g[E];
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const float2 tc = cconj(t[r]);
            g[r] = -cmul(tc, cmulc(v[r], wv[r])).y;                  // Re(1i * conj(t) * conj(psi) * b)
            v[r] = cmul(v[r], tc);
        }
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
            const BufF V = slice(i);
#pragma unroll
            for (int r = 0; r < E; ++r) V.put(vox(r), z[i][r] + A.s1 * g[r]);
        }
        for (int i = KEEP; i < nzp; ++i) {
            const BufF V = slice(i);
#pragma unroll
            for (int r = 0; r < E; ++r) V.put(vox(r), V[vox(r)] + A.s1 * g[r]);
        }
        if constexpr (COL) {
            if (A.a == 0 && A.want_pos) {
                // position terms (STEP03_BACK.m:35-38): MATLAB gradient() of conj(psi0), psi0 is [y][x]
                double dr = 0.0, dc = 0.0;
#pragma unroll
                for (int r = 0; r < E; ++r) {
                    const int y = j + r * T, x = line;
                    const int xp = min(x + 1, N - 1), xm = max(x - 1, 0), yp = min(y + 1, N - 1), ym = max(y - 1, 0);
                    const float2 gx = cscale(csub(A.psi0[y * N + xp], A.psi0[y * N + xm]), xp - xm == 2 ? 0.5f : 1.0f);
                    const float2 gy = cscale(csub(A.psi0[yp * N + x], A.psi0[ym * N + x]), yp - ym == 2 ? 0.5f : 1.0f);
                    dr += (double)(gx.x * v[r].x + gx.y * v[r].y);
                    dc += (double)(gy.x * v[r].x + gy.y * v[r].y);
                }
                dr = group_sum<N>(dr, red);
                dc = group_sum<N>(dc, red);
                if (threadIdx.x == 0) {
                    A.part[G + blockIdx.x] = dr;
                    A.part[2 * G + blockIdx.x] = dc;
                }
            }
            if (A.a == 0 && blockIdx.x == 0 && threadIdx.x == 0) {
                // the loss: the exit pass's workgroup sums in workgroup order
                double e = 0.0;
                for (int i = 0; i < G; ++i) e += A.part[i];
                A.err[0] = e;
            }
        }
        F.template dft<false>(v);
        if (A.a > 0) {
            half(true);
            F.template dft<true>(v);
        }
    } else if constexpr (KIND == STEP) {
        // position += s3 d (Run_MSET_recon.m:155-157), the workgroup sums in workgroup order
        if (A.want_pos && blockIdx.x == 0 && threadIdx.x == 0) {
            double dr = 0.0, dc = 0.0;
            for (int i = 0; i < G; ++i) {
                dr += A.part[G + i];
                dc += A.part[2 * G + i];
            }
            A.x[0] = (float)((double)A.x[0] + (double)A.s3 * dr);
            A.y[0] = (float)((double)A.y[0] + (double)A.s3 * dc);
        }
        if (A.s2 == 0.f) return;
        F.template dft<true>(v);
#pragma unroll
        for (int r = 0; r < E; ++r) probe.put(vox(r), csub(pr[r], cscale(cscale(v[r], inv_n2), A.s2)));
        return;
    }
    // transposed: the next pass runs along the other axis
#pragma unroll
    for (int r = 0; r < E; ++r) out.put(oth(r), v[r]);
}

template <int N> hipError_t position_lines(const PosArgs& P, int k, float2* work, hipStream_t st) {
    constexpr int N2 = N * N;
    const int L = P.L;
    float2 *a = work, *b = work + N2, *trans = work + position_lines_work(N, 0);
    LineArgs A{};
    A.tw = P.tw;
    A.p1d = P.p1d;
    A.phi = work + 2 * N2;
    A.part = (double*)(work + 2 * N2 + 2 * N);
    A.V = P.V;
    A.nz = P.nz;
    A.bin = P.bin;
    A.sigma = P.sigma;
    A.dx = P.dx;
    A.cent = P.cent;
    A.s1 = P.s1;
    A.s2 = P.s2;
    A.s3 = P.s3;
    A.want_pos = (P.want & WANT_POS) != 0;
    A.x = P.xlist + k;
    A.y = P.ylist + k;
    A.sqrtM = P.sqrtM + (size_t)k * N2;
    A.probe = P.probe;
    A.psi0 = P.save;
    A.err = P.err_pos + k;
#define MSET_LINE(KIND, COL) hipLaunchKernelGGL((k_line_pass<N, KIND, COL>), dim3(N / TL), dim3(N), 0, st, A)
#define MSET_LINE2(KIND, COL)              \
    do {                                   \
        if (COL) MSET_LINE(KIND, true);    \
        else MSET_LINE(KIND, false);       \
    } while (0)
    // each pass reads `a` (the probe first) and writes `b`
    auto next = [&]() {
        float2* o = a;
        a = b;
        b = o;
        A.in = a;
        A.out = b;
    };
    A.in = P.probe;
    A.out = b;
    MSET_LINE(PROBE, false);
    next();
    MSET_LINE(SHIFT, true);
    next();
    A.wave = P.save;
    A.trans = trans;
    MSET_LINE(FIRST, false);
    for (int i = 1; i < L; ++i) {
        next();
        A.a = i;
        A.wave = P.save + (size_t)i * N2;
        A.trans = trans + (size_t)i * N2;
        MSET_LINE2(FWD, i % 2 == 1);
    }
    next();
    A.wave = P.save + (size_t)L * N2;
    MSET_LINE2(LAST, L % 2 == 1);
    next();
    MSET_LINE2(EXIT, L % 2 == 0);
    for (int i = L - 1; i >= 0; --i) {
        next();
        A.a = i;
        A.head = i == L - 1;
        A.trans = trans + (size_t)i * N2;
        A.wave = P.save + (size_t)(i + 1) * N2;                 // reference pairing: the wave after plane i
        MSET_LINE2(ADJ, i % 2 == 0);
    }
    if (P.s2 != 0.f) {
        next();
        MSET_LINE(BACK, false);
    }
    if (P.s2 != 0.f || A.want_pos) {
        next();
        MSET_LINE(STEP, true);
    }
#undef MSET_LINE
#undef MSET_LINE2
    return hipGetLastError();
}

}  // namespace

bool position_lines_supported(int n) { return n == 96 || n == 128 || n == 256; }

// two plane buffers, the shift factors, three sums per workgroup, the transmission planes
size_t position_lines_work(int n, int L) { return (2 + (size_t)L) * n * n + 2 * (size_t)n + 3 * (size_t)(n / TL); }

hipError_t launch_position_lines(int n, const PosArgs& P, int k, float2* work, hipStream_t st) {
    switch (n) {
        case 96: return position_lines<96>(P, k, work, st);
        case 128: return position_lines<128>(P, k, work, st);
        case 256: return position_lines<256>(P, k, work, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mset
