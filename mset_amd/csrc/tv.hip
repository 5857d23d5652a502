// tv.hip -- the total-variation regulariser on the device (TV_method.m:5-84, 3D).
//
// Chambolle's projection for min_u 1/2 |u - f|^2 + lambda TV(u) with periodic forward differences:
//   D = TV_div(P) - f / lambda
//   P = TV_project(P + tau TV_del(D)), tau = 1/12
// repeated n_iter times from P = 0, then u = f - lambda TV_div(P) and the error lambda sum |TV_del(u)|.
// An iteration is one launch from one dual field to another (k_tv_iterate), on 7 volumes of scratch, or two launches in
// place on 4 where 7 do not fit the device (k_tv_dual_residual, k_tv_project).
// The dual field P is three float volumes (structure of arrays, so every stencil read is coalesced);
// the operation order of each element follows TV_method.m so that single-precision results match a
// MATLAB single run to rounding.  Volumes are [z][y][x] with MATLAB dims (x, y, z) = (1, 2, 3):
// circshift(A, [1 0 0]) is A(x - 1) and circshift(A, [-1 0 0]) is A(x + 1), periodic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "kernels.hpp"

namespace mset {

namespace {

struct Grid3 {
    int nx, ny, nz;
    __device__ __forceinline__ void coords(long long i, int& x, int& y, int& z) const {
        x = (int)(i % nx);
        const long long r = i / nx;
        y = (int)(r % ny);
        z = (int)(r / ny);
    }
    __device__ __forceinline__ long long at(int x, int y, int z) const { return ((long long)z * ny + y) * nx + x; }
};

// TV_div: P1 + P2 + P3 - P1(x-1) - P2(y-1) - P3(z-1)
__device__ __forceinline__ float tv_div(const Grid3& g, const float* P0, const float* P1, const float* P2, int x, int y,
                                        int z) {
    const long long i = g.at(x, y, z);
    float d = P0[i] + P1[i] + P2[i];
    d = d - P0[g.at(x == 0 ? g.nx - 1 : x - 1, y, z)];
    d = d - P1[g.at(x, y == 0 ? g.ny - 1 : y - 1, z)];
    d = d - P2[g.at(x, y, z == 0 ? g.nz - 1 : z - 1)];
    return d;
}

// q = f / lambda
__global__ void k_tv_scale(const float* __restrict__ f, long long nv, float lambda, float* __restrict__ q) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < nv; i += (long long)gridDim.x * blockDim.x)
        q[i] = f[i] / lambda;
}

// W consecutive elements of a row
template <int W> struct Row {
    float a[W];
};

// One volume: a buffer view with 32-bit offsets (I = unsigned), or a pointer for volumes beyond its reach
template <int W, class I> struct Volume {
    float* p;
    __device__ __forceinline__ Volume(const float* q, size_t) : p(const_cast<float*>(q)) {}
    __device__ __forceinline__ float one(I i) const { return p[i]; }
    __device__ __forceinline__ Row<W> row(I i) const {
        Row<W> r;
        if constexpr (W == 4) {
            const float4 t = *reinterpret_cast<const float4*>(p + i);
            r.a[0] = t.x; r.a[1] = t.y; r.a[2] = t.z; r.a[3] = t.w;
        } else {
            r.a[0] = p[i];
        }
        return r;
    }
    __device__ __forceinline__ void put(I i, const Row<W>& r) const {
        if constexpr (W == 4) *reinterpret_cast<float4*>(p + i) = make_float4(r.a[0], r.a[1], r.a[2], r.a[3]);
        else p[i] = r.a[0];
    }
};
template <int W> struct Volume<W, unsigned> {
    typedef unsigned u32x4 __attribute__((__vector_size__(16)));
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ Volume(const float* q, size_t n)
        : r(__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(q), (short)0, (int)(unsigned)(n * 4), 0x00020000)) {}
    __device__ __forceinline__ float one(unsigned i) const {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, i * 4u, 0, 0));
    }
    __device__ __forceinline__ Row<W> row(unsigned i) const {
        if constexpr (W == 4) return __builtin_bit_cast(Row<4>, __builtin_amdgcn_raw_buffer_load_b128(r, i * 4u, 0, 0));
        else return Row<1>{one(i)};
    }
    __device__ __forceinline__ void put(unsigned i, const Row<W>& v) const {
        if constexpr (W == 4) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, i * 4u, 0, 0);
        else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v.a[0]), r, i * 4u, 0, 0);
    }
};

// One iteration, W elements of a row per thread (4 where rows are whole float4s): the residual D of the elements
// and of their x, y and z successors is formed from P (25 loads for 4 elements, all but 7 of them hits in
// L1 or L2, requested together), so D is never stored and P, q are read once and P written once: 28 bytes of
// memory traffic per element instead of 48 in two launches with a stored D.  q = f / lambda is formed once.  The
// fields alternate between Pi and Po.  A neighbour is the element's index plus a step that wraps at the volume's
// faces, in 32 bits (I) unless the volume needs more: index arithmetic in 64 bits took a third of the kernel's
// instructions.  64 x 128 x 128 volume, per iteration: 13.8 us as two launches, 8.3 us with pointers, 7.8 us with
// views.
template <int W, class I>
__global__ __launch_bounds__(256) void k_tv_iterate(int nx, int ny, int nz, const float* __restrict__ Pi,
                                                    const float* __restrict__ q_, float* __restrict__ Po, I items) {
    const float tau = 1.0f / 12.0f;
    const size_t nv = (size_t)nx * ny * nz;
    using Vol = Volume<W, I>;
    using V = Row<W>;
    const Vol P0(Pi, nv), P1(Pi + nv, nv), P2(Pi + 2 * nv, nv), q(q_, nv);
    const Vol O0(Po, nv), O1(Po + nv, nv), O2(Po + 2 * nv, nv);
    const unsigned rows = (unsigned)nx / W;
    const I row = (I)nx, plane = (I)nx * (I)ny, depth = plane * (I)nz;
    // Workgroups go to the 8 XCDs round-robin: renumbered so that each XCD works on one contiguous part of the
    // volume and finds the neighbouring rows and planes in its own L2
    const unsigned g = gridDim.x, b = g % 8 == 0 ? blockIdx.x % 8 * (g / 8) + blockIdx.x / 8 : blockIdx.x;
    for (I i = (I)b * blockDim.x + threadIdx.x; i < items; i += (I)g * blockDim.x) {
        const I e = i * W, yz = i / rows, z = yz / (unsigned)ny;
        const unsigned x = (unsigned)(i - yz * rows) * W, y = (unsigned)(yz - z * (unsigned)ny);
        // neighbours, periodic (unsigned differences wrap around to the right index)
        const I xp = (x + W == (unsigned)nx ? (I)W - row : (I)W), xm = x == 0 ? row - 1 : (I)0 - 1;
        const I yp = y + 1 == (unsigned)ny ? row - plane : row, ym = y == 0 ? plane - row : (I)0 - row;
        const I zp = z + 1 == (I)nz ? plane - depth : plane, zm = z == 0 ? depth - plane : (I)0 - plane;
        const V a = P0.row(e), b_ = P1.row(e), c = P2.row(e);
        const V bym = P1.row(e + ym), czm = P2.row(e + zm), f = q.row(e);
        const float am = P0.one(e + xm);
        // x successor of the last element
        const float ax = P0.one(e + xp), bx = P1.one(e + xp), cx = P2.one(e + xp), bxym = P1.one(e + xp + ym);
        const float cxzm = P2.one(e + xp + zm), fx = q.one(e + xp);
        // y successors
        const V ay = P0.row(e + yp), by = P1.row(e + yp), cy = P2.row(e + yp), cyzm = P2.row(e + yp + zm), fy = q.row(e + yp);
        const float aym = P0.one(e + yp + xm);
        // z successors
        const V az = P0.row(e + zp), bz = P1.row(e + zp), cz = P2.row(e + zp), bzym = P1.row(e + zp + ym), fz = q.row(e + zp);
        const float azm = P0.one(e + zp + xm);
        // TV_div in its operation order, then - f / lambda
        auto res = [](float p0, float p1, float p2, float p0m, float p1m, float p2m, float g) {
            float d = p0 + p1 + p2;
            d = d - p0m;
            d = d - p1m;
            d = d - p2m;
            return d - g;
        };
        float d[W + 1];
#pragma unroll
        for (int k = 0; k < W; ++k) d[k] = res(a.a[k], b_.a[k], c.a[k], k ? a.a[k - 1] : am, bym.a[k], czm.a[k], f.a[k]);
        d[W] = res(ax, bx, cx, a.a[W - 1], bxym, cxzm, fx);
        V o0, o1, o2;
#pragma unroll
        for (int k = 0; k < W; ++k) {
            const float dy = res(ay.a[k], by.a[k], cy.a[k], k ? ay.a[k - 1] : aym, b_.a[k], cyzm.a[k], fy.a[k]);
            const float dz = res(az.a[k], bz.a[k], cz.a[k], k ? az.a[k - 1] : azm, bzym.a[k], c.a[k], fz.a[k]);
            const float q0 = a.a[k] + tau * (d[k + 1] - d[k]);
            const float q1 = b_.a[k] + tau * (dy - d[k]);
            const float q2 = c.a[k] + tau * (dz - d[k]);
            // den = sqrt(max(1, |q|^2)) and the three quotients with it, each the hardware's estimate corrected by
            // its remainder (Markstein, IBM J. Res. Dev. 34 (1990) 111): the arguments are normal and near 1, so the
            // scaling of a general division or square root is not needed, and the quotients share one reciprocal
            const float m = fmaxf(1.0f, q0 * q0 + q1 * q1 + q2 * q2);
            // beyond the float range (m infinite): r = 0, so finite q give 0 as their division by infinity does
            const bool finite = m <= 3.402823466e38f;
            const float mf = finite ? m : 1.0f;
            const float rs = __builtin_amdgcn_rsqf(mf);
            float den = mf * rs;
            den = __builtin_fmaf(__builtin_fmaf(-den, den, mf), 0.5f * rs, den);
            const float r = finite ? __builtin_fmaf(__builtin_fmaf(-den, rs, 1.0f), rs, rs) : 0.0f;
            auto quot = [&](float a) {
                const float t = a * r;
                return __builtin_fmaf(__builtin_fmaf(-den, t, a), r, t);
            };
            o0.a[k] = quot(q0);
            o1.a[k] = quot(q1);
            o2.a[k] = quot(q2);
        }
        O0.put(e, o0);
        O1.put(e, o1);
        O2.put(e, o2);
    }
}

// The same iteration in two launches, in place with the residual D stored: 4 volumes of scratch
__global__ void k_tv_dual_residual(Grid3 g, const float* __restrict__ P0, const float* __restrict__ P1,
                                   const float* __restrict__ P2, const float* __restrict__ f, float lambda,
                                   float* __restrict__ D) {
    const long long nv = (long long)g.nx * g.ny * g.nz;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < nv; i += (long long)gridDim.x * blockDim.x) {
        int x, y, z;
        g.coords(i, x, y, z);
        D[i] = tv_div(g, P0, P1, P2, x, y, z) - f[i] / lambda;
    }
}

__global__ void k_tv_project(Grid3 g, float* __restrict__ P0, float* __restrict__ P1, float* __restrict__ P2,
                             const float* __restrict__ D) {
    const float tau = 1.0f / 12.0f;
    const long long nv = (long long)g.nx * g.ny * g.nz;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < nv; i += (long long)gridDim.x * blockDim.x) {
        int x, y, z;
        g.coords(i, x, y, z);
        const float d = D[i];
        const float q0 = P0[i] + tau * (D[g.at(x + 1 == g.nx ? 0 : x + 1, y, z)] - d);
        const float q1 = P1[i] + tau * (D[g.at(x, y + 1 == g.ny ? 0 : y + 1, z)] - d);
        const float q2 = P2[i] + tau * (D[g.at(x, y, z + 1 == g.nz ? 0 : z + 1)] - d);
        const float den = sqrtf(fmaxf(1.0f, q0 * q0 + q1 * q1 + q2 * q2));
        P0[i] = q0 / den;
        P1[i] = q1 / den;
        P2[i] = q2 / den;
    }
}

__global__ void k_tv_output(Grid3 g, const float* __restrict__ P0, const float* __restrict__ P1,
                            const float* __restrict__ P2, const float* f, float lambda, float* u) {
    const long long nv = (long long)g.nx * g.ny * g.nz;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < nv; i += (long long)gridDim.x * blockDim.x) {
        int x, y, z;
        g.coords(i, x, y, z);
        u[i] = f[i] - lambda * tv_div(g, P0, P1, P2, x, y, z);   // f and u may alias (same element)
    }
}

constexpr int RED_THREADS = 256;

// per-block partial sums (double) of |TV_del(u)|, summed on the host in block order
__global__ void k_tv_error(Grid3 g, const float* __restrict__ u, double* __restrict__ part) {
    __shared__ double red[RED_THREADS];
    const long long nv = (long long)g.nx * g.ny * g.nz;
    double s = 0.0;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < nv; i += (long long)gridDim.x * blockDim.x) {
        int x, y, z;
        g.coords(i, x, y, z);
        const double c = u[i];
        const double d0 = (double)u[g.at(x + 1 == g.nx ? 0 : x + 1, y, z)] - c;
        const double d1 = (double)u[g.at(x, y + 1 == g.ny ? 0 : y + 1, z)] - c;
        const double d2 = (double)u[g.at(x, y, z + 1 == g.nz ? 0 : z + 1)] - c;
        s += sqrt(d0 * d0 + d1 * d1 + d2 * d2);
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = RED_THREADS / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// per-block maxima of a volume
__global__ void k_max(const float* __restrict__ v, long long n, float* __restrict__ part) {
    __shared__ float red[RED_THREADS];
    float m = -INFINITY;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        m = fmaxf(m, v[i]);
    red[threadIdx.x] = m;
    __syncthreads();
    for (int o = RED_THREADS / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// v = v / s (mode 0) or v = s * v (mode 1): the normalisation around TV (Run_MSET_recon.m:267-269)
__global__ void k_scale(float* __restrict__ v, long long n, float s, int mode) {
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        v[i] = mode == 0 ? v[i] / s : s * v[i];
}

constexpr int RED_BLOCKS = 512;

dim3 grid_of(long long n) {
    const long long b = (n + RED_THREADS - 1) / RED_THREADS;
    return dim3((unsigned)std::max(1LL, std::min(b, 8192LL)));
}

}  // namespace

int tv_ensure(TvWork& w, long long nv) {
    if (w.P && w.n >= 7 * (size_t)nv) return 0;
    tv_release(w);
    if (hipMalloc((void**)&w.part, sizeof(double) * RED_BLOCKS) != hipSuccess) {
        w.part = nullptr;
        return -1;
    }
    for (const size_t volumes : {7, 4}) {
        if (hipMalloc((void**)&w.P, sizeof(float) * volumes * (size_t)nv) == hipSuccess) {
            w.n = volumes * (size_t)nv;
            return 0;
        }
        (void)hipGetLastError();                         // not the next launch's error
        w.P = nullptr;
    }
    return -1;
}

void tv_release(TvWork& w) {
    if (w.P) (void)hipFree(w.P);
    if (w.part) (void)hipFree(w.part);
    w.P = nullptr;
    w.part = nullptr;
    w.n = 0;
}

hipError_t tv_run(TvWork& w, const float* f, float* u, int nx, int ny, int nz, float lambda, int n_iter, double* err,
                  hipStream_t st) {
    const Grid3 g{nx, ny, nz};
    const long long nv = (long long)nx * ny * nz;
    float* P = w.P;
    const dim3 gr = grid_of(nv), bl(RED_THREADS);
    hipError_t e = launch_fill(P, sizeof(float) * 3 * (size_t)nv, st);   // P = 0
    if (e != hipSuccess) return e;
    if (w.n < 7 * (size_t)nv) {
        float* D = w.P + 3 * nv;
        for (int it = 0; it < n_iter; ++it) {
            hipLaunchKernelGGL(k_tv_dual_residual, gr, bl, 0, st, g, P, P + nv, P + 2 * nv, f, lambda, D);
            hipLaunchKernelGGL(k_tv_project, gr, bl, 0, st, g, P, P + nv, P + 2 * nv, D);
        }
    } else {
        // two dual fields and f / lambda
        float *Q = w.P + 3 * nv, *q = w.P + 6 * nv;
        hipLaunchKernelGGL(k_tv_scale, gr, bl, 0, st, f, nv, lambda, q);
        const bool wide = nx % 4 == 0;                   // rows of whole float4s
        const long long items = wide ? nv / 4 : nv;
        const bool narrow_index = nv < (1LL << 30);      // 32-bit byte offsets
        using U64 = unsigned long long;
        for (int it = 0; it < n_iter; ++it) {
            const dim3 gi = grid_of(items);
            if (wide && narrow_index)
                hipLaunchKernelGGL((k_tv_iterate<4, unsigned>), gi, bl, 0, st, nx, ny, nz, P, q, Q, (unsigned)items);
            else if (wide)
                hipLaunchKernelGGL((k_tv_iterate<4, U64>), gi, bl, 0, st, nx, ny, nz, P, q, Q, (U64)items);
            else if (narrow_index)
                hipLaunchKernelGGL((k_tv_iterate<1, unsigned>), gi, bl, 0, st, nx, ny, nz, P, q, Q, (unsigned)items);
            else
                hipLaunchKernelGGL((k_tv_iterate<1, U64>), gi, bl, 0, st, nx, ny, nz, P, q, Q, (U64)items);
            std::swap(P, Q);
        }
    }
    const float *P0 = P, *P1 = P + nv, *P2 = P + 2 * nv;
    hipLaunchKernelGGL(k_tv_output, gr, bl, 0, st, g, P0, P1, P2, f, lambda, u);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (err) {
        hipLaunchKernelGGL(k_tv_error, dim3(RED_BLOCKS), bl, 0, st, g, u, w.part);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        std::vector<double> part(RED_BLOCKS);
        if ((e = hipMemcpyAsync(part.data(), w.part, sizeof(double) * RED_BLOCKS, hipMemcpyDeviceToHost, st)) != hipSuccess)
            return e;
        if ((e = hipStreamSynchronize(st)) != hipSuccess) return e;
        double s = 0.0;
        for (double p : part) s += p;
        *err = (double)lambda * s;
    }
    return hipSuccess;
}

hipError_t volume_max(TvWork& w, const float* v, long long n, float* out, hipStream_t st) {
    float* part = reinterpret_cast<float*>(w.part);      // RED_BLOCKS doubles hold RED_BLOCKS floats
    hipLaunchKernelGGL(k_max, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, st, v, n, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    std::vector<float> h(RED_BLOCKS);
    if ((e = hipMemcpyAsync(h.data(), part, sizeof(float) * RED_BLOCKS, hipMemcpyDeviceToHost, st)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(st)) != hipSuccess) return e;
    float m = -INFINITY;
    for (float x : h) m = std::max(m, x);
    *out = m;
    return hipSuccess;
}

hipError_t volume_scale(float* v, long long n, float s, int mode, hipStream_t st) {
    hipLaunchKernelGGL(k_scale, grid_of(n), dim3(RED_THREADS), 0, st, v, n, s, mode);
    return hipGetLastError();
}

}  // namespace mset
