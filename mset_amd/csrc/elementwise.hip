// elementwise.hip -- bandwidth-bound helper kernels: pattern ingest, transmission planes, slab
// reductions, updates and positivity.  All are grid-stride loops with 16-byte-or-wider coalesced
// accesses where the layout allows; launches are sized to the element count (>= 1024 workgroups when
// the data is large) so the 256 CUs / 8 XCDs are filled.
#include <hip/hip_runtime.h>
#include <type_traits>
#include "kernels.hpp"

namespace mset {

static inline dim3 grid_for(size_t n, int per_thread = 1) {
    size_t g = (n / per_thread + 255) / 256;
    if (g < 1) g = 1;
    if (g > 8192) g = 8192;
    return dim3((unsigned)g);
}

// sqrt(ifftshift(M)) of every pattern (src/CUDA/mset.cu:206-210 does this per position per visit;
// here it is done once at ingest), stored transposed for the row pass that reads it:
// out[k][x][y] = sqrt(M[k][(y + N/2) % N][(x + N/2) % N]).  transpose: each pattern is first transposed
// (STEM_data.diffraction_transpose, STEP00_INIT.m:58-73), i.e. M[k][x][y] is read instead.
__global__ void k_ingest(const float* __restrict__ M, float* __restrict__ out, int n, long long npos, int transpose) {
    const long long n2 = (long long)n * n, tot = n2 * npos;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < tot; i += (long long)gridDim.x * blockDim.x) {
        const long long k = i / n2;
        const int r = (int)(i - k * n2), x = r / n, y = r % n;
        const int ys = (y + n / 2) % n, xs = (x + n / 2) % n;
        out[i] = sqrtf(M[k * n2 + (transpose ? (long long)xs * n + ys : (long long)ys * n + xs)]);
    }
}

// Slices z0 .. z1 - 1 of a pixel, C of them loaded before the first is stored, summed in slice order; with UPD each takes
// the object step first: V[z] += s1 g, one rounding, as in the line passes
template <bool UPD, int C> __device__ __forceinline__ void slices(float* V, size_t n2, int& z, int z1, float s1, float g, float& s) {
    for (; z + C <= z1; z += C) {
        float v[C];
#pragma unroll
        for (int i = 0; i < C; ++i) v[i] = V[(z + i) * n2];
#pragma unroll
        for (int i = 0; i < C; ++i) {
            if (UPD) V[(z + i) * n2] = v[i] = fmaf(s1, g, v[i]);
            s += v[i];
        }
    }
}

// Planes of a volume (blockIdx.y: one workgroup per 256 pixels and bin or part of a bin, so an element costs no
// division; with 64-bit ones these kernels took 4.4 us on 24^3 voxels).
//
// t_a = exp(1i * sigma * (sum_{z in bin a} V) * dx)  (STEP02_FORWARD_4D.m:12-20); with UPD the volume first takes the
// object step, V[z] += s1 G[a] for the slices z of bin a (the per-bin gradient replicated, STEP03_BACK.m:17-21): a
// position's step and the next one's transmission, the volume read once.  Up to 8 slices of a bin are in flight: with a
// store after each load they were a chain of memory round trips, 10.0 -> 4.9 us for the single-slice operator (one bin)
// on 64^3 voxels, 19.5 -> 7.8 us on 256 x 256 x 64.
template <bool UPD>
__global__ __launch_bounds__(256) void k_trans(float* V, const float* __restrict__ G, float2* __restrict__ T, int n2, int nz,
                                               int bin, int L, float s1, int sset, float sigma, float dx) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= n2) return;
    for (int a = blockIdx.y; a < L; a += gridDim.y) {
        const int z1 = min(a * bin + bin, nz);
        int z = a * bin;
        const float g = UPD ? G[(size_t)a * n2 + p] : 0.f;
        float s = 0.f;
        slices<UPD, 8>(V + p, n2, z, z1, s1, g, s);
        slices<UPD, 4>(V + p, n2, z, z1, s1, g, s);
        slices<UPD, 2>(V + p, n2, z, z1, s1, g, s);
        slices<UPD, 1>(V + p, n2, z, z1, s1, g, s);
        // STEP02_FORWARD_4D.m:18-19 rounds sigma * (sum * dx); STEP02_FORWARD_4D_SSET.m:9 (sigma * sum) * dx
        const float ph = sset ? (sigma * s) * dx : sigma * (s * dx);
        float sn, cs;
        sincosf(ph, &sn, &cs);
        T[(size_t)a * n2 + p] = make_float2(cs, sn);
    }
}

// The object step alone, UPDATE_SLICES slices of a bin per thread: a deep bin (the single-slice operator has one of the
// whole depth) takes as many workgroups as its voxels ask for: 14.0 -> 3.6 us on 64^3 voxels, 19.6 -> 7.7 on
// 256 x 256 x 64 against a thread per pixel of a bin; a thread per voxel reads G for each slice and takes 6.1 and 11.0 us,
// 17.7 against 12.6 on 256 x 256 x 128 in bins of 4.
constexpr int UPDATE_SLICES = 4;
__global__ __launch_bounds__(256) void k_update_volume(float* V, const float* __restrict__ G, int n2, int nz, int bin, int parts,
                                                       int rows, float s1) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= n2) return;
    for (int r = blockIdx.y; r < rows; r += gridDim.y) {
        const int a = r / parts;
        int z = a * bin + (r - a * parts) * UPDATE_SLICES;
        const int z1 = min(min(z + UPDATE_SLICES, a * bin + bin), nz);
        const float g = G[(size_t)a * n2 + p];
        float s = 0.f;
        slices<true, 4>(V + p, n2, z, z1, s1, g, s);
        slices<true, 2>(V + p, n2, z, z1, s1, g, s);
        slices<true, 1>(V + p, n2, z, z1, s1, g, s);
    }
}

// Transmission phases for the separable-propagator kernels, which form t = exp(i pi r) where they apply it
// (half the bytes of a complex plane).  r is the f32 phase of k_trans, divided by pi and reduced to [-1, 1]
// in double: t differs from k_trans's sincosf by about 1e-7.  Plane a goes to Tf in the
// layout of the pass that applies it in the forward sweep (rows, [x][y], for even a; columns, [y][x], for
// odd a) and, if Tb is given, to Tb in the layout of its adjoint pass (the other one).
__global__ void k_trans_sep(const float* __restrict__ V, float* __restrict__ Tf, float* __restrict__ Tb, int n, int nz,
                            int bin, int L, float sigma, float dx) {
    const long long n2 = (long long)n * n, tot = n2 * L;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < tot; i += (long long)gridDim.x * blockDim.x) {
        const int a = (int)(i / n2), p = (int)(i - (long long)a * n2);
        const int y = p / n, x = p % n;
        const int z0 = a * bin, z1 = min(z0 + bin, nz);
        float s = 0.f;
        for (int z = z0; z < z1; ++z) s += V[(size_t)z * n2 + p];
        const float ph = sigma * (s * dx);                      // STEP02_FORWARD_4D.m:18-19 rounding order
        double r = (double)ph / M_PI;
        r -= 2.0 * rint(0.5 * r);                               // [-1, 1]
        const long long rowmaj = (long long)y * n + x, colmaj = (long long)x * n + y;
        Tf[(long long)a * n2 + ((a & 1) ? rowmaj : colmaj)] = (float)r;
        if (Tb) Tb[(long long)a * n2 + ((a & 1) ? colmaj : rowmaj)] = (float)r;
    }
}

// The separable kernels leave odd gradient planes transposed ([x][y]); swap them back to [y][x] in place.
__global__ void k_untranspose_odd(float* __restrict__ G, int n, int L) {
    const long long n2 = (long long)n * n, tot = n2 * (L / 2);
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < tot; i += (long long)gridDim.x * blockDim.x) {
        const int a = 2 * (int)(i / n2) + 1;
        const int p = (int)(i % n2), y = p / n, x = p % n;
        if (x < y) {
            float* P = G + (size_t)a * n2;
            const float u = P[(size_t)y * n + x], w = P[(size_t)x * n + y];
            P[(size_t)y * n + x] = w;
            P[(size_t)x * n + y] = u;
        }
    }
}

__global__ void k_fill(uint4* p, size_t n16) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n16; i += (size_t)gridDim.x * blockDim.x)
        p[i] = make_uint4(0, 0, 0, 0);
}
__global__ void k_fill_bytes(unsigned char* p, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0;
}

__device__ __forceinline__ void add_to(float& a, float b) { a += b; }
__device__ __forceinline__ void add_to(float4& a, const float4& b) {
    a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
}

// out[i] = sum_s slab[s][i].  Slabs are summed in slot order (s = 0, 1, ...), so the result is the same for every
// launch shape, and out may be slab 0 (an element is read and written by the same thread); U loads are in flight at
// a time.  Bound by memory where the sum is large (5.2 TB/s for 256 slabs of 2^18 floats); a small one is a chain of
// nslab / U memory latencies on few wavefronts, and takes one float per thread and U = 32.
template <class T, int U>
__global__ __launch_bounds__(256) void k_reduce(const T* slab, int nslab, size_t n, T* out) {
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        T a{};
        int s = 0;
        auto add = [&](auto count) {
            constexpr int C = decltype(count)::value;
            for (; s + C <= nslab; s += C) {
                T v[C];
#pragma unroll
                for (int u = 0; u < C; ++u) v[u] = slab[(size_t)(s + u) * n + i];
#pragma unroll
                for (int u = 0; u < C; ++u) add_to(a, v[u]);
            }
        };
        add(std::integral_constant<int, U>{});
        if constexpr (U > 8) add(std::integral_constant<int, 8>{});
        add(std::integral_constant<int, 1>{});
        out[i] = a;
    }
}

__global__ void k_update_positions(float* x, float* y, const float* __restrict__ d, int npos, float s3) {
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < npos; k += gridDim.x * blockDim.x) {
        x[k] = x[k] + s3 * d[2 * k];
        y[k] = y[k] + s3 * d[2 * k + 1];
    }
}

// rec(rec < 0) = 0  (Run_MSET_recon.m:183-185)
__global__ void k_positivity(float* V, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        V[i] = V[i] < 0.f ? 0.f : V[i];
}

hipError_t launch_ingest_patterns(const float* M, float* sqrtM, int n, long long npos, int transpose, hipStream_t st) {
    hipLaunchKernelGGL(k_ingest, grid_for((size_t)n * n * npos), dim3(256), 0, st, M, sqrtM, n, npos, transpose);
    return hipGetLastError();
}

namespace {
// 256 pixels by planes
dim3 volume_grid(int n2, int planes) { return dim3((unsigned)((n2 + 255) / 256), (unsigned)(planes < 65535 ? planes : 65535)); }
}  // namespace

hipError_t launch_transmission(const float* V, float2* T, int n, int nz, int bin, int sset, float sigma, float dx,
                               hipStream_t st) {
    const int L = (nz + bin - 1) / bin;
    hipLaunchKernelGGL((k_trans<false>), volume_grid(n * n, L), dim3(256), 0, st, const_cast<float*>(V), nullptr, T,
                       n * n, nz, bin, L, 0.f, sset, sigma, dx);
    return hipGetLastError();
}

hipError_t launch_transmission_sep(const float* V, float* Tf, float* Tb, int n, int nz, int bin, float sigma, float dx,
                                   hipStream_t st) {
    const int L = (nz + bin - 1) / bin;
    hipLaunchKernelGGL(k_trans_sep, grid_for((size_t)n * n * L), dim3(256), 0, st, V, Tf, Tb, n, nz, bin, L, sigma, dx);
    return hipGetLastError();
}

hipError_t launch_untranspose_odd(float* G, int n, int L, hipStream_t st) {
    if (L < 2) return hipSuccess;
    hipLaunchKernelGGL(k_untranspose_odd, grid_for((size_t)n * n * (L / 2)), dim3(256), 0, st, G, n, L);
    return hipGetLastError();
}

hipError_t launch_fill(void* p, size_t bytes, hipStream_t st) {
    if (((uintptr_t)p % 16) == 0 && bytes % 16 == 0)
        hipLaunchKernelGGL(k_fill, grid_for(bytes / 16), dim3(256), 0, st, (uint4*)p, bytes / 16);
    else
        hipLaunchKernelGGL(k_fill_bytes, grid_for(bytes), dim3(256), 0, st, (unsigned char*)p, bytes);
    return hipGetLastError();
}

hipError_t launch_reduce_slabs(const float* slab, int nslab, size_t n, float* out, hipStream_t st) {
    // float4 fills the chip from 2^16 floats on.  By 256 and 32 loads in flight: 2 x 96^2 floats in 200 slabs
    // 13.4 -> 6.6 us, 2 x 128^2 in 256 slabs 15.2 -> 7.2; 12 x 96^2 in 200 slabs 16.4 (float4) against 17.2.
    if (n > (size_t)1 << 16 && n % 4 == 0 && ((uintptr_t)slab % 16) == 0 && ((uintptr_t)out % 16) == 0)
        hipLaunchKernelGGL((k_reduce<float4, 8>), grid_for(n / 4), dim3(256), 0, st, (const float4*)slab, nslab, n / 4,
                           (float4*)out);
    else
        hipLaunchKernelGGL((k_reduce<float, 32>), grid_for(n), dim3(256), 0, st, slab, nslab, n, out);
    return hipGetLastError();
}

hipError_t launch_reduce_cslabs(const float2* slab, int nslab, size_t n, float2* out, hipStream_t st) {
    return launch_reduce_slabs((const float*)slab, nslab, 2 * n, (float*)out, st);
}

hipError_t launch_update_volume(float* V, const float* G, int n, int nz, int bin, float s1, hipStream_t st, float2* trans,
                                int sset, float sigma, float dx) {
    const int L = (nz + bin - 1) / bin;
    if (trans)
        hipLaunchKernelGGL((k_trans<true>), volume_grid(n * n, L), dim3(256), 0, st, V, G, trans, n * n, nz, bin, L, s1, sset,
                           sigma, dx);
    else {
        const int parts = (bin + UPDATE_SLICES - 1) / UPDATE_SLICES;
        hipLaunchKernelGGL(k_update_volume, volume_grid(n * n, L * parts), dim3(256), 0, st, V, G, n * n, nz, bin, parts, L * parts,
                           s1);
    }
    return hipGetLastError();
}

hipError_t launch_update_positions(float* x, float* y, const float* dpos, int npos, float s3, hipStream_t st) {
    hipLaunchKernelGGL(k_update_positions, grid_for((size_t)npos), dim3(256), 0, st, x, y, dpos, npos, s3);
    return hipGetLastError();
}

hipError_t launch_positivity(float* V, size_t n, hipStream_t st) {
    hipLaunchKernelGGL(k_positivity, grid_for(n), dim3(256), 0, st, V, n);
    return hipGetLastError();
}

}  // namespace mset
