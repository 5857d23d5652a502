// forward.hip -- launchers of the forward-only kernels (k_fwd, multislice.hpp): one tilt's positions, or the
// positions of several tilts in one persistent launch.
#include "multislice.hpp"

namespace mset {

namespace {
// a separable propagator below 256 is applied as its 1D factors (the general routine's PFAC form)
bool fwd_pfac(int n, const PosArgs& A) { return A.pfac && n != 256 && !A.sset; }
}  // namespace

hipError_t launch_fwd(int n, const PosArgs& A, int grid, int shape, hipStream_t st) {
    if (shape != 0 && (shape != 2 || n != 48)) return hipErrorInvalidValue;
    if (A.sep) {
        if (n != 256 || A.sset) return hipErrorInvalidValue;
        hipLaunchKernelGGL((k_fwd<256, 0, false, true>), dim3(grid), dim3(Cfg<256>::NT), 0, st, A);
    } else if (shape == 2) {
        if (fwd_pfac(n, A)) hipLaunchKernelGGL((k_fwd<48, 2, false, false, true>), dim3(grid), dim3(Cfg<48, 2>::NT), 0, st, A);
        else hipLaunchKernelGGL((k_fwd<48, 2, false, false>), dim3(grid), dim3(Cfg<48, 2>::NT), 0, st, A);
    } else if (fwd_pfac(n, A)) {
        MSET_DISPATCH_SMALL(n, hipLaunchKernelGGL((k_fwd<NN, 0, false, false, true>), dim3(grid), dim3(Cfg<NN>::NT), 0, st, A))
    } else MSET_DISPATCH(n, hipLaunchKernelGGL((k_fwd<NN, 0, false, false>), dim3(grid), dim3(Cfg<NN>::NT), 0, st, A));
    return hipGetLastError();
}

hipError_t launch_fwd_tilts(int n, const PosArgs& A, int grid, int shape, hipStream_t st) {
    if (shape != 0 && (shape != 2 || n != 48)) return hipErrorInvalidValue;
    if (A.sep) {
        if (n != 256 || A.sset) return hipErrorInvalidValue;
        hipLaunchKernelGGL((k_fwd<256, 0, true, true>), dim3(grid), dim3(Cfg<256>::NT), 0, st, A);
    } else if (shape == 2) {
        if (fwd_pfac(n, A)) hipLaunchKernelGGL((k_fwd<48, 2, true, false, true>), dim3(grid), dim3(Cfg<48, 2>::NT), 0, st, A);
        else hipLaunchKernelGGL((k_fwd<48, 2, true, false>), dim3(grid), dim3(Cfg<48, 2>::NT), 0, st, A);
    } else if (fwd_pfac(n, A)) {
        MSET_DISPATCH_SMALL(n, hipLaunchKernelGGL((k_fwd<NN, 0, true, false, true>), dim3(grid), dim3(Cfg<NN>::NT), 0, st, A))
    } else MSET_DISPATCH(n, hipLaunchKernelGGL((k_fwd<NN, 0, true, false>), dim3(grid), dim3(Cfg<NN>::NT), 0, st, A));
    return hipGetLastError();
}

}  // namespace mset
