// forward.hip -- launchers of the forward-only kernels (k_fwd, multislice.hpp): one tilt's positions, or the
// positions of several tilts in one persistent launch.  Below 256 these are the launches that the on-chip separable
// routine (sep_lines.hip) does not take.
#include "multislice.hpp"

namespace mset {

hipError_t launch_fwd(int n, const PosArgs& A, int grid, int shape, hipStream_t st) {
    if (shape != 0 && !(shape == 2 && n == 48) && !(shape == 4 && n == 24)) return hipErrorInvalidValue;
    if (A.sep) {
        if (n != 256 || A.sset) return hipErrorInvalidValue;
        hipLaunchKernelGGL((k_fwd<256, 0, false, true>), dim3(grid), dim3(Cfg<256>::NT), 0, st, A);
    } else if (shape == 2) {
        hipLaunchKernelGGL((k_fwd<48, 2, false, false>), dim3(grid), dim3(Cfg<48, 2>::NT), 0, st, A);
    } else if (shape == 4) {
        hipLaunchKernelGGL((k_fwd<24, 4, false, false>), dim3(grid), dim3(Cfg<24, 4>::NT), 0, st, A);
    } else MSET_DISPATCH(n, hipLaunchKernelGGL((k_fwd<NN, 0, false, false>), dim3(grid), dim3(Cfg<NN>::NT), 0, st, A));
    return hipGetLastError();
}

hipError_t launch_fwd_tilts(int n, const PosArgs& A, int grid, int shape, hipStream_t st) {
    if (shape != 0 && !(shape == 2 && n == 48) && !(shape == 4 && n == 24)) return hipErrorInvalidValue;
    if (A.sep) {
        if (n != 256 || A.sset) return hipErrorInvalidValue;
        hipLaunchKernelGGL((k_fwd<256, 0, true, true>), dim3(grid), dim3(Cfg<256>::NT), 0, st, A);
    } else if (shape == 2) {
        hipLaunchKernelGGL((k_fwd<48, 2, true, false>), dim3(grid), dim3(Cfg<48, 2>::NT), 0, st, A);
    } else if (shape == 4) {
        hipLaunchKernelGGL((k_fwd<24, 4, true, false>), dim3(grid), dim3(Cfg<24, 4>::NT), 0, st, A);
    } else MSET_DISPATCH(n, hipLaunchKernelGGL((k_fwd<NN, 0, true, false>), dim3(grid), dim3(Cfg<NN>::NT), 0, st, A));
    return hipGetLastError();
}

}  // namespace mset
