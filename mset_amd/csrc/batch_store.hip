// batch_store.hip -- launcher of the batched gradient (k_batch, multislice.hpp) with stored exit waves in
// every shape and routine, and its occupancy query; the recomputed and checkpointed variants are launched
// from batch_variants.hip.
#include "multislice.hpp"

namespace mset {

namespace {
// Cfg of the alternative shape; at 16 the default workgroup of one wave is the faster one with every routine
template <int N> constexpr int ALT = N == 16 ? 0 : 1;
// whether it applies a separable propagator as its 1D factors: at 32 they cost a workgroup per CU (1400 positions x 12
// planes 234 us with them, 188 without)
template <int N> constexpr bool ALT_PFAC = N != 32;
}  // namespace

hipError_t launch_batch_variant(int n, const PosArgs& A, int grid, int shape, hipStream_t st);

hipError_t launch_batch(int n, const PosArgs& A, int grid, int shape, hipStream_t st) {
    // shape 1: stored waves; shape 2: stored waves at 48, or the separable 256 routine with stored or
    // checkpointed waves; shape 4: at 24
    if (shape == 1 && A.waves != WAVES_STORE) return hipErrorInvalidValue;
    if (shape == 2 && !(n == 256 && A.sep) && !(n == 48 && A.waves == WAVES_STORE)) return hipErrorInvalidValue;
    if (shape < 0 || shape == 3 || shape > 4 || (shape == 4 && n != 24)) return hipErrorInvalidValue;
    if (A.waves != WAVES_STORE) return launch_batch_variant(n, A, grid, shape, st);
    if (A.sep) {
        if (n != 256 || A.grad_mode != GRAD_REF || A.sset) return hipErrorInvalidValue;
        if (shape == 2) hipLaunchKernelGGL((k_batch<256, 2, WAVES_STORE, true>), dim3(grid), dim3(Cfg<256, 2>::NT), 0, st, A);
        else if (shape) hipLaunchKernelGGL((k_batch<256, 1, WAVES_STORE, true>), dim3(grid), dim3(Cfg<256, 1>::NT), 0, st, A);
        else hipLaunchKernelGGL((k_batch<256, 0, WAVES_STORE, true>), dim3(grid), dim3(Cfg<256>::NT), 0, st, A);
    } else if (shape == 2) {
        if (A.pfac && !A.sset) hipLaunchKernelGGL((k_batch<48, 2, WAVES_STORE, false, true>), dim3(grid), dim3(Cfg<48, 2>::NT), 0, st, A);
        else hipLaunchKernelGGL((k_batch<48, 2, WAVES_STORE, false>), dim3(grid), dim3(Cfg<48, 2>::NT), 0, st, A);
    } else if (shape == 4) {
        if (A.pfac && !A.sset) hipLaunchKernelGGL((k_batch<24, 4, WAVES_STORE, false, true>), dim3(grid), dim3(Cfg<24, 4>::NT), 0, st, A);
        else hipLaunchKernelGGL((k_batch<24, 4, WAVES_STORE, false>), dim3(grid), dim3(Cfg<24, 4>::NT), 0, st, A);
    } else if (shape && A.pfac && n < 128 && !A.sset) {
        MSET_DISPATCH_SMALL(n, hipLaunchKernelGGL((k_batch<NN, ALT<NN>, WAVES_STORE, false, ALT_PFAC<NN>>), dim3(grid), dim3(Cfg<NN, ALT<NN>>::NT), 0, st, A))
    } else if (shape) {
        MSET_DISPATCH(n, hipLaunchKernelGGL((k_batch<NN, ALT<NN>, WAVES_STORE, false>), dim3(grid), dim3(Cfg<NN, ALT<NN>>::NT), 0, st, A))
    } else if (A.pfac && n != 256 && !A.sset) {
        MSET_DISPATCH_SMALL(n, hipLaunchKernelGGL((k_batch<NN, 0, WAVES_STORE, false, true>), dim3(grid), dim3(Cfg<NN>::NT), 0, st, A))
    } else MSET_DISPATCH(n, hipLaunchKernelGGL((k_batch<NN, 0, WAVES_STORE, false>), dim3(grid), dim3(Cfg<NN>::NT), 0, st, A));
    return hipGetLastError();
}

hipError_t occupancy_batch(int n, int shape, int* blocks_per_cu) {
    if (shape == 4 && n == 24)
        return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, (k_batch<24, 4, WAVES_STORE, false>), Cfg<24, 4>::NT, 0);
    if (shape)
        MSET_DISPATCH(n, return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, (k_batch<NN, ALT<NN>, WAVES_STORE, false>), Cfg<NN, ALT<NN>>::NT, 0));
    MSET_DISPATCH(n, return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, (k_batch<NN, 0, WAVES_STORE, false>), Cfg<NN>::NT, 0));
    return hipSuccess;
}

}  // namespace mset
