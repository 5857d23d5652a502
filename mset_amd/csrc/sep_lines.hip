// sep_lines.hip -- launchers of the on-chip separable routine (sep_lines.hpp).
#include "sep_lines.hpp"

namespace mset {

#define MSET_SEP_CASES_64(...)                               \
    case 16: { constexpr int NN = 16; __VA_ARGS__; } break;  \
    case 24: { constexpr int NN = 24; __VA_ARGS__; } break;  \
    case 32: { constexpr int NN = 32; __VA_ARGS__; } break;  \
    case 48: { constexpr int NN = 48; __VA_ARGS__; } break;  \
    case 64: { constexpr int NN = 64; __VA_ARGS__; } break;

#define MSET_SEP_DISPATCH(N, ...)                               \
    switch (N) {                                                \
        MSET_SEP_CASES_64(__VA_ARGS__)                          \
        case 96: { constexpr int NN = 96; __VA_ARGS__; } break; \
        default: return hipErrorInvalidValue;                   \
    }

// sizes whose sequential path is a launch per position (from 96 on it is a chain of line passes)
#define MSET_SEP_DISPATCH_64(N, ...)          \
    switch (N) {                              \
        MSET_SEP_CASES_64(__VA_ARGS__)        \
        default: return hipErrorInvalidValue; \
    }

hipError_t launch_sep_batch(int n, const PosArgs& A, int grid, hipStream_t st) {
    if (!A.pfac || A.sset || A.grad_mode != GRAD_REF || A.waves != WAVES_STORE) return hipErrorInvalidValue;
    MSET_SEP_DISPATCH(n, hipLaunchKernelGGL((k_sep_batch<NN>), dim3(grid), dim3(SepCfg<NN>::NT), 0, st, A))
    return hipGetLastError();
}

hipError_t launch_sep_plain(int n, const PosArgs& A, int k, hipStream_t st) {
    if (!A.pfac || A.sset || A.grad_mode != GRAD_REF) return hipErrorInvalidValue;
    MSET_SEP_DISPATCH_64(n, hipLaunchKernelGGL((k_sep_plain<NN>), dim3(1), dim3(SepCfg<NN>::NT), 0, st, A, k))
    return hipGetLastError();
}

hipError_t launch_sep_fwd(int n, const PosArgs& A, int grid, bool tilts, hipStream_t st) {
    if (!A.pfac || A.sset) return hipErrorInvalidValue;
#define MSET_FWD(N)                                                                                             \
    if (tilts) hipLaunchKernelGGL((k_sep_fwd<N, true>), dim3(grid), dim3(SepCfg<N>::NT), 0, st, A);             \
    else hipLaunchKernelGGL((k_sep_fwd<N, false>), dim3(grid), dim3(SepCfg<N>::NT), 0, st, A)
    if (n == 128) {
        MSET_FWD(128);
    } else {
        MSET_SEP_DISPATCH(n, MSET_FWD(NN))
    }
#undef MSET_FWD
    return hipGetLastError();
}

hipError_t occupancy_sep(int n, bool fwd, int* per_cu) {
    if (fwd && n == 128) return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, (k_sep_fwd<128, false>), SepCfg<128>::NT, 0);
    if (fwd) MSET_SEP_DISPATCH(n, return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, (k_sep_fwd<NN, false>), SepCfg<NN>::NT, 0))
    MSET_SEP_DISPATCH(n, return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, (k_sep_batch<NN>), SepCfg<NN>::NT, 0))
    return hipSuccess;
}

}  // namespace mset
