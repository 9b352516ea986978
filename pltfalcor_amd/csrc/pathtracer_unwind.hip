// The split solve pass's exact unwind kernels (four and one HWSS wavelengths per beam): beam
// transport through the stored vertices and the per-path sums.
#include "pathtracer_split.hpp"

namespace plt {

int launch_solve_unwind(const PtScene& sc, const PtFrame& fr, const SolveBuffers& sb, hipStream_t st) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
        return set_error(PLT_EHIP, "solve_unwind_staged_kernel: device query failed");
    // as many regions per block as leave every CU a block: the larger the group that is sorted, the more
    // alike a wave's events (1280 x 720: 56 regions per block 0.40 ms, 28 the same, 14 0.54 ms)
    const uint32_t regions = (fr.n_paths + kPtBlock - 1) / kPtBlock;
    const uint32_t per = std::max(1u, std::min(uint32_t(kUnwindRegions), regions / uint32_t(cus)));
    const dim3 g((regions + per - 1) / per), b(kUnwindBlock);
    if (fr.hwss == 4) hipLaunchKernelGGL((solve_unwind_staged_kernel<4>), g, b, 0, st, sc, fr, sb, regions);
    else hipLaunchKernelGGL((solve_unwind_staged_kernel<1>), g, b, 0, st, sc, fr, sb, regions);
    return check_launch("solve_unwind_staged_kernel");
}

int launch_solve_walk_unwind(const PtScene& sc, const PtFrame& fr, const SolveBuffers& sb, hipStream_t st) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
        return set_error(PLT_EHIP, "solve_walk_unwind_kernel: device query failed");
    // a block per CU takes its share of the queue: larger shares sort better (1080p frame, walks' unwind
    // and sums: 0.61 ms, with two blocks per CU 0.73 ms, with four 0.91 ms)
    const dim3 g{uint32_t(cus)}, b(kUnwindBlock);
    if (fr.hwss == 4) hipLaunchKernelGGL((solve_walk_unwind_kernel<4>), g, b, 0, st, sc, fr, sb);
    else hipLaunchKernelGGL((solve_walk_unwind_kernel<1>), g, b, 0, st, sc, fr, sb);
    return check_launch("solve_walk_unwind_kernel");
}

int launch_solve_sum(const PtFrame& fr, const SolveBuffers& sb, hipStream_t st) {
    hipLaunchKernelGGL(solve_sum_kernel, dim3((fr.n_paths + kPtBlock - 1) / kPtBlock), dim3(kPtBlock), 0, st, fr, sb);
    return check_launch("solve_sum_kernel");
}

}  // namespace plt
