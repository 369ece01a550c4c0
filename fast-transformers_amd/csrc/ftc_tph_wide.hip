// Chain-parallel scan on the fp16 matrix path, states of 65 to 128 rows
// (ftc_tph_wide_kernel.h): launcher.
#include "ftc_tph_wide_kernel.h"

namespace ftc {
namespace mfma {

void launch_scan_tph_wide(void *ws, const ScanArgs &args, hipStream_t stream) {
    // (grid as for launch_scan_tp)
    const dim3 grid((unsigned)args.total_waves), block(768);
    if (args.tp_d <= 96)
        hipLaunchKernelGGL((scan_tph_wide_kernel<1>), grid, block, 0, stream, (uint32_t *)ws, args);
    else
        hipLaunchKernelGGL((scan_tph_wide_kernel<2>), grid, block, 0, stream, (uint32_t *)ws, args);
}

}  // namespace mfma
}  // namespace ftc
