// Chain-parallel scan on three bf16 pieces, fused attention form: launcher.
#include "ftc_tp_kernel.h"

namespace ftc {
namespace mfma {

void launch_scan_tp_norm(void *ws, const ScanArgs &args, hipStream_t stream) {
    const dim3 grid((unsigned)args.total_waves), block(512);
    if (args.tp_d <= 32)
        hipLaunchKernelGGL((scan_tp_kernel<1, 1, true>), grid, block, 0, stream, (uint32_t *)ws, args);
    else if (args.tp_d <= 64)
        hipLaunchKernelGGL((scan_tp_kernel<1, 2, true>), grid, block, 0, stream, (uint32_t *)ws, args);
    else
        hipLaunchKernelGGL((scan_tp_kernel<2, 2, true>), grid, block, 0, stream, (uint32_t *)ws, args);
}

}  // namespace mfma
}  // namespace ftc
