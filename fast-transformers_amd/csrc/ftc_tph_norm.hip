// Chain-parallel scan on the fp16 matrix path, fused attention form: launcher.
#include "ftc_tph_kernel.h"

namespace ftc {
namespace mfma {

void launch_scan_tph_norm(void *ws, const ScanArgs &args, hipStream_t stream) {
    const dim3 grid((unsigned)args.total_waves), block(768);
    if (args.tp_d <= 32)
        hipLaunchKernelGGL((scan_tph_kernel<1, false, false, true>), grid, block, 0, stream, (uint32_t *)ws, args);
    else
        hipLaunchKernelGGL((scan_tph_kernel<2, false, false, true>), grid, block, 0, stream, (uint32_t *)ws, args);
}

}  // namespace mfma
}  // namespace ftc
