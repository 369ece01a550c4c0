// Chain-parallel scan on the fp16 matrix path (ftc_tph_kernel.h): launcher.
#include "ftc_tph_kernel.h"

namespace ftc {
namespace mfma {

namespace {
template <int KS>
void launch(void *ws, const ScanArgs &args, bool odd, hipStream_t stream) {
    // (grid as for launch_scan_tp)
    const dim3 grid((unsigned)args.total_waves), block(768);
    if (odd)
        hipLaunchKernelGGL((scan_tph_kernel<KS, true>), grid, block, 0, stream, (uint32_t *)ws, args);
    else
        hipLaunchKernelGGL((scan_tph_kernel<KS, false>), grid, block, 0, stream, (uint32_t *)ws, args);
}
}  // namespace

void launch_scan_tph(void *ws, const ScanArgs &args, bool odd, hipStream_t stream) {
    if (args.tp_d <= 32)
        launch<1>(ws, args, odd, stream);
    else
        launch<2>(ws, args, odd, stream);
}

}  // namespace mfma
}  // namespace ftc
