// The three gradient scans of the fused attention in one launch (ftc_tph_kernel.h, GRAD): launcher.
#include "ftc_tph_kernel.h"

namespace ftc {
namespace mfma {

__global__ __launch_bounds__(768, 3) void scan_tph_gradients_kernel(uint32_t *__restrict__ ws_ptr, ScanArgs p) {
    scan_tph_body<2, false, true>(ws_ptr, p);
}

void launch_scan_tph_gradients(void *ws, const ScanArgs &args, hipStream_t stream) {
    hipLaunchKernelGGL(scan_tph_gradients_kernel, dim3((unsigned)args.total_waves), dim3(768), 0, stream,
                       (uint32_t *)ws, args);
}

}  // namespace mfma
}  // namespace ftc
