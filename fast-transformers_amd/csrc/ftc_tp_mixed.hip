// Chain-parallel scans with bf16 rows among them (ftc_tp_kernel.h): kernels and launcher.
//
// A bf16 value is one piece: such rows go from memory into the piece tiles as they are, and a product
// of them is one matrix instruction (three with the state, the chunk product or the fp32 gradient,
// which stay in three pieces, so nothing of them is lost).  A chunk of the 64 x 64 forward issues 24
// matrix instructions per consumer where fp32 rows take 72, and its producers copy instead of cutting:
// 0.63 us a chunk against 1.1 on the two scaled fp16 pieces that such rows had before, which memory
// then bounds (256 chains, L=4096, forward 152 -> 131 us, 5.3 TB/s; 80 chains, L=1000, backward 42 -> 34).
#include "ftc_tp_kernel.h"

namespace ftc {
namespace mfma {
namespace {

// FORWARD: all rows bf16, fp32 results; else the scans of a backward call, which differ in the operand
// that is the fp32 gradient, with bf16 results
template <int ND, int KS2, bool FORWARD>
__device__ __forceinline__ void scan_mixed(uint32_t *__restrict__ ws_ptr, const ScanArgs &p) {
    __shared__ __align__(16) char pieces_mem[FORWARD ? kTpPieceBytes<1, 1, 1> : kTpPieceBytes<3, 1, 1>];
    __shared__ __align__(16) char pt_mem[kTpPtBytes / 2 * 3];
    __shared__ uint32_t order_sh;
    lds_char *const pieces = (lds_char *)pieces_mem, *const pt = (lds_char *)pt_mem;
    uint32_t which, chain;
    tp_workgroup(p, which, chain);
    if constexpr (FORWARD) {
        scan_tp_body<ND, KS2, false, 1, 1, 1, float>(ws_ptr, p, which, chain, pieces, pt, nullptr, &order_sh);
    } else {
        const int rows = p.scan[which / (uint32_t)(p.nseg * p.tp_fblocks)].pad;
        if (!(rows & kRowsBf16A))
            scan_tp_body<ND, KS2, false, 3, 1, 1, bf16_t>(ws_ptr, p, which, chain, pieces, pt, nullptr, &order_sh);
        else if (!(rows & kRowsBf16B))
            scan_tp_body<ND, KS2, false, 1, 3, 1, bf16_t>(ws_ptr, p, which, chain, pieces, pt, nullptr, &order_sh);
        else
            scan_tp_body<ND, KS2, false, 1, 1, 3, bf16_t>(ws_ptr, p, which, chain, pieces, pt, nullptr, &order_sh);
    }
}
template <int ND, int KS2, bool FORWARD>
__global__ __launch_bounds__(512, 2) void scan_tp_bf16_kernel(uint32_t *__restrict__ ws_ptr, ScanArgs p) {
    scan_mixed<ND, KS2, FORWARD>(ws_ptr, p);
}

template <bool FORWARD>
void launch(void *ws, const ScanArgs &args, hipStream_t stream) {
    const dim3 grid((unsigned)args.total_waves), block(512);
#define FTC_LAUNCH(ND, KS2) \
    hipLaunchKernelGGL((scan_tp_bf16_kernel<ND, KS2, FORWARD>), grid, block, 0, stream, (uint32_t *)ws, args)
    if (args.tp_d <= 32) FTC_LAUNCH(1, 1);
    else if (args.tp_d <= 64) FTC_LAUNCH(1, 2);
    else if (args.tp_d <= 96) FTC_LAUNCH(2, 1);
    else FTC_LAUNCH(2, 2);
#undef FTC_LAUNCH
}
}  // namespace

void launch_scan_tp_mixed(void *ws, const ScanArgs &args, hipStream_t stream) {
    if (args.scan[0].pad & kRowsBf16Out)
        launch<false>(ws, args, stream);
    else
        launch<true>(ws, args, stream);
}

}  // namespace mfma
}  // namespace ftc
