// Short causal scans for gfx950: chains of a few positions (a step of decoding, a short piece of
// a prompt), any row widths, fp32 or bf16 rows, a state handed in, out or both.
//
//   out[c, l, f] = sum_{j <= l} (a[c,l,:] . b[c,j,:]) * v[c,j,f]  (REV: j >= l)  + a[c,l,:] . s0[c,:,f]
//
// What bounds such a call is the state (D x F floats in and out against (3 D + 2 F) L values of
// rows) and, on few chains, latency: a chunk of 32 positions on the matrix cores, cut, staged
// and multiplied, takes 11 us where one position is all there is.  Here a value of the state
// is read once, updated in a register for every position, written once, and every load of a
// lane is issued before the first is used.
//
//  * A workgroup of 256 lanes owns 64 columns of one chain's state: 64 / VEC lanes side by side
//    (VEC = 4: 16-byte loads; 1: widths and addresses that do not allow them), the remaining
//    factor takes every kGroups-th row.  A lane keeps its columns of all v rows and its share of
//    all out rows in registers (LM positions) and walks its rows of the state.
//  * The partial out rows are summed in a fixed order: the row groups of a wavefront across
//    lanes, the four wavefronts through LDS.
//  * All arithmetic is fp32 fused multiply-adds on the vector unit.
//
// Measured: one step of 256 chains of 64 x 64 10.1 -> 4.6 us, of 8192 chains 87 -> 48 us (268 MB of
// state in and out: 5.6 TB/s), of 1024 chains of 128 x 128 69 -> 22 us.
#include <algorithm>

#include "ftc_common.h"

namespace ftc {
namespace {

constexpr int kLanes = 256, kCols = 64;
constexpr int kMostRows = 512;  // rows of a state

struct ShortArgs {
    ScanDesc scan[kMfmaMaxScans];
    int32_t H, L, most_blocks;  // most_blocks: blocks of 64 columns of the widest scan
};

template <int VEC>
struct Cols {
    float x[VEC];
};

template <int VEC>
__device__ __forceinline__ Cols<VEC> load_cols(const void *base, int dtype, int64_t at) {
    Cols<VEC> r;
    if (VEC == 4) {
        if (dtype == FTC_F32) {
            const float4 t = *(const float4 *)((const float *)base + at);
            r.x[0] = t.x, r.x[1 % VEC] = t.y, r.x[2 % VEC] = t.z, r.x[3 % VEC] = t.w;
        } else {
            const ushort4 t = *(const ushort4 *)((const uint16_t *)base + at);
            r.x[0] = bf16_to_f32(t.x), r.x[1 % VEC] = bf16_to_f32(t.y);
            r.x[2 % VEC] = bf16_to_f32(t.z), r.x[3 % VEC] = bf16_to_f32(t.w);
        }
    } else {
        r.x[0] = load_as_f32(base, dtype, at);
    }
    return r;
}
template <int VEC>
__device__ __forceinline__ void store_cols(void *base, int dtype, int64_t at, const Cols<VEC> &r) {
    if (VEC == 4) {
        if (dtype == FTC_F32)
            *(float4 *)((float *)base + at) = make_float4(r.x[0], r.x[1 % VEC], r.x[2 % VEC], r.x[3 % VEC]);
        else
            *(ushort4 *)((uint16_t *)base + at) =
                make_ushort4(f32_to_bf16(r.x[0]), f32_to_bf16(r.x[1 % VEC]), f32_to_bf16(r.x[2 % VEC]),
                             f32_to_bf16(r.x[3 % VEC]));
    } else {
        store_from_f32(base, dtype, at, r.x[0]);
    }
}

// LM: positions held in registers (L <= LM); VEC: columns per lane
template <int LM, int VEC>
__global__ __launch_bounds__(kLanes) void short_scan_kernel(ShortArgs p) {
    constexpr int kAcross = kCols / VEC;          // lanes side by side
    constexpr int kGroups = kLanes / kAcross;     // rows of the state taken at a time
    constexpr int kWaves = kLanes / 64;
    constexpr int kUnroll = 4;                    // rows of the state in flight per lane
    const ScanDesc &sd = p.scan[blockIdx.z];
    const int D = sd.a.width, F = sd.v.width, L = p.L;
    const int f = (int)blockIdx.y * kCols + (threadIdx.x % kAcross) * VEC;
    const int group = threadIdx.x / kAcross;
    if ((int)blockIdx.y * kCols >= F) return;     // (another scan of the launch is wider)
    const bool in = f < F;
    const int n = (int)(blockIdx.x / (uint32_t)p.H), h = (int)(blockIdx.x % (uint32_t)p.H);
    // position j of the walk is row j or, walking down, row L - 1 - j
    auto row = [&](int j) -> int64_t { return sd.reverse ? L - 1 - j : j; };
    const int64_t a0 = n * sd.a.stride_n + h * sd.a.stride_h, b0 = n * sd.b.stride_n + h * sd.b.stride_h,
                  v0 = n * sd.v.stride_n + h * sd.v.stride_h + f,
                  o0 = n * sd.out.stride_n + h * sd.out.stride_h + f;
    const float *s_in = sd.initial.ptr
                            ? sd.initial.ptr + n * sd.initial.stride_n + h * sd.initial.stride_h + f
                            : nullptr;
    float *s_out = sd.final_.ptr ? sd.final_.ptr + n * sd.final_.stride_n + h * sd.final_.stride_h + f
                                 : nullptr;

    // the rows of a and b as fp32, the positions of a column side by side
    __shared__ __align__(16) float ab[2][kMostRows][LM];
    for (int i = threadIdx.x; i < LM * D; i += kLanes) {
        const int j = i / D, d = i % D;
        ab[0][d][j] = j < L ? load_as_f32(sd.a.ptr, sd.a.dtype, a0 + row(j) * sd.a.stride_l + d) : 0.f;
        ab[1][d][j] = j < L ? load_as_f32(sd.b.ptr, sd.b.dtype, b0 + row(j) * sd.b.stride_l + d) : 0.f;
    }
    Cols<VEC> v[LM], o[LM];
#pragma unroll
    for (int j = 0; j < LM; j++) {
#pragma unroll
        for (int e = 0; e < VEC; e++) v[j].x[e] = o[j].x[e] = 0.f;
        if (j < L && in) v[j] = load_cols<VEC>(sd.v.ptr, sd.v.dtype, v0 + row(j) * sd.v.stride_l);
    }
    bool staged = false;
    for (int d0 = group; d0 < D || !staged; d0 += kUnroll * kGroups) {
        Cols<VEC> s[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const int d = d0 + u * kGroups;
#pragma unroll
            for (int e = 0; e < VEC; e++) s[u].x[e] = 0.f;
            if (s_in && d < D && in) s[u] = load_cols<VEC>(s_in, FTC_F32, d * sd.initial.stride_d);
        }
        if (!staged) __syncthreads();             // (with the first rows of the state on their way)
        staged = true;
#pragma unroll
        for (int u = 0; u < kUnroll; u++) {
            const int d = d0 + u * kGroups;
            if (d >= D) continue;
#pragma unroll
            for (int j = 0; j < LM; j++)
#pragma unroll
                for (int e = 0; e < VEC; e++) {
                    s[u].x[e] = fmaf(ab[1][d][j], v[j].x[e], s[u].x[e]);
                    o[j].x[e] = fmaf(ab[0][d][j], s[u].x[e], o[j].x[e]);
                }
            if (s_out && in) store_cols<VEC>(s_out, FTC_F32, d * sd.final_.stride_d, s[u]);
        }
    }
    // the row groups of a wavefront, then the wavefronts
    __shared__ float part[kWaves][LM][kCols];
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
#pragma unroll
    for (int j = 0; j < LM; j++)
#pragma unroll
        for (int e = 0; e < VEC; e++) {
            float x = o[j].x[e];
#pragma unroll
            for (int step = kAcross; step < 64; step *= 2) x += __shfl_xor(x, step);
            if (lane < kAcross) part[wave][j][lane * VEC + e] = x;
        }
    __syncthreads();
    for (int i = threadIdx.x; i < L * kAcross; i += kLanes) {
        const int j = i / kAcross, c = (i % kAcross) * VEC;
        if ((int)blockIdx.y * kCols + c >= F) continue;
        Cols<VEC> y;
#pragma unroll
        for (int e = 0; e < VEC; e++)
            y.x[e] = (part[0][j][c + e] + part[1][j][c + e]) + (part[2][j][c + e] + part[3][j][c + e]);
        store_cols<VEC>(sd.out.ptr, sd.out.dtype, o0 - f + (int)blockIdx.y * kCols + c + row(j) * sd.out.stride_l, y);
    }
}

template <int LM>
void launch(bool quads, dim3 grid, const ShortArgs &args, hipStream_t stream) {
    if (quads)
        hipLaunchKernelGGL((short_scan_kernel<LM, 4>), grid, dim3(kLanes), 0, stream, args);
    else
        hipLaunchKernelGGL((short_scan_kernel<LM, 1>), grid, dim3(kLanes), 0, stream, args);
}

}  // namespace

int short_scans(const ScanDesc *scans, int n, int64_t N, int64_t H, int64_t L, hipStream_t stream) {
    note_kernel("short_scan_kernel");
    if (plan_only()) {
        for (int i = 0; i < n; i++)
            note_plan("short_scan_kernel: 1 scan (%s), state %d x %d, %lld chains, %lld rows, workspace 0 bytes",
                      scans[i].reverse ? "first one reverse" : "first one forward", scans[i].a.width,
                      scans[i].v.width, (long long)(N * H), (long long)L);
        return FTC_OK;
    }
    ShortArgs args;
    int widest = 0;
    bool quads = true;  // four columns of v, out and the states at a time
    for (int i = 0; i < n; i++) {
        const ScanDesc &sd = scans[i];
        args.scan[i] = sd;
        widest = std::max(widest, sd.v.width);
        auto fits = [](const void *ptr, int64_t sn, int64_t sh, int64_t sl, int bytes) {
            return (uintptr_t)ptr % (4 * bytes) == 0 && sn % 4 == 0 && sh % 4 == 0 && sl % 4 == 0;
        };
        auto row_fits = [&](const void *ptr, int64_t sn, int64_t sh, int64_t sl, int dtype) {
            return fits(ptr, sn, sh, L > 1 ? sl : 0, dtype == FTC_F32 ? 4 : 2);
        };
        quads = quads && sd.v.width % 4 == 0 &&
                row_fits(sd.v.ptr, sd.v.stride_n, sd.v.stride_h, sd.v.stride_l, sd.v.dtype) &&
                row_fits(sd.out.ptr, sd.out.stride_n, sd.out.stride_h, sd.out.stride_l, sd.out.dtype) &&
                fits(sd.initial.ptr, sd.initial.stride_n, sd.initial.stride_h, sd.initial.stride_d, 4) &&
                fits(sd.final_.ptr, sd.final_.stride_n, sd.final_.stride_h, sd.final_.stride_d, 4);
    }
    args.H = (int32_t)H, args.L = (int32_t)L;
    args.most_blocks = (widest + kCols - 1) / kCols;
    const dim3 grid((unsigned)(N * H), (unsigned)args.most_blocks, (unsigned)n);
    if (L <= 1)
        launch<1>(quads, grid, args, stream);
    else if (L <= 4)
        launch<4>(quads, grid, args, stream);
    else
        launch<8>(quads, grid, args, stream);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return fail(FTC_ERR_HIP, "short scan launch failed: %s", hipGetErrorString(err));
    return FTC_OK;
}

// Scans that are handed a state or hand one on (steps and short pieces of a longer sequence).
// One position always: 4.6 us against 10.1 (256 chains of 64 x 64, fp32), 48 against 87 (8192 chains:
// 268 MB in and out, 5.6 TB/s), 22 against 69 (1024 chains of 128 x 128), 6.4 against 6.8 (2048 of
// 32 x 32, bf16 rows).  With more positions the matrix cores' share grows and the state's does
// not: up to 4 positions on states from 64 x 64 and up to 2048 chains (8192 chains, 4 positions, bf16
// rows: 72 against 67; 2048 chains of 32 x 32: 10.6 against 9.1), up to 8 where the state is
// wider (1024 chains of 128 x 128, 8 positions: 40 against 70) or, fp32 rows, there are at most
// 1024 chains (256 chains of 64 x 64, 8 positions: 8.1 against 10.2; bf16 rows on 8 chains, one
// chunk of the register-fed kernel: 8.2 against 6.1).
bool short_scans_take(const ScanDesc *scans, int n, int64_t N, int64_t H, int64_t L) {
    const int forced = tuning().short_most;  // tuning aid: the most positions
    if (n < 1 || n > kMfmaMaxScans || L > 8 || (forced >= 0 && L > forced)) return false;
    for (int i = 0; i < n; i++) {
        const int64_t D = scans[i].a.width, state = D * scans[i].v.width;
        if (D > kMostRows || !(scans[i].initial.ptr || scans[i].final_.ptr)) return false;
        if (L == 1 || forced > 0) continue;
        const bool fp32 = scans[i].a.dtype == FTC_F32 && scans[i].b.dtype == FTC_F32 && scans[i].v.dtype == FTC_F32;
        if (N * H > 2048 || state < 64 * 64) return false;
        if (L > 4 && state <= 64 * 64 && !(fp32 && N * H <= 1024)) return false;
    }
    return true;
}

}  // namespace ftc
