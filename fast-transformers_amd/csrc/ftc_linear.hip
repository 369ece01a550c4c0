// The encoder's matrix products on the fp16 matrix cores at the precision of fp32, and the passes
// that feed them (include/ftc_causal_product.h: ftc_split_weights, ftc_split_rows,
// ftc_layer_norm_split, ftc_linear_split).
//
//   out[t, f] = sum_k x[t, k] w[f, k] + bias[f]   (+ residual[t, f], or max(., 0))
//
// The fp32 matrix rate of this card is 157 TFLOP/s and the library's products of the encoder's
// sizes reach 111 to 131 of them; fp16 matrix cores do sixteen times that.  As in
// ftc_tph_kernel.h a row is scaled by a power of two and cut into two fp16 pieces, hi = fp16(x s)
// and lo = fp16(x s - hi), and a product is hi hi + hi lo + lo hi, each exact in the fp32
// accumulator.  A row's largest value is scaled to 2^14 .. 2^15, so hi + lo stands for every value
// down to 2^-17 of that to within one unit in the last place of fp32 (and for smaller ones to
// 2^-40 of the row's largest); the sums are fp32 sums of 32 products per rounding, where the
// library rounds after every few: against float64 a product of 40960 x 512 by 512 x 512 is off by
// 1.9e-7 (2-norm) where the library's is by 2.9e-7, of 1024 columns by 2.6e-7 and 4.1e-7.
//
// Measured, 40960 tokens (us, library / here): 512 -> 512 191 / 67, 512 -> 1536 475 / 173, 512 -> 1024
// with relu 310 + 51 / 123, 1024 -> 512 with the residual 305 + 37 / 122, with a norm made again 128; 5000 tokens,
// 256 -> 512 20 / 9; 300 tokens, 128 -> 260 31 / 4.2.  (At the largest sizes the card's power bounds it: 512 -> 1536 on
// zeros 134, 1024 -> 512 100.)
//
// Rows in pieces take the bytes of fp32 rows: block of 32 columns after block, 64 bytes of hi and 64
// of lo each, one cache line per row and k-step.  Whoever writes rows that only a product reads
// writes them in pieces; the scale must be known before the row's first value is cut, so the
// producer has the whole row (layer norm, ftc_split_rows) or a bound (relu: |y| <= max|x| max_f
// sum_k |w[f, k]| + the largest bias, six or seven bits above a row's ordinary values, which the
// seventeen bits above leave room for).  Where the features are too far apart for one bound -- it is
// more than 2^6 times max|x| sum_k |w[f, k]| of the least of them -- a row leaves the product in fp32
// and a pass behind it (cut_rows_kernel) cuts it by its own largest value (where no row needs it,
// 4.6 us for 40960 rows).
#include <algorithm>
#include <type_traits>

#include "ftc_tp_kernel.h"
#include "ftc_tph_kernel.h"

namespace ftc {
namespace {
using namespace mfma;

constexpr int kStep = 32;                // columns per k-step
constexpr int kRowBytes = 4 * kStep;     // a row's bytes of a k-step: hi, lo
// Columns or features of a row (128 rows of 2^20 floats stay within a descriptor's 2^31 bytes) and
// rows of a launch of a wavefront each (HIP takes fewer than 2^32 lanes).
constexpr int64_t kMostColumns = 1 << 20, kMostRows = 1 << 26;

// the power of two that brings a largest magnitude to 2^14 .. 2^15, and its reciprocal
__device__ __forceinline__ void scale_of(float largest, float &s, float &inverse) {
    const int e = (int)((__float_as_uint(largest) >> 23) & 0xffu);  // largest < 2^(e - 126)
    const int up = max(-126, min(126, 141 - e));  // (a row of zeros: 126, so that its scale bounds it)
    s = __uint_as_float((uint32_t)(127 + up) << 23);
    inverse = __uint_as_float((uint32_t)(127 - up) << 23);
}
// four consecutive columns of a row in pieces
__device__ __forceinline__ void store_pieces(char *row, int col, const float4 &x, float s) {
    uint32_t h0, h1, l0, l1;
    cut_quad_f16(x.x, x.y, x.z, x.w, s, h0, h1, l0, l1);
    char *at = row + (col / kStep) * kRowBytes + 2 * (col % kStep);
    *(uint2 *)at = make_uint2(h0, h1);
    *(uint2 *)(at + 2 * kStep) = make_uint2(l0, l1);
}
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
    for (int step = 32; step > 0; step >>= 1) x += __shfl_xor(x, step);
    return x;
}
__device__ __forceinline__ float wave_largest(float x) {
#pragma unroll
    for (int step = 32; step > 0; step >>= 1) x = fmaxf(x, __shfl_xor(x, step));
    return x;
}
__device__ __forceinline__ float largest_of(const float4 &x) {
    return fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w)));
}

// ---- weights: a wavefront per row of any of the matrices --------------------------------------
constexpr int kMostWeights = 48;        // (2.7 KB of kernel arguments)
struct WeightList {
    const float *w[kMostWeights], *bias[kMostWeights];
    int32_t first[kMostWeights + 1];     // rows before each matrix, in all at the end
    int32_t cols[kMostWeights];
    char *pieces[kMostWeights];          // of the matrix
    float *scale[kMostWeights], *bias_out[kMostWeights], *norm[kMostWeights];
    int32_t count;
};
__global__ __launch_bounds__(256) void split_weights_kernel(WeightList list) {
    const int row = (int)(blockIdx.x * 4 + threadIdx.x / 64), lane = threadIdx.x % 64;
    if (row >= list.first[list.count]) return;
    // (one look at all the matrices; one by one, half a microsecond)
    const int m = __popcll(__ballot(lane < list.count && row >= list.first[lane + 1 < kMostWeights ? lane + 1 : kMostWeights]));
    const int r = row - list.first[m], cols = list.cols[m];
    const float *w = list.w[m] + (int64_t)r * cols;
    float largest = 0.f, sum = 0.f;
    for (int c = 4 * lane; c < cols; c += 256) {
        const float4 x = *(const float4 *)(w + c);
        largest = fmaxf(largest, largest_of(x));
        sum += (fabsf(x.x) + fabsf(x.y)) + (fabsf(x.z) + fabsf(x.w));
    }
    largest = wave_largest(largest);
    sum = wave_sum(sum);
    float s, inverse;
    scale_of(largest, s, inverse);
    char *out = list.pieces[m] + (int64_t)r * cols * 4;
    for (int c = 4 * lane; c < cols; c += 256) store_pieces(out, c, *(const float4 *)(w + c), s);
    if (lane == 0) {
        list.scale[m][r] = inverse;
        list.bias_out[m][r] = list.bias[m] ? list.bias[m][r] : 0.f;
        list.norm[m][r] = sum;
    }
}

// ---- rows: a wavefront per row, which it keeps in registers ------------------------------------
// a value of a layer norm's row, less the row's mean, r = 1 / sqrt(variance + eps); rounded the same wherever it is made
__device__ __forceinline__ float normed(float less_mean, float r, float gamma, float beta) {
    return __builtin_fmaf(less_mean * r, gamma, beta);
}
// NORM: layer norm first (torch's: biased variance, two passes over the row in fp32).  Its rows go out, or only what
// they are made of beside x, (mean, r) of each: who reads them as a residual then makes them again from x.
// Bound by memory: 40960 rows of 512, pieces and rows 40.3 us, pieces and (mean, r) 29.7.
constexpr int kMostQuads = 16;           // quads of a row per lane: rows of up to 4096 values
template <int QUADS, bool NORM>
__global__ __launch_bounds__(256) void rows_kernel(const float *__restrict__ x, const float *__restrict__ gamma,
                                                   const float *__restrict__ beta, float eps, int64_t rows,
                                                   int cols, float *__restrict__ out, float2 *__restrict__ stats,
                                                   char *__restrict__ pieces, float *__restrict__ scale) {
    const int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.x / 64;
    const int lane = threadIdx.x % 64;
    if (row >= rows) return;
    float4 v[QUADS];
#pragma unroll
    for (int i = 0; i < QUADS; i++) {
        const int c = 4 * (lane + 64 * i);
        v[i] = c < cols ? *(const float4 *)(x + row * cols + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if (NORM) {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < QUADS; i++) sum += (v[i].x + v[i].y) + (v[i].z + v[i].w);
        const float mean = wave_sum(sum) / (float)cols;
        float squares = 0.f;
#pragma unroll
        for (int i = 0; i < QUADS; i++) {
            if (4 * (lane + 64 * i) >= cols) continue;
            v[i].x -= mean, v[i].y -= mean, v[i].z -= mean, v[i].w -= mean;
            squares += (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);
        }
        const float r = 1.0f / sqrtf(wave_sum(squares) / (float)cols + eps);
#pragma unroll
        for (int i = 0; i < QUADS; i++) {
            const int c = 4 * (lane + 64 * i);
            if (c >= cols) continue;
            const float4 g = gamma ? *(const float4 *)(gamma + c) : make_float4(1.f, 1.f, 1.f, 1.f);
            const float4 b = beta ? *(const float4 *)(beta + c) : make_float4(0.f, 0.f, 0.f, 0.f);
            v[i].x = normed(v[i].x, r, g.x, b.x), v[i].y = normed(v[i].y, r, g.y, b.y);
            v[i].z = normed(v[i].z, r, g.z, b.z), v[i].w = normed(v[i].w, r, g.w, b.w);
            if (out) *(float4 *)(out + row * cols + c) = v[i];
        }
        if (stats && lane == 0) stats[row] = make_float2(mean, r);
    }
    if (!pieces) return;
    float largest = 0.f;
#pragma unroll
    for (int i = 0; i < QUADS; i++) largest = fmaxf(largest, largest_of(v[i]));
    largest = wave_largest(largest);
    float s, inverse;
    scale_of(largest, s, inverse);
#pragma unroll
    for (int i = 0; i < QUADS; i++) {
        const int c = 4 * (lane + 64 * i);
        if (c < cols) store_pieces(pieces + row * cols * 4, c, v[i], s);
    }
    if (lane == 0) scale[row] = inverse;
}

// Rows that the product left in fp32 (scale < 0, a row's values where its pieces go) in pieces, each
// in its place: a wavefront reads 256 columns and writes the same 1024 bytes.  A wavefront looks at
// kCutRows rows.
constexpr int kCutRows = 8;
__global__ __launch_bounds__(256) void cut_rows_kernel(char *rows, float *scale, int64_t count, int cols) {
    const int64_t first = ((int64_t)blockIdx.x * 4 + threadIdx.x / 64) * kCutRows;
    const int lane = threadIdx.x % 64;
    const bool here = lane < kCutRows && first + lane < count && scale[first + lane] < 0.f;
    for (uint64_t left = __ballot(here); left != 0; left &= left - 1) {
        const int64_t r = first + __builtin_ctzll(left);
        char *const row = rows + r * cols * 4;
        float largest = 0.f;
        for (int c = 4 * lane; c < cols; c += 256) largest = fmaxf(largest, largest_of(*(const float4 *)(row + 4 * c)));
        largest = wave_largest(largest);
        float s, inverse;
        scale_of(largest, s, inverse);
        for (int c0 = 0; c0 < cols; c0 += 256) {
            const int c = c0 + 4 * lane;
            float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
            if (c < cols) x = *(const float4 *)(row + 4 * c);
            // (every lane's value is here before any lane writes where it was)
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w)::"memory");
            if (c < cols) store_pieces(row, c, x, s);
        }
        if (lane == 0) scale[r] = inverse;
    }
}

// ---- the product --------------------------------------------------------------------------------
struct LinearArgs {
    const char *x, *w;                   // rows in pieces
    const float *x_scale, *w_scale, *bias, *w_norm;
    const float *residual;               // kResidual, kNormed
    const float2 *stats;                 // kNormed: the residual is the layer norm of those rows
    const float *gamma, *beta;           // (or nullptr: ones, zeros)
    float *out;                          // kPlain, kResidual
    char *out_pieces;                    // kRelu
    float *out_scale;
    int64_t tokens;
    int32_t features, k, feature_tiles;
    bool streamed;                       // the rows go out past what is worth keeping in the caches
};
constexpr int kStreamed = 2;             // (a store's nt bit)
// Bytes that a product reads and writes from which on its rows are streamed.  Up to the Infinity Cache's 256 MB
// the next kernel finds them there; beyond, they only push out what both read again.  Streamed rows have to
// leave in whole lines.  Eight layers at 40960 tokens, d = 512, feed-forward 1024 (us, none / half lines / lines) 6470 /
// 6266 / 6156; four at 30400 2299 / - / 2277; 1024 -> 512 at 40960 tokens 133 / 142 / 128.  From 140 MB on
// instead, four layers at 24576 tokens take 2063 us for 1990, and from none on at 20480 1749 for 1682.
constexpr int64_t kStreamedBytes = (int64_t)176 << 20;
enum { kPlain = 0, kResidual = 1, kRelu = 2, kNormed = 3 };

// a raw buffer of `bytes` bytes
__device__ __forceinline__ u32x4 descriptor(const void *base, uint32_t bytes) {
    const uint64_t a = (uint64_t)base;
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu)),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), kRsrcFlags};
}
// 16 bytes per lane from memory into LDS, lane L to byte `to` + 16 L.  (Written out: the compiler
// does not follow which of the buffers a request of its own fills, and would wait for all
// requests before any read of LDS.  The waits are the k-loop's.)
__device__ __forceinline__ void load_to_lds(const u32x4 rs, uint32_t to, uint32_t offset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :: "s"(to), "v"(offset), "s"(rs) : "memory", "m0");
}

__device__ __forceinline__ void load_dword_to_lds(const u32x4 rs, uint32_t to, uint32_t offset) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                 :: "s"(to), "v"(offset), "s"(rs) : "memory", "m0");
}

// What lanes 8 to 15 of a row of 16 have from lanes 0 to 7 of `other`, the others their own, and the reverse
// (row_ror:8, written to the lanes of two of its four banks).
__device__ __forceinline__ uint32_t upper_from_lower(uint32_t own, uint32_t other) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)own, (int)other, 0x128, 0xf, 0xc, false);
}
__device__ __forceinline__ uint32_t lower_from_upper(uint32_t own, uint32_t other) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)own, (int)other, 0x128, 0xf, 0x3, false);
}
__device__ __forceinline__ uint32_t other_half(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xf, 0xf, false);
}

// A workgroup of four wavefronts takes tiles of TN tokens by TF features one after the other, a
// wavefront half of either.  v_mfma_f32_16x16x32_f16 with the features as rows of the result, so
// that a lane has four consecutive features of one token.  A k-step's rows (128 bytes each) go from
// memory straight into LDS through STAGES buffers, one barrier per step, and are requested STAGES
// steps ahead; a tile's last steps request the first ones of the next tile.
// Split: with 64 x 128 results per wavefront a step reads 24 KB of fragments for 96 matrix
// instructions (1536 cycles); smaller tiles read more of the LDS per instruction, and are there for
// products of few tiles (product_tile, below, where both are measured).
// Which feature row r of a feature tile's rows in LDS is.  Rows that leave in pieces: a lane has eight
// consecutive features, 8 g to 8 g + 7 of 32, in two tiles of 16, so that 16 bytes of hi and 16 of lo are one
// store each, of 64 consecutive bytes of a token (in 8-byte stores of 32: 40960 tokens, 512 -> 1024 135 us for 123).
template <bool PIECES>
__device__ __forceinline__ constexpr int feature_of(int r) {
    return PIECES ? r / 32 * 32 + 8 * (r % 16 / 4) + 4 * (r / 16 % 2) + r % 4 : r;
}
// LATER: a tile's rows go out during the next one's steps 1 to 8, four stores a step, the scaling under the
// matrix instructions (products of at least 10 steps on more than one round of tiles; the tile before waits in
// the registers that four wavefronts on a CU leave).  Otherwise all workgroups of a round write their rows, 33 MB,
// at once and compute nothing meanwhile.  With kStreamed, 40960 tokens, 512 -> 1536 178 -> 167 us, 512 -> 1024
// 119 either way; without, 11536 tokens, 512 -> 1536 65 -> 61; one round of tiles 25.8 -> 27.5.  (Wavefronts that
// only request rows, two beside the four, which then never wait for their stores to land, gained 1 %, small tiles lost up to 15 %.)
constexpr int kLaterSteps = 9;           // the first step and eight
template <int TN, int TF, int STAGES, int EPI, bool LATER = false>
__global__ __launch_bounds__(256, 1) void linear_kernel(LinearArgs p) {
    constexpr int WT = TN / 32, WF = TF / 32;          // tiles of 16 per wavefront
    constexpr int kBuf = (TN + TF) * kRowBytes;
    constexpr int kLoadsX = TN * kRowBytes / 4096, kLoadsW = TF * kRowBytes / 4096;  // per lane
    constexpr int kRequests = kLoadsX + kLoadsW;                                     // of a step
    constexpr int kStores = WT * WF;                                                 // per lane
    // scales and bias of a tile's tokens and features, as each wavefront needs them (64 to a request)
    constexpr int kScaleT = TN / 2 < 64 ? 64 : TN / 2, kScaleF = TF / 2 < 64 ? 64 : TF / 2;
    constexpr int kScales = kScaleT + 2 * kScaleF, kScaleLoads = kScales / 64;
    constexpr int kScaleSets = LATER ? 2 : 1;
    constexpr bool kAdds = EPI == kResidual || EPI == kNormed;
    static_assert(!LATER || (!kAdds && WF > WT && kRequests <= 3 * (WF - WT)), "requests before the stores of a step");
    static_assert(WF % 2 == 0 && TN / 2 <= 64, "the fragments of w in turn; a wavefront's tokens in a request");
    __shared__ __align__(16) char tiles_mem[STAGES * kBuf];
    __shared__ __align__(16) float scales_mem[kScaleSets][4][kScales];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 15, g = lane >> 4;
    const int wt = wave & 1, wf = wave >> 1;
    const uint32_t row_bytes = (uint32_t)p.k * 4;
    const int steps = p.k / kStep;
    // Workgroups go round the eight XCDs: those of one XCD take the feature tiles of a token tile
    // at the same time, so that its rows are read from memory once.
    struct Tile {
        int64_t t0;
        int f0, nt, nf;
        bool there;
        u32x4 x_rs, w_rs;
    };
    auto tile_of = [&](int round) -> Tile {
        const int idx = (int)(blockIdx.x / 8) + round * (int)(gridDim.x / 8);
        Tile t;
        t.t0 = ((int64_t)(idx / p.feature_tiles) * 8 + blockIdx.x % 8) * TN;
        t.f0 = (idx % p.feature_tiles) * TF;
        t.there = t.t0 < p.tokens;
        const int64_t from = t.there ? t.t0 : 0;
        t.nt = t.there ? (int)min((int64_t)TN, p.tokens - t.t0) : 0;
        t.nf = t.there ? min(TF, p.features - t.f0) : 0;
        t.x_rs = descriptor(p.x + from * row_bytes, (uint32_t)t.nt * row_bytes);
        t.w_rs = descriptor(p.w + (int64_t)t.f0 * row_bytes, (uint32_t)t.nf * row_bytes);
        return t;
    };
    // lane's 16 bytes of a load: slot j of the tile holds piece-and-quarter (j % 8) ^ key of row j / 8
    uint32_t x_off[kLoadsX], w_off[kLoadsW];
#pragma unroll
    for (int i = 0; i < kLoadsX; i++) {
        const int j = (i * 4 + wave) * 64 + lane, row = j / 8;
        x_off[i] = (uint32_t)row * row_bytes + 16u * ((j % 8) ^ TpSwizzle<128>::key(row));
    }
#pragma unroll
    for (int i = 0; i < kLoadsW; i++) {
        const int j = (i * 4 + wave) * 64 + lane, row = j / 8;
        w_off[i] = (uint32_t)feature_of<EPI == kRelu>(row) * row_bytes + 16u * ((j % 8) ^ TpSwizzle<128>::key(row));
    }
    lds_char *const tiles = (lds_char *)tiles_mem;
    const uint32_t lds0 = (uint32_t)(uintptr_t)tiles + 1024u * wave;
    const uint32_t scales0 = (uint32_t)(uintptr_t)(lds_char *)scales_mem + (uint32_t)(kScales * 4) * wave;
    constexpr uint32_t kScaleSet = 4 * 4 * kScales;
    // The step whose rows are requested: STAGES steps ahead of the one that is computed, in this
    // tile or in a later one.
    Tile ahead = tile_of(0);
    int ahead_step = 0, ahead_round = 0;
    auto fetch = [&](uint32_t buf, int i) {  // request number i of that step
        const uint32_t at = (uint32_t)ahead_step * kRowBytes, to = lds0 + buf;
        if (i < kLoadsX)
            load_to_lds(ahead.x_rs, to + 4096u * i, x_off[i % kLoadsX] + at);
        else
            load_to_lds(ahead.w_rs, to + TN * kRowBytes + 4096u * (i - kLoadsX), w_off[(i - kLoadsX) % kLoadsW] + at);
    };
    auto advance = [&]() {
        if (++ahead_step == steps) ahead_step = 0, ahead = tile_of(++ahead_round);
    };
    auto fetch_scales = [&](const Tile &t, uint32_t scales0) {
        const u32x4 xs_rs = descriptor(p.x_scale + t.t0, (uint32_t)t.nt * 4u),
                    ws_rs = descriptor(p.w_scale + t.f0, (uint32_t)t.nf * 4u),
                    b_rs = descriptor(p.bias + t.f0, (uint32_t)t.nf * 4u);
        load_dword_to_lds(xs_rs, scales0, 4u * (uint32_t)(wt * (TN / 2) + lane));
#pragma unroll
        for (int i = 0; i < kScaleF / 64; i++) {
            const uint32_t from = 4u * (uint32_t)(wf * (TF / 2) + 64 * i + lane);
            load_dword_to_lds(ws_rs, scales0 + 4u * (kScaleT + 64 * i), from);
            load_dword_to_lds(b_rs, scales0 + 4u * (kScaleT + kScaleF + 64 * i), from);
        }
    };
    int x_addr[2], w_addr[2];  // [piece]; further tiles 16 rows of 128 bytes on
#pragma unroll
    for (int k = 0; k < 2; k++) {
        x_addr[k] = TpSwizzle<128>::addr(wt * (TN / 2) + ln, 64 * k + 16 * g);
        w_addr[k] = TN * kRowBytes + TpSwizzle<128>::addr(wf * (TF / 2) + ln, 64 * k + 16 * g);
    }
    // requests in flight of later steps than the next one
    constexpr int kFlying = (STAGES - 2) * kRequests;
    f32x4 acc[WF][WT];
    Frag xh[WT], xl[WT], w[2][2];
    auto first_frags = [&](const lds_char *buf) {
#pragma unroll
        for (int k = 1; k >= 0; k--) {
            w[0][k] = lds_frag16(buf + w_addr[k]);
#pragma unroll
            for (int j = 0; j < WT; j++) (k ? xh[j] : xl[j]) = lds_frag16(buf + x_addr[1 - k] + j * 16 * kRowBytes);
        }
    };
    // One step, written out in issue order: fragments of the next feature tile and a request for a
    // later step under the matrix instructions of this one, instructions that add to one
    // accumulator at least WT apart.  The barrier stands before the last feature tile's
    // instructions: the wavefront has read all it needs of this step's buffer by then, and under
    // those instructions the first fragments of the next step arrive, whose rows the wait
    // before the barrier has seen land.  Of the requests of the step that takes this buffer over,
    // the first ones run under the same instructions and the others under the next step's; those
    // of a tile's last step all before the rows go out, so that no later wait for them waits for
    // the rows.
    auto compute = [&](const lds_char *buf, const lds_char *next, uint32_t to_now, uint32_t to_before, auto first,
                       auto last, auto wait, auto out) {
        constexpr int kSlots = 3 * WF;
        static_assert(kSlots >= kRequests, "a request per group of matrix instructions");
        auto slot_of = [](int r) -> int { return LATER ? r : r * kSlots / kRequests; };
        Frag xn[WT];
#pragma unroll
        for (int i = 0; i < WF; i++) {
            if (i == WF - 1) {
                wait();
                advance();
            }
#pragma unroll
            for (int m = 0; m < 3; m++) {
                if (i + 1 < WF) {
                    if (m > 0) w[(i + 1) % 2][2 - m] = lds_frag16(buf + w_addr[2 - m] + (i + 1) * 16 * kRowBytes);
                } else if (m < 2) {
                    w[0][1 - m] = lds_frag16(next + w_addr[1 - m]);
                    if (m == 0) {
#pragma unroll
                        for (int j = 0; j < WT; j++) xn[j] = lds_frag16(next + x_addr[0] + j * 16 * kRowBytes);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < WT; j++) xl[j] = lds_frag16(next + x_addr[1] + j * 16 * kRowBytes);
                }
                const int slot = i == WF - 1 ? m : 3 + 3 * i + m;
#pragma unroll
                for (int r = 0; r < kRequests; r++) {
                    if (i == WF - 1 ? (decltype(last)::value ? r * 3 / kRequests == m : slot_of(r) == slot)
                                    : !decltype(first)::value && slot_of(r) == slot)
                        fetch(i == WF - 1 ? to_now : to_before, r);
                }
#pragma unroll
                for (int j = 0; j < WT; j++)
                    acc[i][j] = mfma16h(w[i % 2][m == 0 ? 1 : 0], m == 1 ? xl[j] : xh[j], acc[i][j]);
                if (LATER && m == 1 && i >= WF - 4 && i < WF - 1 && (WF - i) % 2 == 0) out((i - (WF - 4)) / 2);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int j = 0; j < WT; j++) xh[j] = xn[j];
    };
    if (!ahead.there) return;
#pragma unroll
    for (int s = 0; s < STAGES; s++) {
#pragma unroll
        for (int i = 0; i < kRequests; i++) fetch((uint32_t)s * kBuf, i);
        if (s + 1 < STAGES) advance();
    }
    float bound_w = 0.f, bound_b = 0.f, least_w = __builtin_inff();
    if (EPI == kRelu) {  // (the same numbers in every workgroup)
#pragma unroll 4
        for (int i = lane; i < p.features; i += 64) {
            const float norm = p.w_norm[i], bias = p.bias[i];
            bound_w = fmaxf(bound_w, norm);
            bound_b = fmaxf(bound_b, bias);  // (a bias below zero, lowest or -inf, raises nothing)
            // (a feature without weights and with no bias above zero is zero in any row)
            least_w = fminf(least_w, norm == 0.f && !(bias > 0.f) ? __builtin_inff() : norm);
        }
        bound_w = wave_largest(bound_w), bound_b = wave_largest(bound_b);
        least_w = -wave_largest(-least_w);
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((STAGES - 1) * kRequests) : "memory");
    first_frags(tiles);
    uint32_t now = 0;
    auto after = [&](uint32_t buf) -> uint32_t { return buf == (STAGES - 1) * kBuf ? 0u : buf + kBuf; };
    // ---- rows out: every store is made, those outside the tensor outside the descriptor, so that
    // their number is known to the waits ----
    const uint32_t out_row = (uint32_t)p.features * 4u;
    struct Rows {                        // a tile's
        __amdgpu_buffer_rsrc_t rs;
        int f0;
        const float *scales;
        float xs[WT], s_out[WT];
        uint32_t at[WT][2];              // of a pair of feature tiles: either store's 16 bytes
    };
    const uint32_t upper = ln / 8;
    auto token_at = [&](int j) { return (uint32_t)(wt * (TN / 2) + 16 * j + ln) * out_row + 16u * g; };
    auto rows_of = [&](const Tile &t, const float *scales) -> Rows {
        Rows r;
        r.rs = __builtin_amdgcn_make_buffer_rsrc((EPI == kRelu ? (char *)p.out_pieces : (char *)p.out) + t.t0 * out_row, 0,
                                                 (uint32_t)t.nt * out_row, kRsrcFlags);
        r.f0 = t.f0 + wf * (TF / 2);
        r.scales = scales;
#pragma unroll
        for (int j = 0; j < WT; j++) {
            const int tok = 16 * j + ln;
            r.xs[j] = scales[tok];
            r.s_out[j] = 0.f;
            if (EPI == kRelu) {
                float inverse;
                const float x_most = 32768.f * r.xs[j], bound = x_most * bound_w + bound_b;
                scale_of(bound, r.s_out[j], inverse);
                if (!(bound <= 64.f * (x_most * least_w))) r.s_out[j] = 0.f, inverse = -1.f;  // (in fp32)
                const int64_t token = t.t0 + wt * (TN / 2) + tok;
                if (t.f0 == 0 && wf == 0 && g == 0 && token < p.tokens) p.out_scale[token] = inverse;
            }
            const uint32_t whole = EPI == kRelu && r.s_out[j] == 0.f, row = (uint32_t)(wt * (TN / 2) + tok) * out_row;
            const uint32_t whole_other = other_half(whole);
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const uint32_t half = p.streamed ? upper : u;
                const bool own = !p.streamed || half == u;
                const uint32_t wide = own ? whole : whole_other;
                r.at[j][u] = (own ? row : u ? row + 8 * out_row : row - 8 * out_row) + (16u << wide) * g + (64u >> 2 * wide) * half;
            }
        }
        return r;
    };
    struct Features { float4 ws[2], b[2]; };
    auto features_of = [&](const Rows &r, int pair) -> Features {
        Features w;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int fl = feature_of<EPI == kRelu>(32 * pair + 16 * u + 4 * g);
            w.ws[u] = *(const float4 *)(r.scales + kScaleT + fl);
            w.b[u] = *(const float4 *)(r.scales + kScaleT + kScaleF + fl);
        }
        return w;
    };
    // two tiles of 16 features of a token: 32 bytes per lane
    auto pair_out = [&](const Rows &r, const Features &w, int pair, int j, const f32x4 &low, const f32x4 &high,
                        const u32x4 *res) {
        float y[2][4];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const f32x4 &sum = u ? high : low;
            const float xs = r.xs[j];
            y[u][0] = fmaf(sum[0] * xs, w.ws[u].x, w.b[u].x), y[u][1] = fmaf(sum[1] * xs, w.ws[u].y, w.b[u].y);
            y[u][2] = fmaf(sum[2] * xs, w.ws[u].z, w.b[u].z), y[u][3] = fmaf(sum[3] * xs, w.ws[u].w, w.b[u].w);
        }
        uint32_t half[2][4];
        bool whole = false;                  // the row in fp32 instead of pieces
        if (EPI == kRelu) {
            whole = r.s_out[j] == 0.f;
#pragma unroll
            for (int u = 0; u < 2; u++) {
#pragma unroll
                for (int c = 0; c < 4; c++) y[u][c] = y[u][c] < 0.f ? 0.f : y[u][c];  // (keeps NaN, as torch's does)
                cut_quad_f16(y[u][0], y[u][1], y[u][2], y[u][3], r.s_out[j], half[0][2 * u], half[0][2 * u + 1],
                             half[1][2 * u], half[1][2 * u + 1]);
            }
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if (kAdds) y[u][c] += __uint_as_float(res[u][c]);
                if (EPI != kRelu || whole) half[u][c] = __float_as_uint(y[u][c]);
            }
        }
        const int f0 = r.f0 + 32 * pair, f = EPI == kRelu ? f0 : f0 + 4 * g;
        const uint32_t to = 4u * (uint32_t)f0;
        if (p.streamed) {
            // Lanes ln and ln ^ 8 change one half each, so that a store has whole lines: of tokens 0 to 7, of 8 to 15.
            u32x4 low_tokens, high_tokens;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                low_tokens[c] = upper_from_lower(half[0][c], half[1][c]);
                high_tokens[c] = lower_from_upper(half[1][c], half[0][c]);
            }
            const bool there = (EPI == kRelu ? f : f + 16 * (int)upper) < p.features;
            __builtin_amdgcn_raw_buffer_store_b128(low_tokens, r.rs, there ? r.at[j][0] + to : 0x80000000u, 0, kStreamed);
            __builtin_amdgcn_raw_buffer_store_b128(high_tokens, r.rs, there ? r.at[j][1] + to : 0x80000000u, 0, kStreamed);
        } else {
#pragma unroll
            for (int u = 0; u < 2; u++)
                __builtin_amdgcn_raw_buffer_store_b128(
                    u32x4{half[u][0], half[u][1], half[u][2], half[u][3]}, r.rs,
                    (EPI == kRelu ? f : f + 16 * u) < p.features ? r.at[j][u] + to : 0x80000000u, 0, 0);
        }
    };
    // (the tile before this one, of which the rows are still to go out)
    f32x4 old[LATER ? WF : 1][LATER ? WT : 1];
    Rows pending;
    if (LATER) {
        pending.rs = __builtin_amdgcn_make_buffer_rsrc((void *)p.x_scale, 0, 0, kRsrcFlags);
        pending.f0 = 0, pending.scales = scales_mem[0][wave];
#pragma unroll
        for (int j = 0; j < WT; j++) pending.xs[j] = pending.s_out[j] = 0.f, pending.at[j][0] = pending.at[j][1] = 0;
#pragma unroll
        for (int i = 0; i < WF; i++)
#pragma unroll
            for (int j = 0; j < WT; j++) old[LATER ? i : 0][LATER ? j : 0] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int round = 0;; round++) {
        const Tile t = tile_of(round);
        if (!t.there) break;
        const int set = LATER ? round & 1 : 0;
        fetch_scales(t, scales0 + set * kScaleSet);
#pragma unroll
        for (int i = 0; i < WF; i++)
#pragma unroll
            for (int j = 0; j < WT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        uint32_t before = 0;
        auto none = [](int) {};
        auto advance_buffers = [&](uint32_t later) { before = now, now = later; };
        if constexpr (LATER) {
            // Stores of a step, two tokens' of two tiles of features: behind its requests, so that the waits of
            // this step and of the next leave them in flight, and those of the one after do not.
            constexpr int kPut = 4;
            static_assert(WF == 8 && WT == 4, "eight steps");
            auto step = [&](auto first, auto last, auto flying, auto out) {
                const uint32_t later = after(now);
                compute(tiles + now, tiles + later, now, before, first, last,
                        [&]() {
                            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier"
                                         ::"n"(kFlying + decltype(flying)::value) : "memory");
                        },
                        out);
                advance_buffers(later);
            };
            constexpr std::true_type yes{};
            constexpr std::false_type no{};
            step(yes, no, std::integral_constant<int, kScaleLoads>{}, none);
            auto later_step = [&](auto group) {
                constexpr int k = decltype(group)::value, pair = k / 2, j0 = k % 2 * 2;
                const Features w = features_of(pending, pair);
                step(no, no, std::integral_constant<int, kPut + (k == 0 ? kScaleLoads : kPut)>{}, [&](int j) {
                    pair_out(pending, w, pair, j0 + j, old[2 * pair][j0 + j], old[2 * pair + 1][j0 + j], nullptr);
                });
            };
            later_step(std::integral_constant<int, 0>{});
            later_step(std::integral_constant<int, 1>{});
            later_step(std::integral_constant<int, 2>{});
            later_step(std::integral_constant<int, 3>{});
            later_step(std::integral_constant<int, 4>{});
            later_step(std::integral_constant<int, 5>{});
            later_step(std::integral_constant<int, 6>{});
            later_step(std::integral_constant<int, 7>{});
            // (the wait of the step behind them leaves the last one's stores in flight, or waits for them)
            for (int s = kLaterSteps; s < steps - 1; s++) step(no, no, std::integral_constant<int, 0>{}, none);
            step(no, yes, std::integral_constant<int, 0>{}, none);
            pending = rows_of(t, scales_mem[set][wave]);
#pragma unroll
            for (int i = 0; i < WF; i++)
#pragma unroll
                for (int j = 0; j < WT; j++) old[LATER ? i : 0][LATER ? j : 0] = acc[i][j];
        } else {
            auto step = [&](int s, auto first, auto last) {
                // The next step's rows have landed (in flight: those of the steps after it and, where
                // these steps were all requested before the rows of the tile before went out, those
                // rows and this tile's scales), and every wavefront has what it needs of this
                // step's buffer.
                const bool rows_fly = round > 0 && s < STAGES - 1 && steps >= STAGES;
                auto wait = [&]() {
                    constexpr int kMost = kFlying + (kAdds && decltype(last)::value ? 2 * WT + (EPI == kNormed ? WT : 0) : 0),
                                  kMore = kMost + kStores + kScaleLoads < 63 ? kMost + kStores + kScaleLoads : 63;
                    if (rows_fly)
                        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kMore) : "memory");
                    else
                        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kMost) : "memory");
                };
                const uint32_t later = after(now);
                compute(tiles + now, tiles + later, now, before, first, last, wait, none);
                advance_buffers(later);
            };
            // (The first and the last step stand outside the loop: as one of three bodies inside it each left the
            // sums in registers of its own, and up to 124 moves a step brought them back together, waiting for the
            // matrix instructions: 40960 tokens, 512 -> 1536 213 us, 189 this way; 1352, 1024 -> 512 14.8 and 10.2.)
            step(0, std::true_type{}, std::false_type{});
            for (int s = 1; s < steps - 1; s++) step(s, std::false_type{}, std::false_type{});
            const __amdgpu_buffer_rsrc_t r_rs = __builtin_amdgcn_make_buffer_rsrc(
                (char *)(kAdds ? p.residual : p.bias) + (kAdds ? t.t0 * out_row : 0), 0,
                (uint32_t)t.nt * out_row, kRsrcFlags);
            const __amdgpu_buffer_rsrc_t stats_rs = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(EPI == kNormed ? (const void *)(p.stats + t.t0) : (const void *)p.bias), 0, EPI == kNormed ? (uint32_t)t.nt * 8u : 0u,
                kRsrcFlags);
            typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
            u32x2_t of_row[WT];              // (mean, r)
            // (residual rows a pair of feature tiles ahead, the first one under the last step: a wait for them then
            // leaves the stores in flight)
            u32x4 res[2][WT][2];
            auto residual = [&](int pair) {
                const int f = t.f0 + wf * (TF / 2) + 32 * pair;
#pragma unroll
                for (int j = 0; j < WT; j++)
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        res[pair % 2][j][u] = __builtin_amdgcn_raw_buffer_load_b128(
                            r_rs, f + 16 * u + 4 * g < p.features ? token_at(j) + 4u * f + 64u * u : 0x80000000u, 0, 0);
            };
            if (EPI == kNormed) {
#pragma unroll
                for (int j = 0; j < WT; j++)
                    of_row[j] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(
                                                                stats_rs, 8u * (uint32_t)(wt * (TN / 2) + 16 * j + ln), 0, 0));
            }
            if (kAdds) residual(0);
            step(steps - 1, std::false_type{}, std::true_type{});
            // (this tile's scales: seen to have landed by the steps' waits where there are enough of them)
            if (steps <= STAGES) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const Rows rows = rows_of(t, scales_mem[0][wave]);
#pragma unroll
            for (int pair = 0; pair < WF / 2; pair++) {
                const Features w = features_of(rows, pair);
                if (kAdds && pair + 1 < WF / 2) residual(pair + 1);
                if (EPI == kNormed) {
#pragma unroll
                    for (int u = 0; u < 2; u++) {
                        const int f = rows.f0 + 32 * pair + 16 * u + 4 * g;
                        const int from = f < p.features ? f : 0;
                        const float4 ga = p.gamma ? *(const float4 *)(p.gamma + from) : make_float4(1.f, 1.f, 1.f, 1.f);
                        const float4 be = p.beta ? *(const float4 *)(p.beta + from) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                        for (int j = 0; j < WT; j++) {
                            const float mean = __uint_as_float(of_row[j][0]), r = __uint_as_float(of_row[j][1]);
                            u32x4 &v = res[pair % 2][j][u];
                            v = u32x4{__float_as_uint(normed(__uint_as_float(v.x) - mean, r, ga.x, be.x)),
                                      __float_as_uint(normed(__uint_as_float(v.y) - mean, r, ga.y, be.y)),
                                      __float_as_uint(normed(__uint_as_float(v.z) - mean, r, ga.z, be.z)),
                                      __float_as_uint(normed(__uint_as_float(v.w) - mean, r, ga.w, be.w))};
                        }
                    }
                }
#pragma unroll
                for (int j = 0; j < WT; j++)
                    pair_out(rows, w, pair, j, acc[2 * pair][j], acc[2 * pair + 1][j], kAdds ? res[pair % 2][j] : nullptr);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    if constexpr (LATER) {
#pragma unroll
        for (int pair = 0; pair < WF / 2; pair++) {
            const Features w = features_of(pending, pair);
#pragma unroll
            for (int j = 0; j < WT; j++) pair_out(pending, w, pair, j, old[2 * pair][j], old[2 * pair + 1][j], nullptr);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the requests of a tile that is not there)
}

template <int TN, int TF, int STAGES, int PER_CU>
void launch_product(LinearArgs a, hipStream_t stream) {
    a.feature_tiles = (int32_t)((a.features + TF - 1) / TF);
    const int64_t token_tiles = (a.tokens + TN - 1) / TN;
    // (a multiple of the eight XCDs)
    const int64_t tiles = (token_tiles + 7) / 8 * a.feature_tiles;
    const dim3 grid((unsigned)(8 * std::min<int64_t>(tiles, 32 * PER_CU))), block(256);
    if constexpr (TN == 128) {
        if (a.k / kStep > kLaterSteps && tiles > 32 && !a.residual) {
            if (a.out_pieces)
                hipLaunchKernelGGL((linear_kernel<TN, TF, STAGES, kRelu, true>), grid, block, 0, stream, a);
            else
                hipLaunchKernelGGL((linear_kernel<TN, TF, STAGES, kPlain, true>), grid, block, 0, stream, a);
            return;
        }
    }
    if (a.out_pieces)
        hipLaunchKernelGGL((linear_kernel<TN, TF, STAGES, kRelu>), grid, block, 0, stream, a);
    else if (a.stats)
        hipLaunchKernelGGL((linear_kernel<TN, TF, STAGES, kNormed>), grid, block, 0, stream, a);
    else if (a.residual)
        hipLaunchKernelGGL((linear_kernel<TN, TF, STAGES, kResidual>), grid, block, 0, stream, a);
    else
        hipLaunchKernelGGL((linear_kernel<TN, TF, STAGES, kPlain>), grid, block, 0, stream, a);
}

// Which tile a product runs on.  A workgroup's k-step takes the time below (us; two workgroups on a
// CU: together, and one alone), a tile's rows out the third number, and the launch lasts as long as
// its busiest XCD of 32 CUs.  Measured (us, 128 x 256 / 64 x 128 / 64 x 64 / 32 x 64; the library's
// product is none of these):
//   40960 tokens, 512 -> 1536   171 / 193 / 224 / 291     1352 tokens, 1024 -> 512  35 / 14 / 10 / 10
//   40960 tokens, 512 -> 512     75 /  73 /  85 / 106     169 tokens, 1024 -> 256   34 / 13 / 9.6 / 8.0
//   40960 tokens, 1024 -> 512   132 / 152 / 178 / 235     169 tokens, 256 -> 768    14 / 5.8 / 4.6 / 4.4
//   12000 tokens, 256 -> 768     27 /  22 /  22 /  28     2700 tokens, 512 -> 1536  22 / 20 / 20 / 23
// On few tiles a step is the latency of its barrier, its LDS reads and its matrix instructions one
// after the other, so the smallest tile has the shortest; on many the large tile reads the least of
// the L2 and the LDS per matrix instruction (its rate there is 1.13 PFLOP/s of fp16 pieces, what a
// large library product reaches here: the clock under that load is part of the bound).
struct ProductTile {
    int tokens, features, per_cu;
    double step, step_alone, rows;
};
constexpr ProductTile kProductTiles[] = {
    {128, 256, 1, 1.22, 0.89, 4.8}, {64, 128, 2, 0.78, 0.27, 0.5}, {64, 64, 2, 0.47, 0.18, 0.0}, {32, 64, 2, 0.31, 0.13, 0.0}};
int product_tile(int64_t tokens, int64_t features, int64_t steps) {
    int best = 0;
    double least = 0;
    for (int i = 0; i < 4; i++) {
        const ProductTile &t = kProductTiles[i];
        const int64_t token_tiles = (tokens + t.tokens - 1) / t.tokens;
        const int64_t tiles = (token_tiles + 7) / 8 * ((features + t.features - 1) / t.features);
        const int64_t round = 32 * t.per_cu, left = tiles % round;
        const double us = (double)(tiles / round + (left > 32)) * ((double)steps * t.step + t.rows) +
                          (left > 0 && left <= 32 ? (double)steps * t.step_alone + t.rows : 0.);
        if (i == 0 || us < least) least = us, best = i;
    }
    return best;
}

int launched(const char *what) {
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return fail(FTC_ERR_HIP, "%s launch failed: %s", what, hipGetErrorString(err));
    return FTC_OK;
}
bool aligned(const void *p) { return (uintptr_t)p % 16 == 0; }

template <bool NORM>
int launch_rows(const float *x, const float *gamma, const float *beta, float eps, int64_t rows, int64_t cols,
                float *out, float *stats, void *pieces, float *scale, hipStream_t stream) {
    if (cols % kStep != 0 || cols > 256 * kMostQuads)
        return fail(FTC_ERR_UNSUPPORTED, "rows of %lld values", (long long)cols);
    if (!aligned(x) || !aligned(gamma) || !aligned(beta) || !aligned(out) || !aligned(pieces))
        return fail(FTC_ERR_INVALID, "rows must be 16-byte aligned");
    if (rows <= 0) return FTC_OK;
    if (rows >= kMostRows) return fail(FTC_ERR_UNSUPPORTED, "%lld rows", (long long)rows);
    const dim3 grid((unsigned)((rows + 3) / 4)), block(256);
#define FTC_ROWS(Q)                                                                                   \
    hipLaunchKernelGGL((rows_kernel<Q, NORM>), grid, block, 0, stream, x, gamma, beta, eps, rows, (int)cols, out, \
                       (float2 *)stats, (char *)pieces, scale)
    const int64_t quads = (cols + 255) / 256;
    if (quads <= 1) FTC_ROWS(1);
    else if (quads <= 2) FTC_ROWS(2);
    else if (quads <= 4) FTC_ROWS(4);
    else FTC_ROWS(16);
#undef FTC_ROWS
    return launched("row");
}

}  // namespace
}  // namespace ftc

using namespace ftc;

extern "C" {

int ftc_split_weights(const ftc_weight *weights, int32_t count, void *stream) {
    if (!weights || count < 1 || count > kMostWeights) return fail(FTC_ERR_INVALID, "1 to %d weights", kMostWeights);
    WeightList list;
    list.count = count;
    list.first[0] = 0;
    for (int i = 0; i < count; i++) {
        const ftc_weight &w = weights[i];
        if (!w.w || !w.pieces || !w.scale || !w.bias_out || !w.norm || !aligned(w.w) || !aligned(w.pieces))
            return fail(FTC_ERR_INVALID, "weight %d: null or misaligned pointer", i);
        if (w.cols % kStep != 0 || w.cols <= 0 || w.cols > kMostColumns || w.rows <= 0 || w.rows > kMostColumns ||
            w.rows % 4 != 0)
            return fail(FTC_ERR_UNSUPPORTED, "weight %d: %lld x %lld", i, (long long)w.rows, (long long)w.cols);
        list.w[i] = w.w, list.bias[i] = w.bias, list.cols[i] = (int32_t)w.cols;
        list.pieces[i] = (char *)w.pieces, list.scale[i] = w.scale;
        list.bias_out[i] = w.bias_out, list.norm[i] = w.norm;
        list.first[i + 1] = list.first[i] + (int32_t)w.rows;
    }
    hipLaunchKernelGGL(split_weights_kernel, dim3((unsigned)((list.first[count] + 3) / 4)), dim3(256), 0,
                       (hipStream_t)stream, list);
    return launched("weight");
}

int ftc_split_rows(const float *x, int64_t rows, int64_t cols, void *pieces, float *scale, void *stream) {
    if (!x || !pieces || !scale) return fail(FTC_ERR_INVALID, "null pointer");
    return launch_rows<false>(x, nullptr, nullptr, 0.f, rows, cols, nullptr, nullptr, pieces, scale, (hipStream_t)stream);
}

int ftc_layer_norm_split(const float *x, const float *gamma, const float *beta, float eps, int64_t rows,
                         int64_t cols, float *out, void *pieces, float *scale, void *stream) {
    if (!x || !out || (pieces && !scale)) return fail(FTC_ERR_INVALID, "null pointer");
    return launch_rows<true>(x, gamma, beta, eps, rows, cols, out, nullptr, pieces, scale, (hipStream_t)stream);
}

int ftc_layer_norm_stats_split(const float *x, const float *gamma, const float *beta, float eps, int64_t rows,
                               int64_t cols, float *stats, void *pieces, float *scale, void *stream) {
    if (!x || !stats || !pieces || !scale) return fail(FTC_ERR_INVALID, "null pointer");
    if (!aligned(stats)) return fail(FTC_ERR_INVALID, "rows must be 16-byte aligned");
    return launch_rows<true>(x, gamma, beta, eps, rows, cols, nullptr, stats, pieces, scale, (hipStream_t)stream);
}

static int product(const void *x, const float *x_scale, int64_t tokens, const void *w, const float *w_scale,
                   const float *bias, const float *w_norm, int64_t features, int64_t k, const float *residual,
                   const float *stats, const float *gamma, const float *beta, float *out, void *relu_pieces,
                   float *relu_scale, void *stream) {
    if (!x || !x_scale || !w || !w_scale || !bias || (!out && !relu_pieces))
        return fail(FTC_ERR_INVALID, "null pointer");
    if (relu_pieces && (!relu_scale || !w_norm || residual || out))
        return fail(FTC_ERR_INVALID, "relu rows leave in pieces, with a scale and without a residual");
    if (!aligned(x) || !aligned(w) || !aligned(w_scale) || !aligned(bias) || !aligned(residual) || !aligned(out) ||
        !aligned(relu_pieces) || !aligned(stats) || !aligned(gamma) || !aligned(beta))
        return fail(FTC_ERR_INVALID, "rows must be 16-byte aligned");
    if (k % kStep != 0 || k < 2 * kStep || k > kMostColumns || features % 4 != 0 || features <= 0 ||
        features > kMostColumns || (relu_pieces && features % kStep != 0))
        return fail(FTC_ERR_UNSUPPORTED, "a product of %lld columns and %lld features", (long long)k, (long long)features);
    if (tokens <= 0) return FTC_OK;
    LinearArgs a;
    a.x = (const char *)x, a.w = (const char *)w, a.x_scale = x_scale, a.w_scale = w_scale, a.bias = bias;
    a.w_norm = w_norm, a.residual = residual, a.stats = (const float2 *)stats, a.gamma = gamma, a.beta = beta, a.out = out, a.out_pieces = (char *)relu_pieces;
    a.out_scale = relu_scale, a.tokens = tokens, a.features = (int32_t)features, a.k = (int32_t)k;
    a.streamed = 4 * tokens * (k + (residual ? 2 : 1) * features) >= kStreamedBytes;
    const hipStream_t on = (hipStream_t)stream;
    switch (product_tile(tokens, features, k / kStep)) {
    case 0: launch_product<128, 256, 3, 1>(a, on); break;
    case 1: launch_product<64, 128, 3, 2>(a, on); break;
    case 2: launch_product<64, 64, 4, 2>(a, on); break;
    default: launch_product<32, 64, 4, 2>(a, on); break;
    }
    if (relu_pieces) {
        const dim3 cuts((unsigned)((tokens + 4 * kCutRows - 1) / (4 * kCutRows)));
        hipLaunchKernelGGL(cut_rows_kernel, cuts, dim3(256), 0, on, a.out_pieces, relu_scale, tokens,
                           (int)features);
    }
    return launched("product");
}

int ftc_linear_split(const void *x, const float *x_scale, int64_t tokens, const void *w, const float *w_scale,
                     const float *bias, const float *w_norm, int64_t features, int64_t k,
                     const float *residual, float *out, void *relu_pieces, float *relu_scale, void *stream) {
    return product(x, x_scale, tokens, w, w_scale, bias, w_norm, features, k, residual, nullptr, nullptr, nullptr, out,
                   relu_pieces, relu_scale, stream);
}

int ftc_linear_split_normed(const void *x, const float *x_scale, int64_t tokens, const void *w, const float *w_scale,
                            const float *bias, int64_t features, int64_t k, const float *rows, const float *stats,
                            const float *gamma, const float *beta, float *out, void *stream) {
    if (!rows || !stats || !out) return fail(FTC_ERR_INVALID, "null pointer");
    return product(x, x_scale, tokens, w, w_scale, bias, nullptr, features, k, rows, stats, gamma, beta, out, nullptr,
                   nullptr, stream);
}

}  // extern "C"
