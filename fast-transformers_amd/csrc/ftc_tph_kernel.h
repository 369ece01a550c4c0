// Chain-parallel form of the MFMA causal scan for gfx950 on the fp16 matrix path: fp32 rows, states of
// up to 64 x 64 per workgroup (output columns beyond 64 have a workgroup of their own, widths that do
// not fill the block are clipped).
//
//   out[c, l, f] = sum_{j <= l} (a[c,l,:] . b[c,j,:]) * v[c,j,f]      (REV: j >= l)
//
// Division of labour, chunking, LDS tiles, swizzles, segments and the exchange of segment
// sums are those of ftc_tp_kernel.h (one workgroup walks one chain; four consumer wavefronts
// hold the state as slabs of 16 columns and share the chunk product Pt through LDS; producer
// wavefronts -- eight here, in two groups of four that take positions in turn, two quads of
// every operand per lane -- fetch rows four chunks ahead and cut them into piece tiles).  What differs is the arithmetic that
// stands for an fp32 product:
//
//  * Every fp32 value x is scaled by a power of two and cut into TWO fp16 pieces, both rounded
//    to nearest: hi = fp16(x s), lo = fp16(x s - hi).  hi + lo carries 22 significand bits of
//    x s as long as |x s| >= 2^-3 (below that the absolute error stays under 2^-25), and
//    |x s| < 2^16 must hold.  A product is the sum of THREE piece products (lo hi, hi lo,
//    hi hi; lo lo is below 2^-22 of the product) on v_mfma_f32_16x16x32_f16, each exact in the
//    fp32 accumulator: half the matrix instructions, two thirds of the LDS traffic and about
//    a third of the vector instructions of three bf16 pieces, with results as close to
//    float64 as those (the reference's own fp32 order is further away than either).
//  * The scales.  Rows are scaled chunk by chunk by powers of two, 2^(4 - e) with 2^e a
//    ceiling above every magnitude concerned: for b and v, whose products add up in the
//    state, every value of that operand met so far in the walk (a ceiling that only rises);
//    for a, the values of the chunk alone.  Scaled values therefore stay below 16, values
//    down to 2^-7 of the ceiling keep 22 bits, and the error of smaller ones is below 2^-29 of
//    the ceiling.  A ceiling is one for all columns and for the 32 rows of a chunk: where columns,
//    or rows of one chunk, differ by more than 2^7, the small ones lose bits that fp32 sums
//    would keep (2^-20 beside 1: off by up to 8e-2 of their own size).  Wider states, the fused
//    attention and odd widths whose copies run elsewhere stay on kernels that hold every fp32
//    value exactly for that.  The ceilings come about without a
//    pass of their own: while they cut position k of the walk, the producers look at the rows
//    of position k + 1, which they already hold in registers, and enter what they find in
//    that position's slot in LDS with atomic maxima (for b and v only when a value reaches the
//    running ceiling: rare after the first chunks; for a one word per wavefront and
//    position); after the
//    workgroup barrier all twelve wavefronts read the slot.  All of them thus know the same
//    three exponents for every position, and they depend on the rows alone: however a chain
//    is cut into segments, the results are the same bit for bit (as long as the state stays
//    below 2^14 units, s = 0; beyond that the chunk where s rises depends on the cut, and
//    results agree to the rounding of the state's pieces, 2^-22).
//  * The state is kept in the units of the scaled rows (2^(e_b + e_v - 8)); when a ceiling
//    rises it is rescaled (exactly).  It is cut into pieces with one more power of two,
//    2^-s, chosen so that no element leaves fp16's range: every third chunk s rises if an
//    element of the state exceeds 2^(14 + s) (a chunk adds at most 2^13: three more chunks
//    stay below 2^14 + 3 x 2^13 < 65504).  As long as s = 0, the rule, the cut is plain
//    (one packed conversion per pair for the high pieces).  The chunk product needs no scale:
//    |Pt| <= 64 * 16 * 16 = 2^14.
//  * Ot = (S^T a^T) 2^s + v^T Pt is summed in the units of the chunk and leaves the
//    accumulator through one v_ldexp_f32 per value.
#pragma once
#include <type_traits>

#include "ftc_tp_kernel.h"

namespace ftc {
namespace mfma {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x4 mfma16h(const Frag &a, const Frag &b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// Four fp32 values times a power of two -> packed fp16 pieces (x0, x2 in the low halves), all
// rounded to nearest even.  v_fma_mix{lo,hi}_f16 computes fma(x, s, c) in fp32 (exact here:
// x s is exact, and so is the remainder of a rounding) and rounds once to fp16; the third
// operand is the fp16 hi piece, read from the half that op_sel names and negated.  The two
// pairs are cut in turn, so that no instruction reads (or completes) a half-written register
// right after the instruction that wrote it: that costs a wait state each time.
__device__ __forceinline__ void cut_quad_f16(float x0, float x1, float x2, float x3, float s,
                                             uint32_t &h01, uint32_t &h23, uint32_t &l01,
                                             uint32_t &l23) {
    asm("v_fma_mixlo_f16 %0, %4, %8, 0\n\t"
        "v_fma_mixlo_f16 %1, %6, %8, 0\n\t"
        "v_fma_mixhi_f16 %0, %5, %8, 0\n\t"
        "v_fma_mixhi_f16 %1, %7, %8, 0\n\t"
        "v_fma_mixlo_f16 %2, %4, %8, -%0 op_sel:[0,0,0] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %3, %6, %8, -%1 op_sel:[0,0,0] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %2, %5, %8, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %3, %7, %8, -%1 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
        : "=&v"(h01), "=&v"(h23), "=&v"(l01), "=&v"(l23)
        : "v"(x0), "v"(x1), "v"(x2), "v"(x3), "v"(s));
}
// the same without a scale: one packed conversion per pair for the hi pieces
__device__ __forceinline__ void cut_quad_f16_unscaled(float x0, float x1, float x2, float x3,
                                                      uint32_t &h01, uint32_t &h23, uint32_t &l01,
                                                      uint32_t &l23) {
    asm("v_cvt_pk_f16_f32 %0, %4, %5\n\t"
        "v_cvt_pk_f16_f32 %1, %6, %7\n\t"
        "v_fma_mixlo_f16 %2, %4, 1.0, -%0 op_sel:[0,0,0] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixlo_f16 %3, %6, 1.0, -%1 op_sel:[0,0,0] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %2, %5, 1.0, -%0 op_sel:[0,0,1] op_sel_hi:[0,0,1]\n\t"
        "v_fma_mixhi_f16 %3, %7, 1.0, -%1 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
        : "=&v"(h01), "=&v"(h23), "=&v"(l01), "=&v"(l23)
        : "v"(x0), "v"(x1), "v"(x2), "v"(x3));
}
// Four consecutive fp32 values of a row -> 8 bytes of each of the two piece tiles.
__device__ __forceinline__ void cut_quad_to_lds(const u32x4 raw, float s, lds_char *tile,
                                                int piece_bytes, int addr) {
    uint32_t h0, l0, h1, l1;
    cut_quad_f16(__uint_as_float(raw.x), __uint_as_float(raw.y), __uint_as_float(raw.z),
                 __uint_as_float(raw.w), s, h0, h1, l0, l1);
    const u32x2 wh = {h0, h1}, wl = {l0, l1};
    *(lds_vec2 *)(tile + addr) = wh;
    *(lds_vec2 *)(tile + piece_bytes + addr) = wl;
}
__device__ __forceinline__ float max_abs4(const u32x4 raw, float m) {
    m = fmaxf(fmaxf(fabsf(__uint_as_float(raw.x)), fabsf(__uint_as_float(raw.y))), m);
    return fmaxf(fmaxf(fabsf(__uint_as_float(raw.z)), fabsf(__uint_as_float(raw.w))), m);
}

// Exponents travel as E = e + 128 with e clamped to -99 .. 120 (E = 29 .. 248), where 2^e is
// the ceiling: every value met so far is below it.  E = 28: nothing but zeros so far.  A state
// that comes in from elsewhere (another segment, the caller) is kept in units that the rows'
// ceilings set, so zeros count as 2^-40 there: with units of 2^-200 a state of ones would leave
// the range of fp32.
constexpr uint32_t kExpFloor = 28, kExpCeil = 248, kExpOfZeros = 88;
// The running ceilings of b and v travel as words that order like the ceilings and whose low half
// is the exponent to count with: E << 16 | E, and for zeros 0 << 16 | 88.
__device__ __forceinline__ constexpr uint32_t ceiling_word(uint32_t E) {
    return E <= kExpFloor ? kExpOfZeros : E << 16 | E;
}
__device__ __forceinline__ float pow2_field(int field) {  // 2^(field - 127), field clamped
    return __uint_as_float((uint32_t)max(1, min(254, field)) << 23);
}
// wave-uniform integer maxima and minima on the scalar unit (written out: the compiler would
// merge them into three-operand vector instructions)
__device__ __forceinline__ uint32_t scalar_max(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("s_max_u32 %0, %1, %2" : "=s"(r) : "s"(a), "s"(b) : "scc");
    return r;
}
__device__ __forceinline__ uint32_t scalar_min(uint32_t a, uint32_t b) {
    uint32_t r;
    asm("s_min_u32 %0, %1, %2" : "=s"(r) : "s"(a), "s"(b) : "scc");
    return r;
}
// the ceiling exponent of a non-negative float, given as its bits in a scalar register (inf and
// NaN: the largest)
__device__ __forceinline__ uint32_t ceiling_of(uint32_t bits) {
    const uint32_t be = (bits >> 23) & 0xffu;  // the value is below 2^(be - 126)
    return scalar_max(kExpFloor, scalar_min(kExpCeil, be + 2u));
}
// The largest of a non-negative float over the wavefront (wave-uniform): four steps inside
// the rows of 16 lanes on the data-parallel path, then one lane of every row.
// (non-negative floats order like their bit patterns: an integer maximum needs no
// canonicalising copy of the lane it reads across, and folds into one instruction)
template <int CTRL>
__device__ __forceinline__ uint32_t max_with_dpp(uint32_t x) {
    return max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true));
}
// ... over each row of 16 lanes (every lane of a row gets the row's maximum)
__device__ __forceinline__ uint32_t row_max_bits(float m) {
    uint32_t b = __float_as_uint(m);
    b = max_with_dpp<0xb1>(b);   // quad_perm [1, 0, 3, 2]
    b = max_with_dpp<0x4e>(b);   // quad_perm [2, 3, 0, 1]
    b = max_with_dpp<0x141>(b);  // row_half_mirror
    b = max_with_dpp<0x140>(b);  // row_mirror
    return b;
}
__device__ __forceinline__ uint32_t wave_max(float m) {  // (the bits of the largest value)
    const uint32_t b = row_max_bits(m);
    return scalar_max(scalar_max((uint32_t)__builtin_amdgcn_readlane((int)b, 0),
                                 (uint32_t)__builtin_amdgcn_readlane((int)b, 16)),
                      scalar_max((uint32_t)__builtin_amdgcn_readlane((int)b, 32),
                                 (uint32_t)__builtin_amdgcn_readlane((int)b, 48)));
}

// The running ceilings of a, b and v as one wavefront knows them (wave-uniform).
struct Ceilings {
    uint32_t Ea, Wb, Wv;
    __device__ __forceinline__ int Eb() const { return (int)(Wb & 0xffffu); }
    __device__ __forceinline__ int Ev() const { return (int)(Wv & 0xffffu); }
    __device__ __forceinline__ float scale_a() const { return pow2_field(259 - (int)Ea); }
    __device__ __forceinline__ float scale_b() const { return pow2_field(259 - Eb()); }
    __device__ __forceinline__ float scale_v() const { return pow2_field(259 - Ev()); }
    // exponent of the state's units, and of a chunk's output units (a x state)
    __device__ __forceinline__ int state_exp() const { return (int)((Wb + Wv) & 0xffffu) - 264; }
    __device__ __forceinline__ int out_exp() const { return (int)(Ea + ((Wb + Wv) & 0xffffu)) - 396; }
};
typedef __attribute__((address_space(3))) uint32_t lds_u32_t;
typedef __attribute__((address_space(3))) f32x4 lds_fvec4;
// The slot of a position is that of its LDS buffer: words (a, b, v, unused).  The words of b
// and v hold ceilings that only ever rise (a stale one is harmless: it is below the running
// ceiling that every wavefront carries).  The word of a holds the ceiling of the rows of that
// one position, tagged with the position's number in the upper 24 bits, so that what the
// slot held three positions ago is always smaller and needs no clearing.
__device__ __forceinline__ void read_slot(const lds_u32_t *slots, int k, Ceilings &c) {
    const u32x4 s = *(const lds_vec4 *)(slots + 4 * k);
    c.Ea = max(kExpFloor, (uint32_t)__builtin_amdgcn_readfirstlane(s.x) & 0xffu);
    c.Wb = max(c.Wb, (uint32_t)__builtin_amdgcn_readfirstlane(s.y));
    c.Wv = max(c.Wv, (uint32_t)__builtin_amdgcn_readfirstlane(s.z));
}
// Lane maxima of the rows of position `pos` (slot k) against the ceilings of the position
// before it.  a: every row of 16 lanes enters the ceiling of its own values (one lane per row:
// four atomics on one word per wavefront, no trip through scalar registers).  b, v: whoever
// finds a value at or above the running ceiling raises the slot.
__device__ __forceinline__ void raise_slot(lds_u32_t *slots, int k, int pos, const Ceilings &c,
                                           float ma, float mb, float mv, int lane) {
    lds_u32_t *const s = slots + 4 * k;
    const uint32_t ea = ceiling_of(wave_max(ma));
    if (lane == 0)
        __hip_atomic_fetch_max(s + 0, ((uint32_t)(pos + 1) << 8) | ea, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
    // (after nothing but zeros: every normal number is at or above 2^-126)
    const bool over = mb >= pow2_field((int)(c.Wb >> 16) - 1) || mv >= pow2_field((int)(c.Wv >> 16) - 1);
    if (__builtin_amdgcn_ballot_w64(over) != 0) {
        auto word_of = [](uint32_t bits) -> uint32_t {
            return ceiling_word(bits == 0 ? kExpFloor : scalar_max(kExpFloor + 1u, ceiling_of(bits)));
        };
        const uint32_t wb = word_of(wave_max(mb)), wv = word_of(wave_max(mv));
        if (lane == 0) {
            if (wb > c.Wb) __hip_atomic_fetch_max(s + 1, wb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (wv > c.Wv) __hip_atomic_fetch_max(s + 2, wv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    }
}

// GRAD: the gradients of the fused attention (equations in ftc_attention.hip) straight from its inputs:
// a scan's rows become phi(q), phi(k) [j < key_len] and gz = g / den as the producers first touch them, and
// the normaliser's share of a gradient, whose sums are prefix sums of rows weighted by w = 1 (for dq, which
// has the factor dd_l outside) or w_l = dd_l (for dk), is part of the walk.  Those are fp32 sums of fp32 rows: in
// two pieces under the ceiling of all columns, one of features 2^-14 beside the others was up to 1e-4 off, this way
// 8e-7.  The producers leave the weighted rows of a position in LDS as they look at it; two periods later, while
// they look at the next one, a lane takes eight rows of one column, adds what the other lanes' rows and the positions
// before add up to, and puts the sums back in place.  A consumer reads them with the rows that it stores, and
// the rows of q or k whose phi' multiplies the result.  What bounds a chunk of short chains is the producers' stream
// of instructions, of long ones the memory (backward, 80 chains, L=4096 / L=1000, us: 244 / 62; with the sums as
// products of two pieces in the consumers 245 / 60; made where a position is cut, not where the next but one is looked
// at, 261 / 64; dense copies of phi(q), phi(k), gz, the scans of those and a pass over their results 381 / 87).
enum GradRole { kGradQueries = 1, kGradKeys = 2, kGradValues = 3 };

// KS: groups of 32 rows of the state (1: a state of up to 32 rows, which skips the matrix
// instructions and fragment reads of the empty half).
// ODD: fp32 rows of any width on 4-byte boundaries.  The requests stay 16 bytes per lane (the
// hardware asks for 4-byte alignment and checks the descriptor's end word by word); a lane whose
// quad straddles the end of a row clears the words that belong to the next one when the
// look-ahead first touches them, and stores such a quad word by word.  Measured against dense
// zero-padded copies of the operands and results (8 x 16 chains, L=4096, 50 x 50, forward + backward):
// 940 -> 387 us; a chunk costs what one of 64 x 64 does.
template <int KS, bool ODD, bool GRAD>
__device__ __forceinline__ void scan_tph_body(uint32_t *__restrict__ ws_ptr, const ScanArgs &p) {
    static_assert(!GRAD || (KS == 2 && !ODD), "the gradients' form takes 64 x 64 states");
    constexpr int D = 64, F = 64;              // one block of state rows and of output columns
    constexpr int T = 256;                     // producer lanes at a position (four wavefronts of eight)
    constexpr int PF = kTpAhead;               // chunks requested ahead
    constexpr int RBA = D * 2, RBV = F * 2;    // bytes per row of an fp16 piece tile
    constexpr int kTileA = kChunk * RBA, kTileV = kChunk * RBV;
    // (b's second piece starts 256 bytes further on: 512-byte steps would let the compiler read both pieces' halves
    // in one instruction and put the fragments together with eight moves a chunk)
    constexpr int kTileB = kTileA + 256;
    constexpr int kOffB = 2 * kTileA, kOffV = kOffB + 2 * kTileB;
    constexpr int kBufBytes = kOffV + 2 * kTileV;
    constexpr int kTileP = kChunk * 64;        // Pt pieces: 32 rows (i) of 32 j
    constexpr int QA = D / 4, QV = F / 4;
    constexpr int LA = kChunk * QA / T, LV = kChunk * QV / T;
    static_assert(kChunk == 32 && T % QA == 0 && T % QV == 0, "shape");

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool producer = wave >= 4;
    const int w = wave & 3;  // (consumers)

    __shared__ __align__(16) char pieces_mem[3 * kBufBytes];
    __shared__ __align__(16) char pt_mem[3 * 2 * kTileP];
    __shared__ __align__(16) uint32_t slot_mem[16];
    // GRAD, for the rows in each of the three buffers: dd, and the rows of q or k that belong to the result's,
    // quad p of row r in slot p ^ (r mod 16)
    constexpr int kDdBytes = 4 * kChunk, kTileX = kChunk * F * 4;
    __shared__ __align__(16) char dd_mem[GRAD ? 3 * kDdBytes : 1];
    __shared__ __align__(16) char x_mem[GRAD ? 3 * kTileX : 1];
    // ... the weighted rows of position k in buffer k % 4 (written before barrier k - 1), then their running sums
    // (before barrier k + 1, read under the next chunk); quad p of row r in slot p ^ (r mod 16) ^ 4 (r / 16), where neither sixteen rows
    // of a quad nor sixteen columns of every eighth row meet in a bank
    __shared__ __align__(16) char sum_mem[GRAD ? 4 * kTileX : 1];
    auto sum_addr = [](int row, int quad) -> int { return row * F * 4 + 16 * (quad ^ (row % 16) ^ 4 * (row / 16)); };
    // ... and per column the sum over the positions before position k (k % 2), and over the first walk
    __shared__ float carry_mem[GRAD ? 2 : 1][GRAD ? F : 1], first_sum[GRAD ? F : 1];
    lds_char *const unit_pc = (lds_char *)pieces_mem;
    lds_char *const pt_pc = (lds_char *)pt_mem;
    lds_u32_t *const slots = (lds_u32_t *)slot_mem;
    lds_char *const dd_pc = (lds_char *)dd_mem, *const x_pc = (lds_char *)x_mem, *const sum_pc = (lds_char *)sum_mem;

    // ---- which chain (as in scan_tp_kernel) ----
    const uint32_t nseg = (uint32_t)p.nseg;
    const uint32_t chains = (uint32_t)p.waves_per_scan / nseg;
    const uint32_t per_chain = (uint32_t)p.total_waves / chains;  // scans x segments
    const uint32_t full = (chains / 8u) * 8u;
    uint32_t which, chain;
    if (blockIdx.x < full * per_chain) {
        const uint32_t grp = blockIdx.x / (8u * per_chain), r = blockIdx.x % (8u * per_chain);
        which = r / 8u;
        chain = grp * 8u + r % 8u;
    } else {
        const uint32_t t = blockIdx.x - full * per_chain;
        which = t / (chains - full);
        chain = full + t % (chains - full);
    }
    const uint32_t virt = which / nseg;
    const uint32_t scan_id = virt / (uint32_t)p.tp_fblocks;
    const int fb = (int)(virt % (uint32_t)p.tp_fblocks);
    const ScanOperands &op = p.scan[scan_id];
    const int Dw = op.d;                        // state rows: a and b are this wide
    const int fw = min(F, op.f - F * fb);       // output columns of this block
    const bool REV = op.rev != 0;
    const int n = (int)(chain / (uint32_t)p.H), h = (int)(chain % (uint32_t)p.H);
    const int rows = (int)p.L;
    const int total_chunks = (rows + kChunk - 1) / kChunk;
    const bool exchange = p.tp_exchange != 0 && nseg > 1;
    gu32 *const hdr = (gu32 *)ws_ptr;
    gu32 *const flags = hdr + kHdrWords;
    const uint32_t chain_id = virt * chains + chain;  // over all scans of the launch
    int seg = (int)(which % nseg);
    __shared__ uint32_t order_sh;
    if (exchange) {
        if (tid == 0)
            order_sh = __hip_atomic_fetch_add(flags + kMaxWaves + chain_id, 1u, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        seg = (int)__builtin_amdgcn_readfirstlane(order_sh);
        if ((uint32_t)seg >= nseg) {  // the control block was not zero when the launch began
            if (tid == 0)
                __hip_atomic_store(hdr + kHdrError, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
    }
    const int c0 = exchange ? seg * p.tp_seg_chunks : p.tp_start[seg];
    const int nchunks = min(total_chunks, exchange ? c0 + p.tp_seg_chunks : p.tp_start[seg + 1]);
    // the chunks walked for their state alone: so0 .. so0 + n1 - 1 (n1 a multiple of PF)
    const int so0 = exchange ? c0 : 0;
    const int n1 = exchange ? (seg + 1 < (int)nseg ? nchunks - c0 : 0) : c0;
    const int nwalk = n1 + (nchunks - c0);  // (position nwalk: a chunk of zeros)
    auto so_chunk = [&](int v) -> int { return exchange ? so0 + n1 - 1 - v : so0 + v; };
    auto walk_chunk = [&](int v) -> int { return v < n1 ? so_chunk(v) : c0 + (v - n1); };
    constexpr uint32_t kNoRow = 0x80000000u;  // an offset outside every descriptor
    auto chunk_row0 = [&](int c) -> int { return REV ? rows - kChunk * (c + 1) : kChunk * c; };
    if (tid < 16) slot_mem[tid] = 0;
    if (GRAD && tid < F) carry_mem[0][tid] = first_sum[tid] = 0.f;
    const int role = op.pad;  // GRAD
    const bool sums_rows = GRAD && role != kGradValues;
    // (GRAD: rows of k at or beyond the key length count as zero)
    const int key_rows = GRAD && p.key_len ? (int)max((int64_t)0, min((int64_t)rows, p.key_len[n])) : rows;
    Ceilings ce{kExpFloor, kExpOfZeros, kExpOfZeros};
    // Position k of the walk goes through LDS buffer (B0 + k) % 3 (pieces, Pt and slot), with B0
    // such that the first chunk of the walk proper has buffer 0: the consumers' loop over
    // those chunks is unrolled three times and addresses LDS with immediate offsets.
    const int B0 = (3 - n1 % 3) % 3;
    auto next_buf = [](int b) -> int { return b == 2 ? 0 : b + 1; };
#ifdef FTC_TIMELINE
    // tuning aid: 32 time stamps per workgroup behind the pointer that the host passes in
    // p.key_len (FTC_STAMP_PTR), written by lane 0 of consumer 0 (0 .. 15) and of producer 0
    // (16 .. 31) in the fifth chunk of the walk proper
    typedef __attribute__((address_space(1))) uint64_t gu64;
    const bool stamp_on = !GRAD && p.key_len != nullptr && w == 0 && lane == 0;
    gu64 *const stamp_base = (gu64 *)p.key_len + blockIdx.x * 32 + (producer ? 16 : 0);
    // ... and behind those, 64 stamps per workgroup: consumer 0 after the barrier of every chunk
    gu64 *const chunk_stamps = (gu64 *)p.key_len + gridDim.x * 32 + blockIdx.x * 64;
#endif
    FTC_STAMP(14);  // workgroup under way
#ifdef FTC_TIMELINE
    if (stamp_on && !producer) chunk_stamps[0] = __builtin_amdgcn_s_memrealtime();
    if (stamp_on && !producer) stamp_base[12] = __builtin_amdgcn_s_memtime();
#endif

    if (producer) {
        // =========================== producers ===========================
        const int ptid = w * 64 + lane;
        const uint32_t a_slb = (uint32_t)op.a_sl * 4, b_slb = (uint32_t)op.b_sl * 4,
                       v_slb = (uint32_t)op.v_sl * 4;
        const char *a_seg = (const char *)op.a + ((int64_t)n * op.a_sn + (int64_t)h * op.a_sh) * 4;
        const char *b_seg = (const char *)op.b + ((int64_t)n * op.b_sn + (int64_t)h * op.b_sh) * 4;
        const char *v_seg = (const char *)op.v +
                            ((int64_t)n * op.v_sn + (int64_t)h * op.v_sh + F * fb) * 4;
        const __amdgpu_buffer_rsrc_t a_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)a_seg, 0, (rows - 1) * a_slb + Dw * 4, kRsrcFlags);
        const __amdgpu_buffer_rsrc_t b_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)b_seg, 0, (rows - 1) * b_slb + Dw * 4, kRsrcFlags);
        const __amdgpu_buffer_rsrc_t v_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)v_seg, 0, (rows - 1) * v_slb + fw * 4, kRsrcFlags);
        // Two quads (four columns of one row) of every operand per lane and position, 16 rows
        // apart.  Widths that do not fill the block: a lane whose four columns lie beyond the width
        // asks outside the descriptor and cuts zeros (widths are multiples of 4).
        static_assert(LA == 2 && LV == 2 && QA == QV, "two quads per lane");
        const int prow = ptid / QA, pc4 = ptid % QA;
        const bool ab_in = GRAD || 4 * pc4 < Dw;
        const bool v_in = GRAD || 4 * pc4 < fw;
        const uint32_t a_goff = (uint32_t)prow * a_slb + 16u * pc4,
                       b_goff = (uint32_t)prow * b_slb + 16u * pc4,
                       v_goff = (uint32_t)prow * v_slb + 16u * pc4;
        int a_waddr[2], b_waddr[2], v_waddr[2];
#pragma unroll
        for (int q = 0; q < 2; q++)
            a_waddr[q] = TpSwizzle<RBA>::addr(prow + 16 * q, 8 * pc4),
            b_waddr[q] = TpSwizzle<RBA>::addr(prow + 16 * q, 2 * b_tile_column(4 * pc4)),
            v_waddr[q] = TpSwizzle<RBV>::addr(prow + 16 * q, 8 * pc4);
        // (ODD: which of a quad's words 1 .. 3 are the row's own)
        uint32_t ab_own[3], v_own[3];
#pragma unroll
        for (int e = 0; e < 3; e++) {
            ab_own[e] = 4 * pc4 + e + 1 < Dw ? 0xffffffffu : 0u;
            v_own[e] = 4 * pc4 + e + 1 < fw ? 0xffffffffu : 0u;
        }
        auto own_words = [&](u32x4 &r, const uint32_t (&m)[3]) {
            if (ODD) r = u32x4{r.x, r.y & m[0], r.z & m[1], r.w & m[2]};
        };
        struct Raw {
            u32x4 a[2], b[2], v[2];
            u32x4 x[2];               // GRAD: q or k
            uint32_t rden[2], dd[2];  // GRAD
        };
        const uint32_t x_slb = GRAD ? (uint32_t)op.s0_sd * 4 : 0u, x_goff = (uint32_t)prow * x_slb + 16u * pc4;
        const __amdgpu_buffer_rsrc_t x_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(sums_rows ? op.s0 + (int64_t)n * op.s0_sn + (int64_t)h * op.s0_sh : nullptr), 0,
            sums_rows ? (rows - 1) * x_slb + Dw * 4 : 0u, kRsrcFlags);
        // GRAD: 1 / den and dd of the row
        const __amdgpu_buffer_rsrc_t rden_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(GRAD ? p.row_rden + (int64_t)chain * rows : nullptr), 0, rows * 4, kRsrcFlags);
        const __amdgpu_buffer_rsrc_t dd_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(GRAD ? p.row_dd + (int64_t)chain * rows : nullptr), 0, rows * 4, kRsrcFlags);
        // Every request is made every time, whether its rows exist or not (a chunk walked for
        // its state alone needs no rows of a; positions past the end of the walk have no
        // rows): a request outside the descriptor costs no memory traffic and reads as zero,
        // and with a fixed number of requests per chunk the compiler can wait for the oldest
        // ones only.
        auto fetch = [&](Raw &r, int v) {  // v: position of the walk
            const int first = v < nwalk ? chunk_row0(walk_chunk(v)) : -2 * kChunk;
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int row0 = first + 16 * q, row0_x = v >= n1 ? row0 : -2 * kChunk;
                // (the sums wrap: a chunk that starts before the first row has its later rows in place)
                r.a[q] = __builtin_amdgcn_raw_buffer_load_b128(a_rs, ab_in ? a_goff + (uint32_t)row0_x * a_slb : kNoRow, 0, 0);
                r.b[q] = __builtin_amdgcn_raw_buffer_load_b128(b_rs, ab_in ? b_goff + (uint32_t)row0 * b_slb : kNoRow, 0, 0);
                r.v[q] = __builtin_amdgcn_raw_buffer_load_b128(v_rs, v_in ? v_goff + (uint32_t)row0 * v_slb : kNoRow, 0, 0);
                if constexpr (GRAD) {
                    r.x[q] = __builtin_amdgcn_raw_buffer_load_b128(x_rs, sums_rows ? x_goff + (uint32_t)row0_x * x_slb : kNoRow, 0, 0);
                    r.rden[q] = __builtin_amdgcn_raw_buffer_load_b32(rden_rs, 4u * (uint32_t)(prow + row0), 0, 0);
                    r.dd[q] = __builtin_amdgcn_raw_buffer_load_b32(dd_rs, 4u * (uint32_t)(prow + row0), 0, 0);
                }
            }
        };
        // GRAD: the rows as the scan takes them.  phi(0) is one, so rows that are not there are
        // cleared (a scalar test: most chunks lie wholly inside).
        auto feature = [&](u32x4 (&x)[2], int row0, int limit) {
#pragma unroll
            for (int q = 0; q < 2; q++) x[q] = feature_quad(x[q]);
            if (row0 < 0 || row0 + kChunk > limit) {
#pragma unroll
                for (int q = 0; q < 2; q++)
                    if ((uint32_t)(row0 + 16 * q + prow) >= (uint32_t)limit) x[q] = u32x4{0, 0, 0, 0};
            }
        };
        auto over_den = [](u32x4 (&x)[2], const uint32_t (&rden)[2]) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const float z = __uint_as_float(rden[q]);
                x[q] = u32x4{__float_as_uint(z * __uint_as_float(x[q].x)), __float_as_uint(z * __uint_as_float(x[q].y)),
                             __float_as_uint(z * __uint_as_float(x[q].z)), __float_as_uint(z * __uint_as_float(x[q].w))};
            }
        };
        auto as_taken = [&](Raw &r, int v) {  // v: position of the walk
            const int row0 = v < nwalk ? chunk_row0(walk_chunk(v)) : -2 * kChunk;
            if (role == kGradQueries) {
                over_den(r.a, r.rden);
                feature(r.v, row0, key_rows);
            } else if (role == kGradKeys) {
                over_den(r.b, r.rden);
                feature(r.v, row0, rows);
            } else {
                feature(r.a, v >= n1 ? row0 : -2 * kChunk, key_rows);
                feature(r.b, row0, rows);
                over_den(r.v, r.rden);
            }
        };
        // the largest magnitudes of the rows of a position against the ceilings (rows that
        // were not asked for read as zeros); k: that position's slot; pos % 4 == j
        auto look_ahead = [&](Raw &r, int k, int pos, int j) {
#pragma unroll
            for (int q = 0; q < 2; q++) own_words(r.a[q], ab_own), own_words(r.b[q], ab_own), own_words(r.v[q], v_own);
            if constexpr (GRAD) {
                as_taken(r, pos);
                if (sums_rows) {
#pragma unroll
                    for (int q = 0; q < 2; q++) {
                        const float u = role == kGradQueries ? 1.f : __uint_as_float(r.dd[q]);
                        *(lds_fvec4 *)(sum_pc + j * kTileX + sum_addr(prow + 16 * q, pc4)) =
                            f32x4{u * __uint_as_float(r.v[q].x), u * __uint_as_float(r.v[q].y),
                                  u * __uint_as_float(r.v[q].z), u * __uint_as_float(r.v[q].w)};
                    }
                }
            }
            raise_slot(slots, k, pos, ce, max_abs4(r.a[1], max_abs4(r.a[0], 0.f)), max_abs4(r.b[1], max_abs4(r.b[0], 0.f)),
                       max_abs4(r.v[1], max_abs4(r.v[0], 0.f)), lane);
        };
        // A position of the walk goes to its LDS buffer.  The first n1 positions only feed the
        // state: no piece of a.
        auto cut = [&](const Raw &r, int buf, bool own) {
            lds_char *const pc = unit_pc + buf * kBufBytes;
#pragma unroll
            for (int q = 0; q < 2; q++) {
                if (own) cut_quad_to_lds(r.a[q], ce.scale_a(), pc, kTileA, a_waddr[q]);
                cut_quad_to_lds(r.b[q], ce.scale_b(), pc + kOffB, kTileB, b_waddr[q]);
                cut_quad_to_lds(r.v[q], ce.scale_v(), pc + kOffV, kTileV, v_waddr[q]);
            }
            if (GRAD && sums_rows) {
#pragma unroll
                for (int q = 0; q < 2; q++)
                    if (own) *(lds_vec4 *)(x_pc + buf * kTileX + (prow + 16 * q) * F * 4 + 16 * (pc4 ^ prow)) = r.x[q];
                // (lane 0 of a row's sixteen for the first row, lane 1 for the second)
                if (pc4 < 2) *(lds_u32_t *)(dd_pc + buf * kDdBytes + 4 * (prow + 16 * pc4)) = pc4 == 0 ? r.dd[0] : r.dd[1];
            }
            if (!own) {
                asm volatile("" ::"v"(r.a[0]), "v"(r.a[1]));
                if constexpr (GRAD) asm volatile("" ::"v"(r.x[0]), "v"(r.x[1]));
            }
        };
        // GRAD: the running sums of position v in place of its weighted rows.  A wavefront has 16 columns, the
        // lanes of a column eight rows each, in the order of the walk.
        int sum_at[8];
        const int sum_col = 16 * w + lane % 16;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int at = 8 * (lane / 16) + t;
            sum_at[t] = sum_addr(REV ? kChunk - 1 - at : at, sum_col / 4) + 4 * (sum_col % 4);
        }
        auto weighted_rows = [&](float (&x)[8], int j) {  // (v % 4 == j)
#pragma unroll
            for (int t = 0; t < 8; t++) x[t] = *(const lds_f32 *)(sum_pc + j * kTileX + sum_at[t]);
        };
        auto add_rows = [&](float (&x)[8], int v, int j, bool own) {
            // (an exchange: the second walk starts anew, the consumers add what comes before)
            const float before = exchange && v == n1 ? 0.f : carry_mem[j % 2][sum_col];
#pragma unroll
            for (int t = 1; t < 8; t++) x[t] += x[t - 1];
            // (the sums of the even and the odd group of 16 lanes of each half, then of the two halves)
            const uint32_t bits = __float_as_uint(x[7]);
            const auto pair = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
            const float even = __uint_as_float(pair[0]), both = even + __uint_as_float(pair[1]);
            const auto half = __builtin_amdgcn_permlane32_swap(__float_as_uint(both), __float_as_uint(both), false, false);
            const float low = __uint_as_float(half[0]), all = low + __uint_as_float(half[1]);
            if (own) {
                const float ahead = before + ((lane & 32 ? low : 0.f) + (lane & 16 ? even : 0.f));
#pragma unroll
                for (int t = 0; t < 8; t++) *(lds_f32 *)(sum_pc + j * kTileX + sum_at[t]) = x[t] + ahead;
            }
            if (lane < 16) {
                carry_mem[(j + 1) % 2][sum_col] = before + all;
                if (v + 1 == n1) first_sum[sum_col] = before + all;
            }
        };
        // Barrier number k (k = 0: before the consumers' first position; k >= 1: in the
        // middle of position k - 1) finds position k cut and the slot of position k + 1
        // complete.  The last one finds a chunk of zeros.  The two groups of producers take the
        // positions in turn: before barrier k group k % 2 cuts position k, which it has looked at
        // before barrier k - 1, and the other group looks at position k + 1.
        static_assert(PF == 4, "two positions ahead for each of two groups");
        auto walk = [&](auto group_number) {
            constexpr int G = decltype(group_number)::value;
            Raw raw[2];
            fetch(raw[0], G), fetch(raw[1], G + 2);
            wg_barrier();  // the slots are zero
            if (G == 0) look_ahead(raw[0], B0, 0, 0);
            wg_barrier();  // the slot of position 0 is complete
            int buf = B0;
            auto period = [&](int v, int j, bool own, bool more) {  // v % 4 == j
                const bool stamped = own && v == n1 + 4;
                if (stamped) FTC_STAMP(0);
                read_slot(slots, buf, ce);
                if (j % 2 == G) {
                    cut(raw[j / 2], buf, own);
                    if (stamped) FTC_STAMP(2);
                    if (more) fetch(raw[j / 2], v + PF);
                } else {
                    float x[8];
                    if (sums_rows) weighted_rows(x, (j + 3) % 4);  // (they arrive during the look)
                    look_ahead(raw[(j + 1) % 4 / 2], next_buf(buf), v + 1, (j + 1) % 4);
                    if (sums_rows && v > 0) add_rows(x, v - 1, (j + 3) % 4, v > n1);
                    if (stamped) FTC_STAMP(1);
                }
                buf = next_buf(buf);
                if (stamped) FTC_STAMP(3);
                wg_barrier();
                __builtin_amdgcn_sched_barrier(0);  // one chunk at a time, in this order
                if (stamped) FTC_STAMP(4);
            };
            for (int v = 0; v < n1; v += PF) {
#pragma unroll
                for (int j = 0; j < PF; j++) period(v + j, j, false, true);
            }
            // (whole trips in the loop, the rest after it)
            int v = n1;
            for (; v + PF <= nwalk + 1; v += PF) {
#pragma unroll
                for (int j = 0; j < PF; j++) period(v + j, j, true, true);
            }
#pragma unroll
            for (int j = 0; j < PF - 1; j++) {
                if (v + j > nwalk) return;
                period(v + j, j, true, false);
            }
        };
        if (wave < 8)
            walk(std::integral_constant<int, 0>());
        else
            walk(std::integral_constant<int, 1>());
        return;
    }

    // =========================== consumers ===========================
    const int ln = lane & 15, g = lane >> 4;
    const uint32_t o_slb = (uint32_t)op.o_sl * 4;
    char *o_seg = (char *)op.out + ((int64_t)n * op.o_sn + (int64_t)h * op.o_sh + F * fb) * 4;
    const __amdgpu_buffer_rsrc_t o_rs =
        __builtin_amdgcn_make_buffer_rsrc((void *)o_seg, 0, (rows - 1) * o_slb + fw * 4, kRsrcFlags);
    // Pt quadrant of this wavefront (see scan_tp_kernel)
    const int jh = w == 0 ? 0 : w == 1 ? 1 : ((w == 2) == REV ? 1 : 0);
    const int ih = w == 0 ? 0 : w == 1 ? 1 : 1 - jh;
    int a_addr[2][2], b_addr[2][2];  // [local i tile][ks], [ks][u]
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
#pragma unroll
        for (int x = 0; x < 2; x++)
            a_addr[x][ks] = TpSwizzle<RBA>::addr(16 * (x ^ ih) + ln, 2 * (32 * ks + 8 * g));
#pragma unroll
        for (int u = 0; u < 2; u++)
            b_addr[ks][u] = kOffB + TpSwizzle<RBA>::addr(
                                        16 * jh + ln, 2 * b_tile_column(32 * ks + 8 * g + 4 * u));
    }
    int bt_addr[4][2], vt_addr[2];
#pragma unroll
    for (int u2 = 0; u2 < 2; u2++) {
        const int row = 8 * g + (ln >> 2) + 4 * u2;
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
            bt_addr[dt][u2] = kOffB + TpSwizzle<RBA>::addr(
                row, 2 * b_tile_column(32 * (dt / 2) + 4 * (dt % 2) + 8 * (ln & 3)));
        vt_addr[u2] = kOffV + TpSwizzle<RBV>::addr(row, 2 * (16 * w + 4 * (ln & 3)));
    }
    const int pt_waddr = TpSwizzle<64>::addr(16 * ih + ln, 2 * (16 * jh + 4 * g));
    int pt_raddr[2];
#pragma unroll
    for (int x = 0; x < 2; x++) pt_raddr[x] = TpSwizzle<64>::addr(16 * (x ^ ih) + ln, 16 * g);
    bool keep[4];  // (lane masks in scalar registers)
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int j = 16 * jh + 4 * g + r, i = 16 * ih + ln;
        keep[r] = REV ? (j >= i) : (j <= i);
    }
    // (columns beyond the width are not stored; ODD: a quad that straddles the width is stored
    // word by word, by the one wavefront that has such a quad)
    const int o_cols = fw - (16 * w + 4 * g);
    const bool o_in = o_cols >= (ODD ? 4 : 1);
    const bool o_straddles = ODD && fw % 4 != 0 && fw / 16 == w;
    uint32_t o_lane[2];
#pragma unroll
    for (int x = 0; x < 2; x++)
        o_lane[x] = (uint32_t)(16 * (x ^ ih) + ln) * o_slb + 4u * (16 * w + 4 * g) + (o_in ? 0u : kNoRow);
    constexpr int NT = 2 * KS;  // state tiles of 16 rows
    f32x4 S[4];                 // the slab, in units of 2^Ucur
#pragma unroll
    for (int dt = 0; dt < 4; dt++) S[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    int Ucur = 0;
    constexpr int kPa[3] = {1, 0, 0}, kPb[3] = {0, 1, 0};  // piece products, smallest first
    auto state_row = [&](int dt, int r) -> int { return 32 * (dt / 2) + 8 * g + 4 * (dt % 2) + r; };
    const bool st_in = 16 * w + ln < fw;
    auto scale_state = [&](int e) {  // S <- S 2^e
#pragma unroll
        for (int dt = 0; dt < NT; dt++)
#pragma unroll
            for (int r = 0; r < 4; r++) S[dt][r] = __builtin_amdgcn_ldexpf(S[dt][r], e);
    };
    auto add_caller_state = [&]() {  // in units of 2^Ucur
        const float *base =
            op.s0 + (int64_t)n * op.s0_sn + (int64_t)h * op.s0_sh + F * fb + 16 * w + ln;
#pragma unroll
        for (int dt = 0; dt < NT; dt++) {
            float x[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int d = state_row(dt, r);
                const bool in = st_in && d < Dw;
                x[r] = *(in ? base + (int64_t)d * op.s0_sd : op.s0);
                x[r] = in ? __builtin_amdgcn_ldexpf(x[r], -Ucur) : 0.f;
            }
            S[dt] += f32x4{x[0], x[1], x[2], x[3]};
        }
    };

    // GRAD with an exchange: the sums of the weighted rows before the segment, in this lane's four columns
    f32x4 Z = {0.f, 0.f, 0.f, 0.f};
    Frag af[2][2][2], bfr[2][2], bt[4][2], vf[2];
    // row-major fragment number i of a chunk (12: b for the quadrant first, then a)
    auto rm_frag = [&](const lds_char *pc, int i) {
        const int k = i % 2, ks = (i / 2) % 2, x = i / 4;
        if (ks >= KS) return;
        if (x == 0)
            bfr[ks][k] = lds_frag8x2(pc + k * kTileB + b_addr[ks][0], pc + k * kTileB + b_addr[ks][1]);
        else
            af[x - 1][ks][k] = lds_frag16(pc + k * kTileA + a_addr[x - 1][ks]);
    };
    // position-major fragment number i of a chunk (10: v first, then b^T tile by tile)
    auto tr_frag_into = [&](Frag (&btx)[4][2], Frag (&vfx)[2], const lds_char *pc, int i) {
        if (i >= 2 && (i - 2) / 4 >= KS) return;  // tiles 2, 3: rows 32 .. 63
        if (i < 2)
            vfx[i] = lds_frag_tr(pc + i * kTileV + vt_addr[0], pc + i * kTileV + vt_addr[1]);
        else {
            const int dt = (i - 2) / 2, k = (i - 2) % 2;
            btx[dt][k] = lds_frag_tr(pc + k * kTileB + bt_addr[dt][0], pc + k * kTileB + bt_addr[dt][1]);
        }
    };
    int buf = B0;  // LDS buffer of the chunk at hand
    wg_barrier();  // the slots are zero
    wg_barrier();  // the slot of position 0 is complete
    wg_barrier();  // barrier 0: position 0 is cut
    read_slot(slots, B0, ce);
    Ucur = ce.state_exp();
    if (!GRAD && op.s0 && !exchange) add_caller_state();
    if (n1 > 0) {
        // ---- the first n1 positions of the walk: state update only ----
        // The loop is skewed by one position: while the matrix instructions of position k - 1
        // run, the fragments of position k arrive in the other set of registers.
        int U_prev = Ucur;                 // units of the fragments about to be multiplied
        Frag bt2[4][2] = {}, vf2[2] = {};  // (the first round multiplies zeros)
        for (int c = 0; c < n1; c += PF) {
#pragma unroll
            for (int j = 0; j < PF; j++) {
                const lds_char *pc = unit_pc + buf * kBufBytes;
                read_slot(slots, buf, ce);  // the ceilings of position c + j
                if (U_prev != Ucur) {       // the ceilings rose: the state shrinks
                    scale_state(Ucur - U_prev);
                    Ucur = U_prev;
                }
#pragma unroll
                for (int i = 0; i < 12; i++) {
                    const bool rows_exist = (i % 4) / 2 < KS;
                    if (j % 2 == 0) {
                        if (rows_exist) S[i % 4] = mfma16h(bt2[i % 4][kPa[i / 4]], vf2[kPb[i / 4]], S[i % 4]);
                        if (i < 10) tr_frag_into(bt, vf, pc, i);
                    } else {
                        if (rows_exist) S[i % 4] = mfma16h(bt[i % 4][kPa[i / 4]], vf[kPb[i / 4]], S[i % 4]);
                        if (i < 10) tr_frag_into(bt2, vf2, pc, i);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                U_prev = ce.state_exp();
                buf = next_buf(buf);
                wg_barrier();
#ifdef FTC_TIMELINE
                if (stamp_on && c + j < 30) chunk_stamps[32 + c + j] = __builtin_amdgcn_s_memrealtime();
#endif
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the last of these positions (n1 is even: its fragments are in the second set)
        if (U_prev != Ucur) {
            scale_state(Ucur - U_prev);
            Ucur = U_prev;
        }
#pragma unroll
        for (int i = 0; i < 12; i++) {
            if ((i % 4) / 2 < KS) S[i % 4] = mfma16h(bt2[i % 4][kPa[i / 4]], vf2[kPb[i / 4]], S[i % 4]);
            if (!GRAD) rm_frag(unit_pc + buf * kBufBytes, i);  // our own first chunk is cut
            __builtin_amdgcn_sched_barrier(0);
        }
        read_slot(slots, buf, ce);  // the ceilings of our own first chunk
    } else if (!GRAD) {
#pragma unroll
        for (int i = 0; i < 12; i++) rm_frag(unit_pc, i);
    }
    if (exchange) {
        // ---- the sum of this segment's rows goes out, the state before the segment comes in ----
        const uint32_t total_units = (uint32_t)p.total_waves;
        gfloat *const sums = (gfloat *)(hdr + kControlBytes / 4);
        constexpr int DX = GRAD ? 2 : 1;  // (Z rides along in a tile of its own)
        // (four at a time need the registers of the fragments, and those read behind the exchange: 8 chains, L=512, which
        // exchange nothing, 15.04 -> 15.14 us)
        StateExchange<DX, 1, GRAD ? 1 : 2> xch(flags, sums, 4u * total_units,
                                (uint32_t)w * total_units + chain_id * nseg + (uint32_t)seg, seg,
                                (int)nseg, p.group, lane);
        f32x16 Sx[DX][1], X[DX][1];
        if (GRAD) {
            Sx[DX - 1][0] = f32x16{};
#pragma unroll
            for (int r = 0; r < 4; r++) Sx[DX - 1][0][r] = first_sum[16 * w + 4 * g + r];
        }
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                Sx[0][0][4 * dt + r] = dt < NT ? __builtin_amdgcn_ldexpf(S[dt][r], Ucur) : 0.f;
        if (n1 > 0) xch.publish_sum(Sx);
        xch.gather(Sx, X);
        if (xch.failed && lane == 0)
            __hip_atomic_store(hdr + kHdrError, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // the units of the first chunk of the second pass (its ceilings are already known)
        Ucur = ce.state_exp();
#pragma unroll
        for (int dt = 0; dt < NT; dt++)
#pragma unroll
            for (int r = 0; r < 4; r++) S[dt][r] = __builtin_amdgcn_ldexpf(X[0][0][4 * dt + r], -Ucur);
        if (GRAD) {
#pragma unroll
            for (int r = 0; r < 4; r++) Z[r] = X[DX - 1][0][r];
        }
        if (!GRAD && op.s0) add_caller_state();
    }
    if (GRAD) {  // (not before: two tiles are exchanged, and 48 registers of fragments beside them spilled)
#pragma unroll
        for (int i = 0; i < 12; i++) rm_frag(unit_pc, i);
    }
    // ---- the walk proper ----
    // `ce` holds the ceilings of the chunk at hand, Ucur the units of S.  dU < 0: the
    // state's units rise by -dU with this chunk (S is rescaled once all of it has been cut).
    int dU = Ucur - ce.state_exp();
    int s = 0;  // S is cut as S 2^(dU - s)
    auto lane_max_state = [&]() -> float {
        float m = 0.f;
#pragma unroll
        for (int dt = 0; dt < NT; dt++)
            m = fmaxf(fmaxf(fmaxf(fabsf(S[dt][0]), fabsf(S[dt][1])), fmaxf(fabsf(S[dt][2]), fabsf(S[dt][3]))), m);
        return m;
    };
    {
        if (dU != 0) {
            scale_state(dU);
            Ucur -= dU;
            dU = 0;
        }
        const float m = lane_max_state();
        while (s < 100 && __builtin_amdgcn_ballot_w64(m > pow2_field(127 + 14 + s)) != 0) s++;
    }
    float kappa = pow2_field(127 + dU - s);  // scale of the cut of S
    int s_cut = s;                            // ... and the s that went into it
    float mS = 0.f;                           // largest |S| seen while cutting
    Frag sf[2][2];
    // tile 2 ks + u of S_w -> words 2 u, 2 u + 1 of the fragments of k-step ks
    // (`track`: also note the largest magnitude.  One state in three is looked at, the one
    // cut for the chunks in LDS buffer 0: s then rises when an element exceeds 2^(14 + s)
    // units, three more chunks add at most 3 x 2^13, and 2^14 + 3 x 2^13 is below what fp16
    // holds.)
    auto cut_s = [&](int ks, int u, bool track) {
        const f32x4 x = S[2 * ks + u];
        if (track)
            mS = fmaxf(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))), mS);
        cut_quad_f16(x[0], x[1], x[2], x[3], kappa, sf[ks][0].w[2 * u], sf[ks][0].w[2 * u + 1], sf[ks][1].w[2 * u],
                     sf[ks][1].w[2 * u + 1]);
    };
    cut_s(0, 0, true);
    cut_s(0, 1, true);

    // Ot_w of the chunk before in the units of that chunk (exponent Xo), and where its rows
    // go (before the first chunk: nowhere)
    f32x4 O[2];
#pragma unroll
    for (int x = 0; x < 2; x++) O[x] = f32x4{0.f, 0.f, 0.f, 0.f};
    int Xo = 0;
    uint32_t o_off = (uint32_t)(rows + kChunk) * o_slb;  // (also beyond the end with kNoRow on top of it)
    int o_row0 = 0, o_buf = 0, o_sum = 0;  // GRAD
    auto store_rows = [&](int x) {
        float y0 = __builtin_amdgcn_ldexpf(O[x][0], Xo), y1 = __builtin_amdgcn_ldexpf(O[x][1], Xo),
              y2 = __builtin_amdgcn_ldexpf(O[x][2], Xo), y3 = __builtin_amdgcn_ldexpf(O[x][3], Xo);
        if (GRAD && sums_rows) {
            const int row = 16 * (x ^ ih) + ln;
            f32x4 slope = *(const lds_fvec4 *)(x_pc + o_buf * kTileX + row * F * 4 + 16 * ((4 * w + g) ^ ln));
#pragma unroll
            for (int r = 0; r < 4; r++)  // phi'(x); NaN: one (gz is NaN then)
                slope[r] = fminf(1.f, __builtin_amdgcn_exp2f(slope[r] * 1.44269502f));
            const f32x4 sum = *(const lds_fvec4 *)(sum_pc + o_sum + sum_addr(row, 4 * w + g)) + Z;
            const float dd = *(const lds_f32 *)(dd_pc + o_buf * kDdBytes + 4 * row), u = role == kGradQueries ? dd : 1.f;
            y0 = fmaf(u, sum[0], y0) * slope[0], y1 = fmaf(u, sum[1], y1) * slope[1];
            y2 = fmaf(u, sum[2], y2) * slope[2], y3 = fmaf(u, sum[3], y3) * slope[3];
            if (role == kGradKeys && o_row0 + kChunk > key_rows) {  // (rows beyond the key length)
                const bool live = o_row0 + row < key_rows;
                y0 = live ? y0 : 0.f, y1 = live ? y1 : 0.f, y2 = live ? y2 : 0.f, y3 = live ? y3 : 0.f;
            }
        }
        buffer_store_out(o_rs, o_off + o_lane[x], y0, y1, y2, y3, (float *)nullptr);
        if (o_straddles) {
            const uint32_t first = o_off + o_lane[x] - (o_in ? 0u : kNoRow);
            const bool some = o_cols < 4;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y0), o_rs, some && o_cols > 0 ? first : kNoRow, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y1), o_rs, some && o_cols > 1 ? first + 4u : kNoRow, 0, 0);
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y2), o_rs, some && o_cols > 2 ? first + 8u : kNoRow, 0, 0);
        }
    };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // One chunk, in LDS buffer B (a compile-time number, so that every LDS access of the body
    // has its buffer in the instruction's immediate offset).  Sums that end in one place are
    // chained through one accumulator, with other matrix instructions in between: Ot_w =
    // (S_w^T a^T) 2^s + v_w^T Pt needs no addition at all while s = 0, which is the rule.
    auto chunk_body = [&](int c, auto buffer_number) {
        constexpr int B = decltype(buffer_number)::value, BN = (B + 1) % 3;
        const lds_char *pc = unit_pc + B * kBufBytes;
        const lds_char *pn = unit_pc + BN * kBufBytes;
        lds_char *const ptc = pt_pc + B * (2 * kTileP);
        Frag pf[2][2];
        f32x4 P;  // (cleared by the first matrix instruction of its sum)
        if (c == c0 + 4) FTC_STAMP(0);
        __builtin_amdgcn_sched_barrier(0);
        // phase 1: (1) the quadrant in turn with (2b) Ot_w = S_w^T a^T for rows 0 .. 31 of
        // the state; underneath: the rows of the chunk before go out, tiles 2, 3 of S_w are
        // cut into pieces, the position-major reads
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int m = i % 3, ks = i / 3, x = i % 2, mo = i / 2;
            if (i == 0) store_rows(0);
            if (i == 1) store_rows(1);
            if (ks < KS) P = mfma16h(bfr[ks][kPa[m]], af[0][ks][kPb[m]], i == 0 ? zero : P);
            O[x] = mfma16h(sf[0][kPa[mo]], af[x][0][kPb[mo]], mo == 0 ? zero : O[x]);
            if ((i == 1 || i == 3) && KS > 1) cut_s(1, i / 2, B == 0);
            tr_frag_into(bt, vf, pc, i);
            if (!GRAD && i < 4) tr_frag_into(bt, vf, pc, 6 + i);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (c == c0 + 4) FTC_STAMP(1);
        // all of S is cut: it takes the units of this chunk, and s follows its size
        if (__builtin_expect(dU != 0, 0)) {
            scale_state(dU);
            mS = __builtin_amdgcn_ldexpf(mS, dU);
            s = max(0, s + min(dU, 0));
            Ucur -= dU;
        }
        if (B == 0) {
            while (s < 100 && __builtin_amdgcn_ballot_w64(mS > pow2_field(127 + 14 + s)) != 0) s++;
            mS = 0.f;
        }
        if (c == c0 + 4) FTC_STAMP(2);
        __builtin_amdgcn_sched_barrier(0);
        // phase 2: (2b) for rows 32 .. 63 in turn with (3) S_w += b^T v_w for tiles 0 and 1;
        // underneath: the quadrant is masked, cut and handed to the others
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int x = i % 2, m = i / 2;
            if (KS > 1) O[x] = mfma16h(sf[1][kPa[m]], af[x][1][kPb[m]], O[x]);
            if (GRAD && i >= 2) tr_frag_into(bt, vf, pc, 4 + i);  // (phase 1 has no registers for them)
            S[i % 2] = mfma16h(bt[i % 2][kPa[m]], vf[kPb[m]], S[i % 2]);
            if (i == 1) {
                uint32_t h0, l0, h1, l1;
#pragma unroll
                for (int r = 0; r < 4; r++) P[r] = keep[r] ? P[r] : 0.f;
                cut_quad_f16_unscaled(P[0], P[1], P[2], P[3], h0, h1, l0, l1);
                const u32x2 wh = {h0, h1}, wl = {l0, l1};
                *(lds_vec2 *)(ptc + pt_waddr) = wh;
                *(lds_vec2 *)(ptc + kTileP + pt_waddr) = wl;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (c == c0 + 4) FTC_STAMP(4);
        wg_barrier();
        if (c == c0 + 4) FTC_STAMP(5);
#ifdef FTC_TIMELINE
        if (stamp_on && c - c0 < 30) chunk_stamps[c - c0 + 1] = __builtin_amdgcn_s_memrealtime();
#endif
        // All of Pt is in LDS, the next chunk is cut and its slot complete.
        // phase 3: (3) for tiles 2 and 3, then (2a) Ot_w += v_w^T Pt; underneath: the next
        // chunk's row-major fragments are requested and tiles 0, 1 of S_w cut into pieces
#pragma unroll
        for (int x = 0; x < 2; x++)
#pragma unroll
            for (int k = 0; k < 2; k++) pf[x][k] = lds_frag16(ptc + k * kTileP + pt_raddr[x]);
        const int Xc = ce.out_exp();
        const u32x4 slot_next = *(const lds_vec4 *)(slots + 4 * BN);
        if (__builtin_expect(s_cut != 0, 0)) {  // (rare: the state has grown beyond 2^14 units)
            const float r_cut = pow2_field(127 + s_cut);
            O[0] *= r_cut;
            O[1] *= r_cut;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int m = i / 2;
            if (KS > 1) S[2 + i % 2] = mfma16h(bt[2 + i % 2][kPa[m]], vf[kPb[m]], S[2 + i % 2]);
            rm_frag(pn, 2 * i);
            rm_frag(pn, 2 * i + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        // the ceilings of the next chunk
        ce.Ea = max(kExpFloor, (uint32_t)__builtin_amdgcn_readfirstlane(slot_next.x) & 0xffu);
        ce.Wb = max(ce.Wb, (uint32_t)__builtin_amdgcn_readfirstlane(slot_next.y));
        ce.Wv = max(ce.Wv, (uint32_t)__builtin_amdgcn_readfirstlane(slot_next.z));
        // (dU > 0: small values after nothing but zeros; the state's units fall, so s rises)
        dU = Ucur - ce.state_exp();
        s += max(dU, 0);
        kappa = pow2_field(127 + dU - s);
        s_cut = s;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int x = i % 2, m = i / 2;
            O[x] = mfma16h(vf[kPa[m]], pf[x][kPb[m]], O[x]);
            if (i == 1 || i == 3) cut_s(0, i / 2, BN == 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        o_off = (uint32_t)chunk_row0(c) * o_slb;
        o_row0 = chunk_row0(c), o_buf = B, o_sum = (c - c0) % 4 * kTileX;  // (n1 is a multiple of 4)
        Xo = Xc;
        if (c == c0 + 4) FTC_STAMP(6);
    };
    {
        int c = c0;
        for (; c + 3 <= nchunks; c += 3) {
            chunk_body(c, std::integral_constant<int, 0>());
            chunk_body(c + 1, std::integral_constant<int, 1>());
            chunk_body(c + 2, std::integral_constant<int, 2>());
        }
        if (c < nchunks) chunk_body(c++, std::integral_constant<int, 0>());
        if (c < nchunks) chunk_body(c++, std::integral_constant<int, 1>());
    }
    store_rows(0);
    store_rows(1);
    FTC_STAMP(15);  // last rows on their way
#ifdef FTC_TIMELINE
    if (stamp_on) stamp_base[13] = __builtin_amdgcn_s_memtime();
#endif
    if (!GRAD && op.s_out && seg == (int)nseg - 1) {
        float *base =
            op.s_out + (int64_t)n * op.so_sn + (int64_t)h * op.so_sh + F * fb + 16 * w + ln;
#pragma unroll
        for (int dt = 0; dt < NT; dt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int d = state_row(dt, r);
                if (st_in && d < Dw) base[(int64_t)d * op.so_sd] = __builtin_amdgcn_ldexpf(S[dt][r], Ucur);
            }
    }
    // the last consumer of the launch leaves the control block zeroed
    if (exchange) {
        const uint32_t total_units = (uint32_t)p.total_waves;
        // (not where a consumer has gathered, so that others are waited for under the walk: all of them count then while
        // the last ones look at their flags; attention, 64 chains, L=1600 52.7 -> 54.9 us, 40, L=2000 44.6 -> 46.9)
        uint32_t done = 0;
        if (lane == 0)
            done = __hip_atomic_fetch_add(hdr + kHdrDone, 1u, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
        done = __builtin_amdgcn_readfirstlane(done);
        if (done == 4u * total_units - 1) {
            for (uint32_t i = lane; i < 4u * total_units; i += kWave)
                __hip_atomic_store(flags + i, kFlagEmpty, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            for (uint32_t i = lane; i < total_units / nseg; i += kWave)
                __hip_atomic_store(flags + kMaxWaves + i, 0u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            if (lane == 0)
                __hip_atomic_store(hdr + kHdrDone, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

template <int KS, bool ODD>
__global__ __launch_bounds__(768, 3) void scan_tph_kernel(uint32_t *__restrict__ ws_ptr, ScanArgs p) {
    scan_tph_body<KS, ODD, false>(ws_ptr, p);
}

}  // namespace mfma
}  // namespace ftc
