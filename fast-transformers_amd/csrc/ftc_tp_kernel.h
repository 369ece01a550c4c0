// Chain-parallel form of the MFMA causal scan for gfx950, states of up to 128 x 128, fp32 rows in three
// bf16 pieces and bf16 rows in one.  Described for fp32 rows and a 64 x 64 state; a state of more rows is walked in two blocks of
// 64 (ND = 2: two positions of the walk per chunk, each on its own 64 columns of a and b and
// its own rows of the slabs; their quadrants of Pt are added before the cut, the result rows
// are stored after the second, and both read one v tile), output columns beyond 64 have a
// workgroup of their own, and widths that do not fill the last block are clipped.
//
//   out[c, l, f] = sum_{j <= l} (a[c,l,:] . b[c,j,:]) * v[c,j,f]      (REV: j >= l)
//
// One workgroup walks one chain, chunk after chunk.  With enough chains a workgroup takes a
// whole chain and every row is read once; nothing is exchanged between workgroups and no
// workspace is touched.  With fewer, a chain is cut into segments, one workgroup each, and
// the state before a segment comes about in one of two ways:
//  * short chains: the workgroup first runs the state update alone -- step (3) below, a
//    third of the matrix work and no chunk product -- over the chunks before its own, so
//    that it starts from the same state, bit for bit, that a single walk would have reached
//    (later segments are made shorter, so that all workgroups of a chain finish together);
//  * long chains: it first runs the state update alone over its OWN chunks, publishes that
//    sum and adds up the sums of the segments before it (StateExchange, ftc_mfma_kernel.h).
// What makes a single chain fast enough is that the work of a chunk is spread over four
// matrix cores: the 64 x 64 state is held as four slabs of 16 columns, one per consumer
// wavefront (one per SIMD), and the 32 x 32 chunk product Pt is computed once, a quadrant
// per wavefront, and shared through LDS.
//
//  * Wavefronts 4..7 (producers) fetch the rows of a chunk, cut every fp32 value into its
//    three bf16 pieces and write them as row-major piece tiles into LDS, four chunks
//    ahead (as in ftc_wg_kernel.h).  Of the chunks that only feed the state they take rows
//    0 .. 15 of b and v; the consumers, who have little to do there, take rows 16 .. 31.
//  * Wavefronts 0..3 (consumers), v_mfma_f32_16x16x32_bf16 (A: row = lane % 16, B: column =
//    lane % 16, both with k-slots t = 0..7 of lane group g = lane / 16; accumulator: column
//    = lane % 16, rows 4 g + r).  Consumer w owns output columns 16 w .. 16 w + 15:
//      (1)  Pt quadrant (jh, ih) = b[16 jh ..] a[16 ih ..]^T over d, masked (the quadrant of
//           the fourth wavefront lies wholly beyond the causal mask: zeros), cut into
//           pieces and written to LDS as rows i with j contiguous;
//      (2b) Ot_w  = S_w^T a^T       16 f x 32 i, contraction over d;
//      (3)  S_w  += b^T v_w         64 d x 16 f, contraction over the chunk's positions j;
//           ((2b) of rows 0 .. 31 runs in turn with (1), of rows 32 .. 63 with (3): a sum
//           waits for its last product while the others go on)
//      -- barrier: all of Pt is in LDS --
//      (2a) Ot_w += v_w^T Pt        contraction over j;   Ot_w is stored under (1) of the
//           next chunk, when its last matrix instructions have long finished.
//    Row m of state tile dt = 2 ks + u stands for d = 32 ks + 8 (m / 4) + 4 u + m % 4 (the
//    b^T fragments of (3) are read in that column order), so that the accumulator registers
//    of S_w (column f = lane % 16, rows 4 g + r of tiles 2 ks and 2 ks + 1) are, as they
//    stand, the A operand of k-step ks of (2b) with k-slots d = 32 ks + 8 g + t -- the order
//    of a 16-byte read of a row of a or b, whose fragments serve (1) and (2b) alike.
//  * One workgroup barrier per chunk, after Pt is written.  The piece tiles rotate through
//    three LDS buffers and Pt through two (three where the loop is unrolled, tp_unrolled): when the barrier of chunk c falls, the producers
//    have cut chunk c + 1 (the consumers request its row-major fragments right away, under
//    (2a)) and go on to cut chunk c + 2 into the buffer of chunk c - 1, which nobody has
//    read since the barrier before.
#pragma once
#include <type_traits>

#include "ftc_wg_kernel.h"

namespace ftc {
namespace mfma {

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(const Frag &a, const Frag &b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// k-slots 0..3 from the 8 bytes at p0, 4..7 from those at p1
__device__ __forceinline__ Frag lds_frag8x2(const lds_char *p0, const lds_char *p1) {
    const u32x2 lo = *(const lds_vec2 *)p0;
    const u32x2 hi = *(const lds_vec2 *)p1;
    return Frag{{lo.x, lo.y, hi.x, hi.y}};
}

// XOR swizzle of this kernel's LDS tiles: 16-byte slot p of row r sits at slot p ^ key(r).
// The LDS has 64 banks of 4 bytes.  It serves 16-byte reads 16 lanes at a time, in the groups
// {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same plus 32; 8-byte reads 32 lanes at a
// time; 8-byte writes 16 lanes at a time (all probed with pairs of lanes and the bank
// conflict counter).  The keys make every access pattern below free of bank conflicts under
// these rules: the row-major fragments (16 bytes per lane, 16 rows x 2 slot columns per
// group), the two 8-byte reads of the b fragments, the transposing reads, the producers'
// writes of whole rows, and Pt's writes and reads (rows of 64 bytes).
template <int RB>
struct TpSwizzle {
    static_assert(RB == 64 || RB == 128, "rows of 64 or 128 bytes");
    static constexpr int kSlots = RB / 16;
    __device__ static __forceinline__ constexpr int key(int r) {
        const int lo = ((r >> 2) & 1), hi = ((r >> 2) ^ (r >> 3)) & 1;
        if (RB == 64) return lo | (hi << 1);
        return lo | (((r >> 1) & 1) << 1) | (hi << 2);
    }
    __device__ static __forceinline__ constexpr int addr(int row, int off) {
        return (row * kSlots + ((off >> 4) ^ key(row))) * 16 + (off & 15);
    }
};

// Column order of the b tiles.  Row m of state tile dt = 2 ks + u stands for
// d = 32 ks + 8 (m / 4) + 4 u + m % 4, and the transposing reads that fetch b^T for such a
// tile want its 16 columns side by side (two full 16-byte slots per row: free of bank
// conflicts under the swizzle): within each block of 32 columns the groups of four with
// u = 0 come first, then those with u = 1.  (d a multiple of 4.)
__device__ __forceinline__ constexpr int b_tile_column(int d) {
    return 32 * (d / 32) + 16 * ((d / 4) % 2) + 4 * ((d % 32) / 8) + d % 4;
}

// sum over the four groups of 16 lanes, in every lane: v_permlane16_swap exchanges the odd groups
// of its first operand with the even groups of its second, v_permlane32_swap the halves
__device__ __forceinline__ float sum_of_lane_groups(float x) {
    const uint32_t b = __float_as_uint(x);
    const auto p16 = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const float y = __uint_as_float(p16[0]) + __uint_as_float(p16[1]);
    const uint32_t c = __float_as_uint(y);
    const auto p32 = __builtin_amdgcn_permlane32_swap(c, c, false, false);
    return __uint_as_float(p32[0]) + __uint_as_float(p32[1]);
}

// Piece products of an X operand in PX pieces and a Y operand in PY (three for fp32 values, one for
// bf16 ones), smallest first: all but those below the last place of fp32.
template <int PX, int PY>
struct Products {
    static constexpr int count = PX == 3 && PY == 3 ? 6 : PX * PY;
    __device__ static constexpr int x(int m) {
        constexpr int all[6] = {0, 1, 2, 0, 1, 0};
        return PX == 1 ? 0 : PY == 1 ? 2 - m : all[m];
    }
    __device__ static constexpr int y(int m) {
        constexpr int all[6] = {2, 1, 0, 1, 0, 0};
        return PY == 1 ? 0 : PX == 1 ? 2 - m : all[m];
    }
};
// four consecutive values of a row in memory: fp32 (three pieces) or bf16 (one)
template <int P>
struct RowQuad {
    typedef u32x4 raw;
    static constexpr int bytes = 4;  // per value
    __device__ static __forceinline__ raw load(__amdgpu_buffer_rsrc_t rs, uint32_t at) {
        return __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0);
    }
    __device__ static __forceinline__ void to_lds(const raw r, lds_char *tile, int piece_bytes, int addr) {
        split_quad_to_lds(r, tile, piece_bytes, addr);
    }
};
template <>
struct RowQuad<1> {
    typedef u32x2 raw;
    static constexpr int bytes = 2;
    __device__ static __forceinline__ raw load(__amdgpu_buffer_rsrc_t rs, uint32_t at) {
        return __builtin_amdgcn_raw_buffer_load_b64(rs, at, 0, 0);
    }
    __device__ static __forceinline__ void to_lds(const raw r, lds_char *tile, int, int addr) {
        *(lds_vec2 *)(tile + addr) = r;
    }
};

// which words of a quad of columns from `col` on are a row's own, of `width` columns (the first one is)
template <bool ODD>
struct OwnWords {
    uint32_t m[3];
    __device__ __forceinline__ OwnWords(int col, int width) {
#pragma unroll
        for (int e = 0; e < 3; e++) m[e] = col + e + 1 < width ? 0xffffffffu : 0u;
    }
    template <typename Raw>
    __device__ __forceinline__ Raw of(const Raw r) const {
        if constexpr (ODD) return Raw{r.x, r.y & m[0], r.z & m[1], r.w & m[2]};
        return r;
    }
};

// which scan (and block of columns and segment: `which`) and which chain a workgroup takes:
// workgroups of one scan in groups of 8 (one per XCD), the groups of the scans of a launch side by
// side, so that scans reading the same rows share an L2 (also the segments of a chain, which read the
// same early rows)
__device__ __forceinline__ void tp_workgroup(const ScanArgs &p, uint32_t &which, uint32_t &chain) {
    const uint32_t chains = (uint32_t)p.waves_per_scan / (uint32_t)p.nseg;
    const uint32_t per_chain = (uint32_t)p.total_waves / chains;  // scans x segments
    const uint32_t full = (chains / 8u) * 8u;
    if (blockIdx.x < full * per_chain) {
        const uint32_t grp = blockIdx.x / (8u * per_chain), r = blockIdx.x % (8u * per_chain);
        which = r / 8u;
        chain = grp * 8u + r % 8u;
    } else {
        const uint32_t t = blockIdx.x - full * per_chain;
        which = t / (chains - full);
        chain = full + t % (chains - full);
    }
}
// LDS of a workgroup: bytes of the three buffers of a, b and v in pieces, and of Pt's two
template <int PA, int PB, int PV>
constexpr int kTpPieceBytes = 3 * (PA + PB + PV) * kChunk * 128;
constexpr int kTpPtBytes = 2 * 3 * kChunk * 64;
// Whether a kernel's loop over chunks is unrolled three times, with its buffers in the instructions' offsets
// (and three of Pt).  The fused attention, where the vector instructions of a producer and a consumer together
// take 58 % of their SIMD's issue (SQ_ACTIVE_INST_VALU, 29 % of a wavefront's life): 535 of them a chunk -> 515 this
// way, with the quadrant in two sums for four and its edges on branches; 80 chains, L=1000 36.4 -> 34.7 us, L=4096
// 137 -> 124.  bf16 rows, where a consumer's stream is what a chunk waits for: forward, 64 chains, L=2048 32.4 -> 30.5,
// 80 chains, L=1000 21.4 -> 19.9; 16384 positions of 128 chains of 32 x 128, training step 1799 -> 1756.  Not three
// pieces with two blocks: 108 registers would spill.
constexpr bool tp_unrolled(int ND, int pieces) { return ND == 1 || pieces < 9; }
constexpr int kTpZBytes = 4 * 2 * 2 * 64;  // z of the four consumers, fused attention with two blocks

// KS2: groups of 32 rows in the state's last block (1: a state of 65 .. 96 rows, whose last
// block skips the matrix instructions and fragment reads of its empty half)
// NORM: causally masked linear attention in the same walk (see ftc_wg_kernel.h for the equations):
// the producers apply phi(x) = elu(x) + 1 to a and b as they cut them and zero the rows of b at or
// beyond the key length.  The denominators phi(a_l) . sum_{j <= l} phi(b_j) are what the consumers
// have at hand: the column sums of the masked quadrants of Pt, and phi(a) times z, the sum of
// phi(b) over the chunks before.  z is one more column of the state whose "values" are ones; of each
// block of 64 rows consumer w keeps the half that belongs to k-step w / 2 (its first one: such
// consumers walk the two halves in the other order) and multiplies it with the 16 positions of its
// own quadrant: twelve matrix instructions, a cut and a reduction over the lane groups.  A
// position's two contributions meet in LDS behind the chunk's barrier, and rows are divided as they
// are stored.
// PA, PB, PV: pieces of the values of a, b and v: three for fp32 rows, one for bf16 rows, which are
// multiplied as they are; TO: the type of the result's rows
// ODD: fp32 rows of any width on 4-byte boundaries, as in ftc_tph_kernel.h: requests of 16 bytes all the
// same, words that belong to the next row cleared as a quad is cut, quads that straddle the end of a row
// stored word by word.  A chunk costs what it costs at the next multiple of 4; what is saved are copies
// (forward, 25 x 33, 99 chains, L=1531 77 -> 33 us, odd_on_three_pieces)
template <int ND, int KS2, bool NORM, int PA, int PB, int PV, typename TO, bool ODD = false>
__device__ __forceinline__ void scan_tp_body(uint32_t *__restrict__ ws_ptr, const ScanArgs &p, uint32_t which,
                                             uint32_t chain, lds_char *unit_pc, lds_char *pt_pc,
                                             float (*den_mem)[NORM ? kChunk : 1][2], uint32_t *order_sh) {
    constexpr int D = 64, F = 64;              // one block of state rows and of output columns
    constexpr int T = 256;                     // producer lanes
    constexpr int PF = kTpAhead;               // chunks requested ahead
    constexpr int RBA = D * 2, RBV = F * 2;    // bytes per row of a bf16 piece tile
    constexpr int kTileA = kChunk * RBA, kTileV = kChunk * RBV;
    constexpr int kOffB = PA * kTileA, kOffV = (PA + PB) * kTileA;
    constexpr int kBufBytes = (PA + PB) * kTileA + PV * kTileV;
    typedef Products<PB, PA> OfP;   // the quadrant of Pt
    typedef Products<3, PA> OfO;    // S^T a^T
    typedef Products<PB, PV> OfS;   // b^T v
    typedef Products<PV, 3> OfV;    // v^T Pt
    typedef RowQuad<PA> QuadA;
    typedef RowQuad<PB> QuadB;
    typedef RowQuad<PV> QuadV;
    constexpr int kTileP = kChunk * 64;        // Pt pieces: 32 rows (i) of 32 j
    constexpr int QA = D / 4, QV = F / 4;
    constexpr int LA = kChunk * QA / T, LV = kChunk * QV / T;
    static_assert(kChunk == 32 && T % QA == 0 && T % QV == 0, "shape");
    // (the fused attention's rows have 32, 64 or 128 values)
    constexpr bool kFullRows = NORM && KS2 == 2;
    constexpr bool kUnrolled = tp_unrolled(ND, PA + PB + PV);
    // Segments may start at half a trip of the first walk (two blocks: a chunk is two positions, so they may
    // without it).  Not with bf16 rows, whose launches took 0.1 us longer with the code, whole chains too (forward,
    // 58 chains, L=196 7.98 -> 8.10 us; 38, L=1291 18.4 in half steps, 18.1 in whole ones).
    constexpr bool kHalfTrips = ND == 1 && PA + PB + PV == 9;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool producer = wave >= 4;
    const int w = wave & 3;

    const uint32_t nseg = (uint32_t)p.nseg;
    const uint32_t chains = (uint32_t)p.waves_per_scan / nseg;
    // (a scan with more than 64 output columns counts as two, one per block of columns)
    const uint32_t virt = which / nseg;
    uint32_t scan_id = ODD ? 0 : virt / (uint32_t)p.tp_fblocks;
    if (ODD) {
#pragma unroll
        for (int i = 1; i < kMaxScans; i++)
            if ((int)virt >= p.tp_first[i]) scan_id = i;
    }
    const int fb = ODD ? (int)virt - p.tp_first[scan_id] : (int)(virt % (uint32_t)p.tp_fblocks);
    const ScanOperands &op = p.scan[scan_id];
    const int Dw = op.d;                        // state rows in all: a and b are this wide
    const int fw = min(F, op.f - F * fb);       // output columns of this block
    const bool REV = op.rev != 0;
    const int n = (int)(chain / (uint32_t)p.H), h = (int)(chain % (uint32_t)p.H);
    const int rows = (int)p.L;
    const int total_chunks = (rows + kChunk - 1) / kChunk;
    // Chunks are numbered in walking order; this workgroup's own are c0 .. nchunks - 1.  The
    // state before them comes from one of two places:
    //  * no exchange: the workgroup first walks chunks 0 .. c0 - 1 for their state alone;
    //  * exchange (p.tp_exchange, longer chains): it first walks its OWN chunks for their
    //    state alone, publishes that sum, and adds up the sums of the segments before it
    //    (StateExchange in ftc_mfma_kernel.h: flags and state slots in the workspace, fixed
    //    order of summation, bounded waits).  Segments are then taken in the order in which
    //    the workgroups of a chain start running (a ticket per chain), so that a workgroup
    //    only ever waits for workgroups that are running already.
    const bool exchange = p.tp_exchange != 0 && nseg > 1;
    gu32 *const hdr = (gu32 *)ws_ptr;
    gu32 *const flags = hdr + kHdrWords;
    const uint32_t chain_id = virt * chains + chain;  // over all scans of the launch
    int seg = (int)(which % nseg);
    if (exchange) {
        if (tid == 0)
            *order_sh = __hip_atomic_fetch_add(flags + kMaxWaves + chain_id, 1u, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        seg = (int)__builtin_amdgcn_readfirstlane(*order_sh);
        if ((uint32_t)seg >= nseg) {  // the control block was not zero when the launch began
            if (tid == 0)
                __hip_atomic_store(hdr + kHdrError, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
    }
    const int c0 = exchange ? seg * p.tp_seg_chunks : p.tp_start[seg];
    const int nchunks = min(total_chunks, exchange ? c0 + p.tp_seg_chunks : p.tp_start[seg + 1]);
    // the chunks walked for their state alone: so0 .. so0 + n1 - 1 (n1 a multiple of PF / 2; the
    // last segment of an exchange has no reader for its sum)
    const int so0 = exchange ? c0 : 0;
    const int n1c = exchange ? (seg + 1 < (int)nseg ? nchunks - c0 : 0) : c0;
    // A chunk is walked as ND positions, one per block of 64 state rows (columns of a and
    // b): position v has block v % ND.  v < n1: a chunk walked for its state alone; then
    // chunk c0 + (v - n1) / ND.  With an exchange the first pass runs against the direction
    // of the second, so that the second starts with the rows that the caches saw last.
    const int n1 = ND * n1c;
    const int nwalk = n1 + ND * (nchunks - c0);  // (position nwalk: a chunk of zeros)
    auto so_chunk = [&](int v) -> int { return exchange ? so0 + n1c - 1 - v / ND : so0 + v / ND; };
    auto walk_chunk = [&](int v) -> int { return v < n1 ? so_chunk(v) : c0 + (v - n1) / ND; };
    constexpr uint32_t kNoRow = 0x80000000u;  // an offset outside every descriptor
    // groups of 32 rows of block hb
    auto block_ks = [](int hb) -> int { return hb == ND - 1 ? KS2 : 2; };
    auto chunk_row0 = [&](int c) -> int { return REV ? rows - kChunk * (c + 1) : kChunk * c; };
    // Position k of the walk goes through LDS buffer (B0 + k) % 3, the first one of the walk proper through
    // buffer 0, so that a loop over those chunks that is unrolled three times knows its buffers.
    const int B0 = kUnrolled ? __builtin_amdgcn_readfirstlane((3 - n1 % 3) % 3) : 0;
    __syncthreads();
#ifdef FTC_TIMELINE
    // tuning aid: 32 time stamps per workgroup behind the pointer that the host passes in
    // p.key_len (FTC_STAMP_PTR), written by lane 0 of consumer 0 (0 .. 15) and of producer 0
    // (16 .. 31) in chunk 4 (NORM: that is the caller's key lengths, and nothing is stamped)
    typedef __attribute__((address_space(1))) uint64_t gu64;
    const bool stamp_on = !NORM && p.key_len != nullptr && w == 0 && lane == 0;
    gu64 *const stamp_base = (gu64 *)p.key_len + blockIdx.x * 32 + (producer ? 16 : 0);
#endif
    FTC_STAMP(14);  // workgroup under way

    if (producer) {
        // =========================== producers ===========================
        const int ptid = w * 64 + lane;
        const uint32_t a_slb = (uint32_t)op.a_sl * QuadA::bytes, b_slb = (uint32_t)op.b_sl * QuadB::bytes,
                       v_slb = (uint32_t)op.v_sl * QuadV::bytes;
        const char *a_seg = (const char *)op.a + ((int64_t)n * op.a_sn + (int64_t)h * op.a_sh) * QuadA::bytes;
        const char *b_seg = (const char *)op.b + ((int64_t)n * op.b_sn + (int64_t)h * op.b_sh) * QuadB::bytes;
        const char *v_seg = (const char *)op.v +
                            ((int64_t)n * op.v_sn + (int64_t)h * op.v_sh + F * fb) * QuadV::bytes;
        const __amdgpu_buffer_rsrc_t a_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)a_seg, 0, (rows - 1) * a_slb + Dw * QuadA::bytes, kRsrcFlags);
        const __amdgpu_buffer_rsrc_t b_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)b_seg, 0, (rows - 1) * b_slb + Dw * QuadB::bytes, kRsrcFlags);
        const __amdgpu_buffer_rsrc_t v_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)v_seg, 0, (rows - 1) * v_slb + fw * QuadV::bytes, kRsrcFlags);
        // Widths that do not fill their last block of 64: a lane whose four columns lie
        // beyond the width asks outside the descriptor and cuts zeros (widths are multiples
        // of 4).  A lane has the same columns in both of its quads.
        bool ab_in[ND];
#pragma unroll
        for (int hb = 0; hb < ND; hb++) ab_in[hb] = kFullRows || 4 * (ptid % QA) + D * hb < Dw;
        const bool v_in = 4 * (ptid % QV) < fw;
        const OwnWords<ODD> ab_own[2] = {{4 * (ptid % QA), Dw}, {4 * (ptid % QA) + D, Dw}}, v_own(4 * (ptid % QV), fw);
        uint32_t a_goff[LA], b_goff[LA], v_goff[LV];
        int a_waddr[LA], b_waddr[LA], v_waddr[LV];
#pragma unroll
        for (int q = 0; q < LA; q++) {
            const int u = q * T + ptid, row = u / QA, c4 = u % QA;
            a_goff[q] = (uint32_t)row * a_slb + 4u * QuadA::bytes * c4;
            b_goff[q] = (uint32_t)row * b_slb + 4u * QuadB::bytes * c4;
            a_waddr[q] = TpSwizzle<RBA>::addr(row, 8 * c4);
            b_waddr[q] = TpSwizzle<RBA>::addr(row, 2 * b_tile_column(4 * c4));
        }
#pragma unroll
        for (int q = 0; q < LV; q++) {
            const int u = q * T + ptid, row = u / QV, c4 = u % QV;
            v_goff[q] = (uint32_t)row * v_slb + 4u * QuadV::bytes * c4;
            v_waddr[q] = TpSwizzle<RBV>::addr(row, 8 * c4);
        }
        struct Raw {
            typename QuadA::raw a[LA];
            typename QuadB::raw b[LA];
            typename QuadV::raw v[LV];
        };
        Raw raw[PF];
        // Every request is made every time, whether its rows exist or not (of a chunk walked
        // for its state alone the producers need rows 0 .. 15 of b and v only, see below;
        // positions past the end of the walk have no rows): a request outside the descriptor
        // costs no memory traffic and reads as zero, and with a fixed number of requests per
        // chunk the compiler can wait for the oldest ones only (s_waitcnt vmcnt(n) with n the
        // number of younger requests) instead of for all.
        static_assert(LA == 2 && LV == 2, "quad 0 of a lane: rows 0 .. 15, quad 1: rows 16 .. 31");
        auto fetch = [&](Raw &r, int v, int hb) {  // v: position of the walk, hb = v % ND
            const int row0 = v < nwalk ? chunk_row0(walk_chunk(v)) : -2 * kChunk;
            const int row0_x = v >= n1 ? row0 : -2 * kChunk;
            const uint32_t col_a = (uint32_t)(D * QuadA::bytes * hb), col_b = (uint32_t)(D * QuadB::bytes * hb);
#pragma unroll
            for (int q = 0; q < LA; q++) {
                r.a[q] = QuadA::load(a_rs, ab_in[hb] ? a_goff[q] + col_a + (uint32_t)row0_x * a_slb : kNoRow);
                r.b[q] = QuadB::load(b_rs, ab_in[hb] ? b_goff[q] + col_b + (uint32_t)(q == 0 ? row0 : row0_x) * b_slb
                                                     : kNoRow);
            }
            // (the second block of a chunk multiplies the v tile of the first: no second copy)
            if (hb == 0) {
#pragma unroll
                for (int q = 0; q < LV; q++)
                    r.v[q] = QuadV::load(v_rs, v_in ? v_goff[q] + (uint32_t)(q == 0 ? row0 : row0_x) * v_slb : kNoRow);
            }
        };
        // NORM: keys at or beyond this row count as zero (phi(0) = 1, so do the rows that do not
        // exist, and the columns)
        const int key_rows = NORM && p.key_len ? (int)max((int64_t)0, min((int64_t)rows, p.key_len[n])) : rows;
        auto feature_a = [&](const auto x, int hb) {
            if constexpr (NORM) {
                u32x4 y = feature_quad(x);
                if (!ab_in[hb]) y = u32x4{0, 0, 0, 0};
                return y;
            } else {
                return x;
            }
        };
        auto feature_b = [&](const auto x, int hb, int v, int q) {  // quad q of position v
            if constexpr (NORM) {
                u32x4 y = feature_quad(x);
                const int row0 = v < nwalk ? chunk_row0(walk_chunk(v)) : -2 * kChunk;
                // (a scalar test: most chunks lie wholly below the limit)
                if (row0 < 0 || row0 + kChunk > key_rows) {
                    asm volatile("" : "+v"(y.x));  // (a branch, not eight selects in every chunk)
                    if ((uint32_t)(row0 + 16 * q + ptid / QA) >= (uint32_t)key_rows) y = u32x4{0, 0, 0, 0};
                }
                if (!ab_in[hb]) y = u32x4{0, 0, 0, 0};
                return y;
            } else {
                return x;
            }
        };
        // position k of the walk goes to its LDS buffer through register set k % PF.  The
        // first n1 positions (a multiple of PF / 2) only feed the state: no piece of a, and the
        // consumers, who have little to do there, cut rows 16 .. 31 of b and v themselves.
        auto cut = [&](const Raw &r, int buf, bool own, int hb, int v) {
            lds_char *const pc = unit_pc + buf * kBufBytes;
#pragma unroll
            for (int q = 0; q < LA; q++) {
                if (own) QuadA::to_lds(ab_own[hb].of(feature_a(r.a[q], hb)), pc, kTileA, a_waddr[q]);
                if (own || q == 0)
                    QuadB::to_lds(ab_own[hb].of(feature_b(r.b[q], hb, v, q)), pc + kOffB, kTileA, b_waddr[q]);
            }
            if (hb == 0) {
#pragma unroll
                for (int q = 0; q < LV; q++)
                    if (own || q == 0) QuadV::to_lds(v_own.of(r.v[q]), pc + kOffV, kTileV, v_waddr[q]);
            }
            // (a request whose answer is not used would be moved out of the loop: the waits
            // are the same either way)
            if (!own) asm volatile("" ::"v"(r.a[0]), "v"(r.a[1]), "v"(r.b[1]));
            if (!own && hb == 0) asm volatile("" ::"v"(r.v[1]));
        };
        // Barrier number k (k = 0: before the first position; k >= 1: in the middle of
        // position k - 1) finds position k cut.  The last one finds a chunk of zeros.
        // Two loops whose bodies are straight-line code, so that the waits inside them count
        // requests instead of draining them.
        int buf = B0;
        auto state_only = [&](int v, int j) {  // (v + j: the position, j: its register set)
            cut(raw[j], buf, false, j % ND, v + j);
            fetch(raw[j], v + j + PF, j % ND);
            buf = buf == 2 ? 0 : buf + 1;
            wg_barrier();
            __builtin_amdgcn_sched_barrier(0);  // one chunk at a time, in this order
        };
        // (half a trip in front where n1 is not a multiple of PF: the sets are requested in the order in which
        // they are used, and both ways leave them in the order that the loops count on)
        int first = 0;
        if (kHalfTrips && n1 % PF != 0) {
            static_assert(PF == 4, "half a trip: the sets of its second half first");
            fetch(raw[2], 0, 0), fetch(raw[3], 1, 0), fetch(raw[0], 2, 0), fetch(raw[1], 3, 0);
            state_only(-2, 2);
            state_only(-2, 3);
            first = 2;
        } else {
#pragma unroll
            for (int j = 0; j < PF; j++) fetch(raw[j], j, j % ND);
        }
        for (int v = first; v < n1; v += PF) {
#pragma unroll
            for (int j = 0; j < PF; j++) state_only(v, j);
        }
        // (whole trips in the loop, the rest after it: a way out of the middle of the loop
        // would join the paths at the loop's head and spoil the counting)
        int v = n1;
        for (; v + PF <= nwalk + 1; v += PF) {
#pragma unroll
            for (int j = 0; j < PF; j++) {
                if (v + j == n1 + 4) FTC_STAMP(0);
                cut(raw[j], buf, true, j % ND, v + j);
                if (v + j == n1 + 4) FTC_STAMP(1);
                fetch(raw[j], v + j + PF, j % ND);
                buf = buf == 2 ? 0 : buf + 1;
                if (v + j == n1 + 4) FTC_STAMP(2);
                wg_barrier();
                __builtin_amdgcn_sched_barrier(0);  // one chunk at a time, in this order
                if (v + j == n1 + 4) FTC_STAMP(3);
            }
        }
#pragma unroll
        for (int j = 0; j < PF - 1; j++) {
            if (v + j > nwalk) return;
            cut(raw[j], buf, true, j % ND, v + j);
            buf = buf == 2 ? 0 : buf + 1;
            wg_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
        return;
    }

    // =========================== consumers ===========================
    const int ln = lane & 15, g = lane >> 4;
    constexpr int kOutBytes = sizeof(TO);
    const uint32_t o_slb = (uint32_t)op.o_sl * kOutBytes;
    char *o_seg = (char *)op.out + ((int64_t)n * op.o_sn + (int64_t)h * op.o_sh + F * fb) * kOutBytes;
    const __amdgpu_buffer_rsrc_t o_rs =
        __builtin_amdgcn_make_buffer_rsrc((void *)o_seg, 0, (rows - 1) * o_slb + fw * kOutBytes, kRsrcFlags);
    // Pt quadrant of this wavefront: the two on the diagonal, the one inside the mask, and
    // (consumer 3, so that all four run the same instructions) the one outside it: zeros
    const int jh = w == 0 ? 0 : w == 1 ? 1 : ((w == 2) == REV ? 1 : 0);
    const int ih = w == 0 ? 0 : w == 1 ? 1 : 1 - jh;
    // Position tiles are numbered from this wavefront's own: local tile x is tile x ^ ih, so
    // that the quadrant always multiplies local tile 0.
    // NORM: k-steps of a block's rows in this consumer's order, its own half of z first
    const int ks0 = NORM && KS2 == 2 ? w >> 1 : 0;
    // row-major fragments of a and b: k-slots t <-> d = 32 ks + 8 g + t (one 16-byte read)
    // (b: its tile keeps the two groups of four apart, see b_tile_column: two 8-byte reads)
    int a_addr[2][2], b_addr[2][2];  // [local i tile][ks], [ks][u]
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
#pragma unroll
        for (int x = 0; x < 2; x++)
            a_addr[x][ks] = TpSwizzle<RBA>::addr(16 * (x ^ ih) + ln, 2 * (32 * (ks ^ ks0) + 8 * g));
#pragma unroll
        for (int u = 0; u < 2; u++)
            b_addr[ks][u] = kOffB + TpSwizzle<RBA>::addr(
                                        16 * jh + ln, 2 * b_tile_column(32 * (ks ^ ks0) + 8 * g + 4 * u));
    }
    // State tile dt = 2 ks + u: row m <-> d = 32 ks + 8 (m / 4) + 4 u + m % 4, so that the
    // accumulator registers of tiles 2 ks and 2 ks + 1 (rows 4 g + r) are k-slots 0..7 of
    // k-step ks in the order above.
    // Transposing reads: lane s of a group of 16 supplies 8 bytes (4 columns) of row
    // 8 g + s / 4 (+ 4); the group's lane i then holds column i % 4 of the group that lane
    // i / 4 supplied.
    //  b^T, tile dt: lane i <-> row m = i of the tile, so lane s supplies columns
    //  32 ks + 4 u + 8 (s % 4) + 0..3;  v: columns 16 w + 4 (s % 4) + 0..3
    int bt_addr[4][2], vt_addr[2];
#pragma unroll
    for (int u2 = 0; u2 < 2; u2++) {
        const int row = 8 * g + (ln >> 2) + 4 * u2;
#pragma unroll
        for (int dt = 0; dt < 4; dt++)
            bt_addr[dt][u2] = kOffB + TpSwizzle<RBA>::addr(
                row, 2 * b_tile_column(32 * ((dt / 2) ^ ks0) + 4 * (dt % 2) + 8 * (ln & 3)));
        vt_addr[u2] = kOffV + TpSwizzle<RBV>::addr(row, 2 * (16 * w + 4 * (ln & 3)));
    }
    // Pt in LDS: row i, j contiguous.  Written 4 values at a time (j = 16 jh + 4 g + r), read
    // as fragments with k-slots j = 8 g + t
    const int pt_waddr = TpSwizzle<64>::addr(16 * ih + ln, 2 * (16 * jh + 4 * g));
    int pt_raddr[2];
#pragma unroll
    for (int x = 0; x < 2; x++) pt_raddr[x] = TpSwizzle<64>::addr(16 * (x ^ ih) + ln, 16 * g);
    uint32_t keep[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int j = 16 * jh + 4 * g + r, i = 16 * ih + ln;
        keep[r] = (REV ? (j >= i) : (j <= i)) ? 0xffffffffu : 0u;
        asm volatile("" : "+v"(keep[r]));
    }
    uint32_t o_lane[2];
#pragma unroll
    for (int x = 0; x < 2; x++)
        o_lane[x] = (uint32_t)(16 * (x ^ ih) + ln) * o_slb + (uint32_t)kOutBytes * (16 * w + 4 * g);
    const int o_cols = fw - (16 * w + 4 * g);
    const bool o_in = o_cols >= (ODD ? 4 : 1);  // (columns beyond the width are not stored)
    const bool o_straddles = ODD && fw > 0 && fw % 4 != 0 && fw / 16 == w;

    f32x4 S[ND][4];  // the slab's rows, block by block
#pragma unroll
    for (int hb = 0; hb < ND; hb++)
#pragma unroll
        for (int dt = 0; dt < 4; dt++) S[hb][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    // the caller's state: lane (f = 16 w + ln, g), tile dt, register r <-> row d below
    auto state_row = [&](int dt, int r) -> int { return 32 * (dt / 2) + 8 * g + 4 * (dt % 2) + r; };
    const bool st_in = 16 * w + ln < fw;
    auto add_caller_state = [&]() {
        const float *base =
            op.s0 + (int64_t)n * op.s0_sn + (int64_t)h * op.s0_sh + F * fb + 16 * w + ln;
#pragma unroll
        for (int hb = 0; hb < ND; hb++)
#pragma unroll
            for (int dt = 0; dt < 4; dt++) {
                // (rows and columns beyond the widths: nothing is read, zero is added)
                float x[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int d = D * hb + state_row(dt, r);
                    const bool in = st_in && d < Dw;
                    x[r] = *(in ? base + (int64_t)d * op.s0_sd : op.s0);
                    x[r] = in ? x[r] : 0.f;
                }
                S[hb][dt] += f32x4{x[0], x[1], x[2], x[3]};
            }
    };
    // (with an exchange the sums that travel are those of the rows alone; every segment adds
    // the caller's state on top of what it gathers)
    if (!NORM && op.s0 && !exchange) add_caller_state();
    // NORM: this consumer's half of z, block by block (tiles 0 and 1 in its order, all columns alike)
    const bool has_z = NORM && (KS2 == 2 || w < 2);
    // (two blocks: z is in LDS, one copy per consumer that only it uses, and a chunk's sum is added to it
    // as a whole.  Accumulated in registers by the matrix instructions 130 chains of 4000 positions were
    // 5.2e-7 from float64, this way 1.2e-7; added as a whole in registers 21 of them spilled, and 128
    // chains of 856 took 128 us against 90.)
    f32x4 Z[ND][2];
    typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
    lds_f32x4 *const z_mem = (lds_f32x4 *)(pt_pc + kTpPtBytes) + 8 * ND * w + g;
#pragma unroll
    for (int hb = 0; hb < ND; hb++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
            Z[hb][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (NORM && ND > 1) z_mem[8 * hb + 4 * t] = Z[hb][t];
        }
    const Frag ones = {{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u}};
    // The products of up to eight chunks are added up by themselves (R) before they are added to the
    // state, where there are registers for it; the state in use is S + R.  (The sums of the matrix
    // instructions fall short by a part of the last place of the sum each, which keys and weights that
    // are all positive add up.  bf16 rows: the state handed out after 1000 positions was 2.7e-7 off
    // without it, 1.0e-7 on the kernels that split L.)
    // NORM: each chunk's products by themselves, and z's of up to eight chunks (300 chains of 4000 positions
    // walked whole were 7e-7 from float64 without either, the workgroup form's short segments are 3e-7; R in place
    // of the chunk's own sums: 80 chains, L=4096 1.08e-7 against 1.06e-7, and 15 more registers that spilled).  Not
    // while chunks are walked for their state alone, nor with two blocks: those registers would spill.
    // ODD: also while chunks are walked for their state (220 -> 237 registers); with two blocks each
    // chunk's products by themselves, a tile's sum added to the state as soon as it is whole (in the first
    // walk only where the last block has 32 rows: else 111 registers would spill).  127 x 127 backward,
    // 15 chains, L=710: 2-norm error 3.6e-7 -> 2.7e-7 at the same time.
    constexpr bool kMixed = PA + PB + PV < 9, kApart = (ODD && ND == 1) || kMixed, kFirstApart = kMixed || (ODD && ND == 1),
                   kChunkSums = (ODD && ND > 1) || (NORM && ND == 1), kFirstSums = ODD && ND > 1 && KS2 == 1,
                   kApartZ = NORM && ND == 1;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 R[ND][4], Zr[ND][2];
    f32x4 chunk_sum[4];
    auto add_product = [&](int hb, int dt, const Frag &x, const Frag &y, bool first) {
        if (kChunkSums)
            chunk_sum[dt] = mfma16(x, y, first ? zero : chunk_sum[dt]);
        else if (kApart)
            R[hb][dt] = mfma16(x, y, R[hb][dt]);
        else
            S[hb][dt] = mfma16(x, y, S[hb][dt]);
    };
    auto add_chunk_sums = [&](int hb, int first, int end) {
        if (kChunkSums)
#pragma unroll
            for (int dt = first; dt < end; dt++) S[hb][dt] += chunk_sum[dt];
    };
    auto state = [&](int hb, int dt, int r) -> float { return kApart ? S[hb][dt][r] + R[hb][dt][r] : S[hb][dt][r]; };
    auto sum_of_keys = [&](int hb, int t, int r) -> float { return Z[hb][t][r] + Zr[hb][t][r]; };
    auto clear_apart = [&]() {
#pragma unroll
        for (int hb = 0; hb < ND; hb++)
#pragma unroll
            for (int dt = 0; dt < 4; dt++) {
                if (kApart) R[hb][dt] = zero;
                if (kApartZ) Zr[hb][dt % 2] = zero;
            }
    };
    auto add_apart = [&]() {
        if (kApart || kApartZ) {
#pragma unroll
            for (int hb = 0; hb < ND; hb++)
#pragma unroll
                for (int dt = 0; dt < 4; dt++) {
                    if (kApart && dt / 2 < (hb == ND - 1 ? KS2 : 2)) S[hb][dt] += R[hb][dt];
                    if (kApartZ && dt < 2) Z[hb][dt] += Zr[hb][dt];
                }
            clear_apart();
        }
    };

    // A wavefront issues in order, and four of them share the LDS: reads are therefore
    // written out between the matrix instructions they run under, one at a time, and
    // scheduling barriers keep the compiler from regrouping them.
    Frag af[2][2][PA], bfr[2][PB], bt[4][PB], vf[PV];
    // row-major fragment number i of a chunk (18 of fp32 rows: b for the quadrant first, then a)
    constexpr int kRowFrags = 2 * PB + 4 * PA;
    auto rm_frag = [&](const lds_char *pc, int i, int hb) {  // hb: the block of that position
        if (i >= kRowFrags) return;
        if (i < 2 * PB) {
            const int k = i % PB, ks = i / PB;
            if (ks < block_ks(hb))
                bfr[ks][k] = lds_frag8x2(pc + k * kTileA + b_addr[ks][0], pc + k * kTileA + b_addr[ks][1]);
        } else {
            const int k = (i - 2 * PB) % PA, ks = ((i - 2 * PB) / PA) % 2, x = (i - 2 * PB) / (2 * PA);
            if (ks < block_ks(hb)) af[x][ks][k] = lds_frag16(pc + k * kTileA + a_addr[x][ks]);
        }
    };
    // position-major fragment number i of a chunk (15 of fp32 rows: v first, then b^T tile by tile)
    // (pcv: the buffer that holds the chunk's v tile, which is the one of its first block)
    constexpr int kTrFrags = PV + 4 * PB;
    auto tr_frag_into = [&](Frag (&btx)[4][PB], Frag (&vfx)[PV], const lds_char *pc,
                            const lds_char *pcv, int i, int hb) {
        if (i >= kTrFrags) return;
        if (i < PV)
            vfx[i] = lds_frag_tr(pcv + i * kTileV + vt_addr[0], pcv + i * kTileV + vt_addr[1]);
        else {
            const int dt = (i - PV) / PB, k = (i - PV) % PB;
            if (dt / 2 >= block_ks(hb)) return;  // tiles 2, 3: rows 32 .. 63
            btx[dt][k] = lds_frag_tr(pc + k * kTileA + bt_addr[dt][0], pc + k * kTileA + bt_addr[dt][1]);
        }
    };
    auto prev_buf = [](int b) -> int { return b == 0 ? 2 : b - 1; };

    auto next_buf = [](int b) -> int { return b == 2 ? 0 : b + 1; };
    int buf = B0;  // LDS buffer of the position at hand
    if (n1 > 0) {
        // ---- the first n1 positions of the walk: state update only ----
        if (kFirstApart) clear_apart();
        // product i of the 24 of a position: tile by tile, or (sums of a chunk by themselves) two tiles after
        // the other two, whose sums are added meanwhile
        auto add_first = [&](int hb, int i, const Frag (&btx)[4][PB], const Frag (&vfx)[PV]) {
            const int dt = kFirstSums ? 2 * (i / 12) + i % 2 : i % 4, m = kFirstSums ? i % 12 / 2 : i / 4;
            if (kFirstSums && (i == 14 || i == 15)) S[hb][i - 14] += chunk_sum[i - 14];
            if (dt / 2 >= block_ks(hb) || m >= OfS::count) return;
            const Frag &x = btx[dt][OfS::x(m)], &y = vfx[OfS::y(m)];
            if (kFirstSums)
                chunk_sum[dt] = mfma16(x, y, m == 0 ? zero : chunk_sum[dt]);
            else if (kFirstApart)
                R[hb][dt] = mfma16(x, y, R[hb][dt]);
            else
                S[hb][dt] = mfma16(x, y, S[hb][dt]);
        };
        auto add_keys = [&](int hb, int i, const Frag (&btx)[4][PB]) {
            if (ND == 1) {
                if (i < 6) Z[hb][i % 2] = mfma16(btx[i % 2][2 - i / 2], ones, Z[hb][i % 2]);
            } else {
                if (i < 6) Zr[0][i % 2] = mfma16(btx[i % 2][2 - i / 2], ones, i < 2 ? zero : Zr[0][i % 2]);
                if (i == 7 || i == 8) Z[0][i - 7] = z_mem[8 * hb + 4 * (i - 7)];
                if (i == 12 || i == 13) z_mem[8 * hb + 4 * (i - 12)] = Z[0][i - 12] + Zr[0][i - 12];
            }
        };
        // The consumers have little to do here, so they share the producers' work: rows
        // 16 .. 31 of b and v of these chunks are fetched and cut by the consumers (lane
        // 64 w + lane takes the quad that producer lane of the same number would take).
        // The loop is skewed by one chunk: while the matrix instructions of chunk k - 1 run,
        // the fragments of chunk k arrive in the other set of registers.
        const int cid = w * 64 + lane, crow = (T + cid) / QA, cc4 = (T + cid) % QA;
        const uint32_t b_slb = (uint32_t)op.b_sl * QuadB::bytes, v_slb = (uint32_t)op.v_sl * QuadV::bytes;
        const char *b_seg = (const char *)op.b + ((int64_t)n * op.b_sn + (int64_t)h * op.b_sh) * QuadB::bytes;
        const char *v_seg = (const char *)op.v +
                            ((int64_t)n * op.v_sn + (int64_t)h * op.v_sh + F * fb) * QuadV::bytes;
        const __amdgpu_buffer_rsrc_t b_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)b_seg, 0, (rows - 1) * b_slb + Dw * QuadB::bytes, kRsrcFlags);
        const __amdgpu_buffer_rsrc_t v_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)v_seg, 0, (rows - 1) * v_slb + fw * QuadV::bytes, kRsrcFlags);
        bool b_in[ND];
#pragma unroll
        for (int hb = 0; hb < ND; hb++) b_in[hb] = kFullRows || 4 * cc4 + D * hb < Dw;
        const bool v_in = 4 * cc4 < fw;
        const OwnWords<ODD> b_own[2] = {{4 * cc4, Dw}, {4 * cc4 + D, Dw}}, v_own(4 * cc4, fw);
        const uint32_t b_goff = (uint32_t)crow * b_slb + 4u * QuadB::bytes * cc4,
                       v_goff = (uint32_t)crow * v_slb + 4u * QuadV::bytes * cc4;
        const int b_waddr = TpSwizzle<RBA>::addr(crow, 2 * b_tile_column(4 * cc4)),
                  v_waddr = TpSwizzle<RBV>::addr(crow, 8 * cc4);
        struct RawC {
            typename QuadB::raw b;
            typename QuadV::raw v;
        };
        RawC rawc[PF];
        // (every request every time, as the producers do: from position n1 on outside the
        // descriptor)
        auto cfetch = [&](RawC &r, int v, int hb) {  // hb = v % ND
            const int row0 = v < n1 ? chunk_row0(so_chunk(v)) : -2 * kChunk;
            r.b = QuadB::load(b_rs, b_in[hb] ? b_goff + (uint32_t)(D * QuadB::bytes * hb) + (uint32_t)row0 * b_slb
                                             : kNoRow);
            if (hb == 0) r.v = QuadV::load(v_rs, v_in ? v_goff + (uint32_t)row0 * v_slb : kNoRow);
        };
        const int key_rows = NORM && p.key_len ? (int)max((int64_t)0, min((int64_t)rows, p.key_len[n])) : rows;
        auto ccut_b = [&](const RawC &r, int bufk, int v) {
            typename QuadB::raw x = r.b;
            if constexpr (NORM) {  // (position v of the walk, as the producers do)
                x = feature_quad(x);
                const int row0 = chunk_row0(so_chunk(v));
                if (row0 < 0 || row0 + kChunk > key_rows) {
                    if ((uint32_t)(row0 + crow) >= (uint32_t)key_rows) x = u32x4{0, 0, 0, 0};
                }
                if (!b_in[v % ND]) x = u32x4{0, 0, 0, 0};
            }
            QuadB::to_lds(b_own[v % ND].of(x), unit_pc + bufk * kBufBytes + kOffB, kTileA, b_waddr);
        };
        auto ccut_v = [&](const RawC &r, int bufk) {
            QuadV::to_lds(v_own.of(r.v), unit_pc + bufk * kBufBytes + kOffV, kTileV, v_waddr);
        };
        Frag bt2[4][PB] = {}, vf2[PV] = {};  // (the first round multiplies zeros)
        int bufn = next_buf(B0);           // LDS buffer of the position after the one at hand
        auto state_only = [&](int c, int j) {  // (position c + j, in register set j)
            const lds_char *pc = unit_pc + buf * kBufBytes;
            const lds_char *pcv = j % ND == 0 ? pc : unit_pc + prev_buf(buf) * kBufBytes;
            // position c + j + 1 is cut under the matrix instructions of position
            // c + j - 1 (position n1 is all the producers')
            const bool cut_next = j < PF - 1 || c + PF < n1;
            const RawC &rn = rawc[(j + 1) % PF];
            const int hp = (j + ND - 1) % ND;  // block of the position before
#pragma unroll
            for (int i = 0; i < 24; i++) {
                if (j % 2 == 0) {
                    add_first(hp, i, bt2, vf2);
                    if constexpr (NORM)
                        add_keys(hp, i, bt2);
                    tr_frag_into(bt, vf, pc, pcv, i, j % ND);
                } else {
                    add_first(hp, i, bt, vf);
                    if constexpr (NORM)
                        add_keys(hp, i, bt);
                    tr_frag_into(bt2, vf2, pc, pcv, i, j % ND);
                }
                if (i == 15 && cut_next) ccut_b(rn, bufn, c + j + 1);
                if (i == 19 && cut_next && (j + 1) % ND == 0) ccut_v(rn, bufn);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (kFirstSums) add_chunk_sums(hp, 2, 2 * block_ks(hp));
            cfetch(rawc[(j + 1) % PF], c + j + 1 + PF, (j + 1) % ND);
            buf = bufn;
            bufn = next_buf(bufn);
            wg_barrier();
            __builtin_amdgcn_sched_barrier(0);
        };
        int first = 0;
        if (kHalfTrips && n1 % PF != 0) {  // (half a trip in front, as the producers do)
            cfetch(rawc[2], 0, 0), cfetch(rawc[3], 1, 0), cfetch(rawc[0], 2, 0), cfetch(rawc[1], 3, 0);
            ccut_b(rawc[2], B0, 0);
            ccut_v(rawc[2], B0);
            cfetch(rawc[2], PF, 0);
            wg_barrier();
            state_only(-2, 2);
            state_only(-2, 3);
            first = 2;
        } else {
#pragma unroll
            for (int j = 0; j < PF; j++) cfetch(rawc[j], j, j % ND);
            ccut_b(rawc[0], B0, 0);
            ccut_v(rawc[0], B0);
            cfetch(rawc[0], PF, 0);
            wg_barrier();
        }
        FTC_STAMP(13);  // first chunk cut
        for (int c = first; c < n1; c += PF) {
#pragma unroll
            for (int j = 0; j < PF; j++) state_only(c, j);
            if (kFirstApart && c % 8 < PF) add_apart();
        }
        // the last of these positions (n1 is even: its fragments are in the second set)
#pragma unroll
        for (int i = 0; i < 24; i++) {
            add_first(ND - 1, i, bt2, vf2);
            if constexpr (NORM)
                add_keys(ND - 1, i, bt2);
            rm_frag(unit_pc + buf * kBufBytes, i, 0);  // our own first chunk is cut
            __builtin_amdgcn_sched_barrier(0);
        }
        if (kFirstSums) add_chunk_sums(ND - 1, 2, 2 * KS2);
    } else {
        wg_barrier();
        FTC_STAMP(13);  // first chunk cut
#pragma unroll
        for (int i = 0; i < kRowFrags; i++) rm_frag(unit_pc, i, 0);
    }
    if (exchange) {
        // ---- the sum of this segment's rows goes out, the state before the segment comes in ----
        const uint32_t total_units = (uint32_t)p.total_waves;
        gfloat *const sums = (gfloat *)(hdr + kControlBytes / 4);
        // the flag words and state slots of consumer w of the segment with ticket t are those
        // of "ticket" w * total_units + t (as in ftc_wg_kernel.h)
        constexpr int DX = NORM ? ND + 1 : ND;  // (z rides along in a tile of its own)
        // (bf16 rows keep the registers with which two workgroups share a CU where the state has 32 rows; two blocks have
        // none to spare)
        constexpr int kBatch = ND == 1 && PA + PB + PV == 9 ? 2 : 1;
        StateExchange<DX, 1, kBatch> xch(flags, sums, 4u * total_units,
                                (uint32_t)w * total_units + chain_id * nseg + (uint32_t)seg, seg,
                                (int)nseg, p.group, lane);
        if (kFirstApart && n1 > 0) add_apart();
        f32x16 Sx[DX][1], X[DX][1];
        if (NORM) {
            Sx[DX - 1][0] = f32x16{};
#pragma unroll
            for (int i = 0; i < 8 * ND; i++) Sx[DX - 1][0][i] = ND == 1 ? Z[i / 8][i / 4 % 2][i % 4] : z_mem[8 * (i / 8) + 4 * (i / 4 % 2)][i % 4];
        }
#pragma unroll
        for (int hb = 0; hb < ND; hb++)
#pragma unroll
            for (int dt = 0; dt < 4; dt++)
#pragma unroll
                for (int r = 0; r < 4; r++) Sx[hb][0][4 * dt + r] = S[hb][dt][r];
        if (n1 > 0) xch.publish_sum(Sx);
        xch.gather(Sx, X);
        if (xch.failed && lane == 0)
            __hip_atomic_store(hdr + kHdrError, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int hb = 0; hb < ND; hb++)
#pragma unroll
            for (int dt = 0; dt < 4; dt++)
#pragma unroll
                for (int r = 0; r < 4; r++) S[hb][dt][r] = X[hb][0][4 * dt + r];
        if (NORM) {
#pragma unroll
            for (int i = 0; i < 2 * ND; i++) {
                const f32x4 z = {X[DX - 1][0][4 * i], X[DX - 1][0][4 * i + 1], X[DX - 1][0][4 * i + 2],
                                 X[DX - 1][0][4 * i + 3]};
                Z[i / 2][i % 2] = z;
                if (ND > 1) z_mem[4 * i] = z;
            }
        }
        if (!NORM && op.s0) add_caller_state();
    }
    if (kFirstApart && n1 > 0 && !exchange) add_apart();
    clear_apart();
    // S_w as pieces in A operand order (slots 0..3 from tile 2 ks, 4..7 from tile 2 ks + 1).
    // Tiles 0 and 1 are final after phase 3 and are cut under phase 4, tiles 2 and 3 after
    // phase 4 and are cut under phase 1 of the next chunk.
    Frag sf[2][3];
    auto cut_s = [&](int hb, int ks, int q) {
        uint32_t o[3];
        split_pair_under_mfma(state(hb, 2 * ks + q / 2, 2 * (q % 2)), state(hb, 2 * ks + q / 2, 2 * (q % 2) + 1), o);
#pragma unroll
        for (int k = 0; k < 3; k++) sf[ks][k].w[q] = o[k];
    };
#pragma unroll
    for (int q = 0; q < 4; q++) cut_s(0, 0, q);

    // A matrix instruction that accumulates into the result of the one before it waits for
    // that result (about twice the issue interval of independent ones), so every phase
    // below keeps four to six accumulators in turn: the quadrant and Ot_w are summed in
    // parts that are added at the end, and phases are interleaved.
    // Ot_w of the chunk before, and where its rows go (before the first chunk: nowhere, an
    // offset beyond the descriptor, whose stores are dropped)
    f32x4 O4[2][2];
#pragma unroll
    for (int i = 0; i < 4; i++) O4[i / 2][i % 2] = f32x4{0.f, 0.f, 0.f, 0.f};
    uint32_t o_off = 0x80000000u;
    // lane (i = 16 (x ^ ih) + ln, g) holds f = 16 w + 4 g + 0..3
    float r_den[2] = {0.f, 0.f};  // NORM: reciprocals of the denominators of O's rows
    auto store_rows = [&](int x) {
        f32x4 o = O4[x][0] + O4[x][1];
        if (NORM) o *= r_den[x];
        buffer_store_out(o_rs, o_in ? o_off + o_lane[x] : kNoRow, o[0], o[1], o[2], o[3], (TO *)nullptr);
        if (o_straddles) {
            const uint32_t first = o_off + o_lane[x];
#pragma unroll
            for (int e = 0; e < 3; e++)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[e]), o_rs,
                                                      o_cols < 4 && o_cols > e ? first + 4u * e : kNoRow, 0, 0);
        }
    };
    const bool den_out = NORM && w == 0 && fb == 0 && op.s_out;
    const __amdgpu_buffer_rsrc_t den_rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(den_out ? op.s_out + (int64_t)n * op.so_sn + (int64_t)h * op.so_sh : nullptr), 0,
        den_out ? 4u * (uint32_t)rows : 0u, kRsrcFlags);
    // sums that the quadrant is added up from
    constexpr int kPSums = (NORM && ND == 1) || OfP::count == 1 ? 2 : 4;
    f32x4 Pkeep = {0.f, 0.f, 0.f, 0.f};  // the quadrant summed over the blocks so far
    f32x4 Az = {0.f, 0.f, 0.f, 0.f};     // NORM: phi(a) z of the quadrant's positions
    // (B: the LDS buffer of the chunk's first position, a compile-time number where the loop is unrolled)
    auto chunk_body = [&](int c, auto buffer_number) {
        constexpr int B = decltype(buffer_number)::value;
        const int pt_buf = kUnrolled ? B : c & 1;
#pragma unroll
        for (int hb = 0; hb < ND; hb++) {  // block hb of the state rows
            if (kUnrolled) buf = (B + hb) % 3;
            const lds_char *pc = unit_pc + buf * kBufBytes;
            const lds_char *pcv = hb == 0 ? pc : unit_pc + prev_buf(buf) * kBufBytes;
            lds_char *const ptc = pt_pc + pt_buf * (3 * kTileP);
            // The quadrants of a chunk's blocks are added up before they are cut: only the
            // last block of a chunk hands Pt to the others and multiplies it with v.
            const bool last_block = hb == ND - 1;
            Frag pf[2][3];
            f32x4 P4[4];
            Frag zf[3];  // NORM: z in pieces
            float P_sum = 0.f;
            // (the first product of a sum adds to a constant)
            if (c == c0 + 4) FTC_STAMP(0);
            __builtin_amdgcn_sched_barrier(0);
            // the quadrant is added up, masked, cut and handed to the others, step by step underneath
            // the products (bf16 rows: two matrix instructions, and already in phase 1)
            constexpr bool kEarlyQuadrant = OfP::count == 1;
            f32x4 P;
            uint32_t plo[3], phi[3];
            auto quadrant = [&](int step) {
                if (step == 1) {
                    P = kPSums == 2 ? P4[0] + P4[1] : (P4[0] + P4[1]) + (P4[2] + P4[3]);
                    if (hb > 0) P += Pkeep;
                    if (!last_block) Pkeep = P;
                }
                if (step == 2 && last_block)
                    split_pair_under_mfma(__uint_as_float(__float_as_uint(P[0]) & keep[0]),
                                          __uint_as_float(__float_as_uint(P[1]) & keep[1]), plo);
                if (step == 4 && last_block)
                    split_pair_under_mfma(__uint_as_float(__float_as_uint(P[2]) & keep[2]),
                                          __uint_as_float(__float_as_uint(P[3]) & keep[3]), phi);
                if (step == 6 && last_block) {
#pragma unroll
                    for (int k = 0; k < 3; k++) {
                        const u32x2 xk = {plo[k], phi[k]};
                        *(lds_vec2 *)(ptc + k * kTileP + pt_waddr) = xk;
                    }
                }
            };
            // phase 1: (1) the quadrant in turn with (2b) Ot_w = S_w^T a^T for rows 0 .. 31 of the
            // state; underneath: the rows of the chunk before go out, tiles 2, 3 of S_w are cut into
            // pieces, the first position-major reads.  (Two matrix instructions to an iteration:
            // one takes four times what another instruction takes to issue, and with the products
            // in phases of their own those without vector work beside them ran at the matrix
            // rate and the others at the rate of issue, twice as long as either.)
#pragma unroll
            for (int i = 0; i < 12; i++) {
                const int ks = i % 2, m = i / 2, x = i % 2;
                if (hb == 0 && i < 2) store_rows(i);
                if (ks < block_ks(hb) && m < OfP::count)
                    P4[i % kPSums] = mfma16(bfr[ks][OfP::x(m)], af[0][ks][OfP::y(m)], i < kPSums ? zero : P4[i % kPSums]);
                else if (i < kPSums)
                    P4[i % kPSums] = zero;
                if (m < OfO::count)
                    O4[x][0] = mfma16(sf[0][OfO::x(m)], af[x][0][OfO::y(m)], i < 2 && hb == 0 ? zero : O4[x][0]);
                if (i < 4 && block_ks(hb) > 1) cut_s(hb, 1, i);
                if (kEarlyQuadrant) quadrant(i - 4);
                if (NORM && ND > 1 && (i == 5 || i == 7)) Z[0][i / 2 - 2] = z_mem[8 * hb + 4 * (i / 2 - 2)];
                if (NORM && i >= 8) {  // z in pieces
                    uint32_t o[3];
                    if (ND > 1)
                        split_pair_under_mfma(Z[0][(i - 8) / 2][2 * (i % 2)], Z[0][(i - 8) / 2][2 * (i % 2) + 1], o);
                    else
                        split_pair_under_mfma(sum_of_keys(hb, (i - 8) / 2, 2 * (i % 2)),
                                              sum_of_keys(hb, (i - 8) / 2, 2 * (i % 2) + 1), o);
#pragma unroll
                    for (int k = 0; k < 3; k++) zf[k].w[i - 8] = o[k];
                }
                tr_frag_into(bt, vf, pc, pcv, i, hb);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (c == c0 + 4) FTC_STAMP(1);
            // phase 2: (2b) for rows 32 .. 63 in turn with (3) S_w += b^T v_w for tiles 0 and 1;
            // underneath: the last position-major reads, and the quadrant
#pragma unroll
            for (int i = 0; i < 12; i++) {
                const int x = i % 2, m = i / 2;
                if (block_ks(hb) > 1 && m < OfO::count)
                    O4[x][1] = mfma16(sf[1][OfO::x(m)], af[x][1][OfO::y(m)], i < 2 && hb == 0 ? zero : O4[x][1]);
                else if (i < 2 && hb == 0)
                    O4[x][1] = zero;
                if (i < 2 * OfS::count)
                    add_product(hb, i % 2, bt[i % 2][OfS::x(i / 2)], vf[OfS::y(i / 2)], i < 2);
                if (i < 3) tr_frag_into(bt, vf, pc, pcv, 12 + i, hb);
                if constexpr (NORM) {
                    if (i < 6) {
                        Az = mfma16(zf[OfO::x(i)], af[0][0][OfO::y(i)], i == 0 && hb == 0 ? zero : Az);
                    } else {
                        f32x4 &sum = kApartZ ? Zr[hb][i % 2] : Zr[0][i % 2];
                        sum = mfma16(bt[i % 2][5 - i / 2], ones, kApartZ || i >= 8 ? sum : zero);
                    }
                }
                if (NORM && ND > 1 && (i == 7 || i == 8)) Z[0][i - 7] = z_mem[8 * hb + 4 * (i - 7)];
                if (!kEarlyQuadrant) quadrant(i);
                if (NORM && i == 7 && last_block) {
                    float m4[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) m4[r] = __uint_as_float(__float_as_uint(P[r]) & keep[r]);
                    P_sum = (m4[0] + m4[1]) + (m4[2] + m4[3]);
                }
                if (NORM && i == 9 && last_block) {
                    P_sum = sum_of_lane_groups(P_sum);
                    if (g == 0) den_mem[pt_buf][16 * ih + ln][w >> 1] = (has_z ? Az[0] : 0.f) + P_sum;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (c == c0 + 4) FTC_STAMP(2);
            buf = next_buf(buf);
            wg_barrier();
            if (c == c0 + 4) FTC_STAMP(4);
            // All of Pt is in LDS and the next chunk is cut: its row-major fragments are
            // requested under what follows.
            add_chunk_sums(hb, 0, 2);
            // phase 4: (3) for tiles 2 and 3 in turn with (2a) Ot_w += v_w^T Pt; underneath:
            // tiles 0, 1 of S_w cut into pieces
            const lds_char *pn = unit_pc + buf * kBufBytes;
            if (last_block) {
#pragma unroll
                for (int x = 0; x < 2; x++)
#pragma unroll
                    for (int k = 0; k < 3; k++) pf[x][k] = lds_frag16(ptc + k * kTileP + pt_raddr[x]);
            }
            if constexpr (NORM) {
                if (last_block) {
#pragma unroll
                    for (int x = 0; x < 2; x++) {
                        const float *part = den_mem[pt_buf][16 * (x ^ ih) + ln];
                        const float den = (part[0] + part[1]) + p.eps;
                        r_den[x] = 1.0f / den;
                        // (the caller's copy of the denominators, for the backward)
                        if (den_out)
                            __builtin_amdgcn_raw_buffer_store_b32(
                                __float_as_uint(den), den_rs,
                                g == 0 ? 4u * (uint32_t)(chunk_row0(c) + 16 * (x ^ ih) + ln) : kNoRow, 0, 0);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (block_ks(hb) > 1 && i < 2 * OfS::count)
                    add_product(hb, 2 + i % 2, bt[2 + i % 2][OfS::x(i / 2)], vf[OfS::y(i / 2)], i < 2);
                if (NORM && ND > 1 && i < 2) z_mem[8 * hb + 4 * i] = Z[0][i] + Zr[0][i];
                cut_s((hb + 1) % ND, 0, i);
                rm_frag(pn, i, (hb + 1) % ND);  // (past the last chunk: a buffer of zeros)
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < 12; i++) {
                if (4 + i < 2 * OfS::count && block_ks(hb) > 1) {
                    const int t = 4 + i;
                    add_product(hb, 2 + t % 2, bt[2 + t % 2][OfS::x(t / 2)], vf[OfS::y(t / 2)], false);
                }
                const int x = i % 2, m = i / 2;
                if (last_block && m < OfV::count)
                    O4[x][m % 2] = mfma16(vf[OfV::x(m)], pf[x][OfV::y(m)], O4[x][m % 2]);
                if (i == 10 && block_ks(hb) > 1) add_chunk_sums(hb, 2, 4);
                rm_frag(pn, 4 + i, (hb + 1) % ND);
                if (i < 2) rm_frag(pn, 16 + i, (hb + 1) % ND);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (c == c0 + 4) FTC_STAMP(5);
            if ((kApart || kApartZ) && last_block && (c - c0) % 8 == 7) add_apart();
            o_off = (uint32_t)chunk_row0(c) * o_slb;
            if (c == c0 + 4) FTC_STAMP(6);
        }
    };
    if constexpr (kUnrolled) {
        int c = c0;
        for (; c + 3 <= nchunks; c += 3) {
            chunk_body(c, std::integral_constant<int, 0>());
            chunk_body(c + 1, std::integral_constant<int, ND % 3>());
            chunk_body(c + 2, std::integral_constant<int, 2 * ND % 3>());
        }
        if (c < nchunks) chunk_body(c++, std::integral_constant<int, 0>());
        if (c < nchunks) chunk_body(c++, std::integral_constant<int, ND % 3>());
    } else {
        for (int c = c0; c < nchunks; c++) chunk_body(c, std::integral_constant<int, 0>());
    }
    add_apart();
    store_rows(0);
    store_rows(1);
    FTC_STAMP(15);  // last rows on their way
    if (!NORM && op.s_out && seg == (int)nseg - 1) {
        float *base =
            op.s_out + (int64_t)n * op.so_sn + (int64_t)h * op.so_sh + F * fb + 16 * w + ln;
#pragma unroll
        for (int hb = 0; hb < ND; hb++)
#pragma unroll
            for (int dt = 0; dt < 4; dt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int d = D * hb + state_row(dt, r);
                    if (st_in && d < Dw) base[(int64_t)d * op.so_sd] = S[hb][dt][r];
                }
    }
    // the last consumer of the launch leaves the control block zeroed (as in ftc_wg_kernel.h)
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

template <int ND, int KS2, bool NORM, bool ODD = false>
__global__ __launch_bounds__(512, 2) void scan_tp_kernel(uint32_t *__restrict__ ws_ptr, ScanArgs p) {
    __shared__ __align__(16) char pieces_mem[kTpPieceBytes<3, 3, 3>];
    __shared__ __align__(16) char pt_mem[kTpPtBytes / 2 * (tp_unrolled(ND, 9) ? 3 : 2) + (NORM && ND > 1 ? kTpZBytes : 0)];
    __shared__ __align__(16) float den_mem[NORM ? 3 : 1][NORM ? kChunk : 1][2];
    __shared__ uint32_t order_sh;
    uint32_t which, chain;
    tp_workgroup(p, which, chain);
    scan_tp_body<ND, KS2, NORM, 3, 3, 3, float, ODD>(ws_ptr, p, which, chain, (lds_char *)pieces_mem, (lds_char *)pt_mem,
                                                     den_mem, &order_sh);
}

}  // namespace mfma
}  // namespace ftc
