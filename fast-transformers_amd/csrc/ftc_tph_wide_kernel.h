// The chain-parallel scan of ftc_tph_kernel.h (two scaled fp16 pieces per fp32 value) for states of
// 65 to 128 rows: fp32 rows, widths multiples of 4 on 16-byte boundaries.
//
// A chunk is walked as two positions, one per block of 64 state rows (columns of a and b), as
// scan_tp_kernel<2, ...> does on three bf16 pieces; everything else is the narrow form's: eight
// producer wavefronts cut rows into piece tiles, four consumers hold 16 columns of the state each
// (here 128 rows of them, 32 registers) and share Pt through LDS, one barrier per position.
//
//  * Both blocks of a chunk are scaled alike, so that Pt and Ot are plain sums over the blocks: the
//    ceilings are kept per chunk and the look-ahead runs two positions ahead, the rows of
//    block hb of chunk q + 1 while block hb of chunk q is cut.
//  * |Pt| <= 128 x 16 x 16 = 2^15 is still within fp16 as it is; the state grows per chunk as in
//    the narrow form (32 positions whatever the width).
//  * v is cut once per chunk, with the first block; the consumers keep its fragments.  b^T of tiles
//    2 and 3 is read in phase 2 instead of phase 1, which keeps the consumers within 168
//    registers with twice the state.
//
// What bounds it: a position takes 0.95 us whatever the block (66 matrix instructions per chunk and
// consumer are a quarter of that; the rest is the producers' chain of look-ahead, cut and barrier,
// as in the narrow form), and at 256 workgroups 3.9 TB/s of rows between L2 and memory.  128 chains,
// L=4096, 128 x 128, forward + backward: 1.29 -> 0.98 ms against three bf16 pieces (1.07 with a
// reduction of the look-ahead's maxima per position instead of per chunk); 16 chains, L=4096,
// 100 x 100 253 -> 211 us; 128 chains, L=1000, 128 x 64 217 -> 181.
#pragma once
#include "ftc_tph_kernel.h"

namespace ftc {
namespace mfma {

// KS2: groups of 32 rows in the second block (1: states of 65 to 96 rows)
template <int KS2>
__global__ __launch_bounds__(768, 3) void scan_tph_wide_kernel(uint32_t *__restrict__ ws_ptr, ScanArgs p) {
    constexpr int D = 64, F = 64, ND = 2;      // a block of state rows and of output columns; blocks
    constexpr int T = 512;                     // producer lanes (eight wavefronts)
    constexpr int PF = ND * kTpAhead;          // positions requested ahead
    constexpr int RBA = D * 2, RBV = F * 2;    // bytes per row of an fp16 piece tile
    constexpr int kTileA = kChunk * RBA, kTileV = kChunk * RBV;
    constexpr int kOffB = 2 * kTileA, kOffV = 4 * kTileA;
    constexpr int kBufBytes = 4 * kTileA + 2 * kTileV;
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
    lds_char *const unit_pc = (lds_char *)pieces_mem;
    lds_char *const pt_pc = (lds_char *)pt_mem;
    lds_u32_t *const slots = (lds_u32_t *)slot_mem;

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
    // The chunks walked for their state alone: so0 .. so0 + n1c - 1 (n1c a multiple of kTpAhead).
    // Position v of the walk is block v % 2; v < n1: of a chunk walked for its state alone.
    const int so0 = exchange ? c0 : 0;
    const int n1c = exchange ? (seg + 1 < (int)nseg ? nchunks - c0 : 0) : c0;
    const int n1 = ND * n1c;
    const int nwalk = n1 + ND * (nchunks - c0);  // (position nwalk: a chunk of zeros)
    auto so_chunk = [&](int v) -> int { return exchange ? so0 + n1c - 1 - v / ND : so0 + v / ND; };
    auto walk_chunk = [&](int v) -> int { return v < n1 ? so_chunk(v) : c0 + (v - n1) / ND; };
    constexpr uint32_t kNoRow = 0x80000000u;  // an offset outside every descriptor
    auto block_ks = [](int hb) -> int { return hb == ND - 1 ? KS2 : 2; };
    auto chunk_row0 = [&](int c) -> int { return REV ? rows - kChunk * (c + 1) : kChunk * c; };
    if (tid < 16) slot_mem[tid] = 0;
    Ceilings ce{kExpFloor, kExpOfZeros, kExpOfZeros};
    // Position k has LDS buffer (B0 + k) % 3 and chunk k / 2 of the walk has slot (S0 + k / 2) % 3,
    // such that the walk proper begins with number 0 of either: its loop is unrolled three chunks.
    const int B0 = (3 - n1 % 3) % 3, S0 = (3 - n1c % 3) % 3;
    auto next_buf = [](int b) -> int { return b == 2 ? 0 : b + 1; };

    if (producer) {
        // =========================== producers ===========================
        const int ptid = (wave - 4) * 64 + lane;
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
        // One quad (four columns of one row) of every operand per lane and position; a lane whose
        // columns lie beyond the width asks outside the descriptor and cuts zeros.
        static_assert(LA == 1 && LV == 1 && QA == QV, "one quad per lane");
        const int prow = ptid / QA, pc4 = ptid % QA;
        const bool second_in = D + 4 * pc4 < Dw;  // (the first block's columns all exist)
        const bool v_in = 4 * pc4 < fw;
        const uint32_t a_goff = (uint32_t)prow * a_slb + 16u * pc4, b_goff = (uint32_t)prow * b_slb + 16u * pc4,
                       v_goff = (uint32_t)prow * v_slb + 16u * pc4;
        const int a_waddr = TpSwizzle<RBA>::addr(prow, 8 * pc4),
                  b_waddr = TpSwizzle<RBA>::addr(prow, 2 * b_tile_column(4 * pc4)),
                  v_waddr = TpSwizzle<RBV>::addr(prow, 8 * pc4);
        struct Raw {
            u32x4 a, b, v;
        };
        Raw raw[PF];  // (v: of first blocks)
        // (every request every time, as in scan_tph_kernel)
        auto fetch = [&](Raw &r, int v, int hb) {  // v: position of the walk, hb = v % 2
            const int row0 = v < nwalk ? chunk_row0(walk_chunk(v)) : -2 * kChunk;
            const int row0_x = v >= n1 ? row0 : -2 * kChunk;
            const bool in = hb == 0 || second_in;
            const uint32_t col = 4u * D * hb;
            r.a = __builtin_amdgcn_raw_buffer_load_b128(
                a_rs, in ? a_goff + col + (uint32_t)row0_x * a_slb : kNoRow, 0, 0);
            r.b = __builtin_amdgcn_raw_buffer_load_b128(
                b_rs, in ? b_goff + col + (uint32_t)row0 * b_slb : kNoRow, 0, 0);
            if (hb == 0)
                r.v = __builtin_amdgcn_raw_buffer_load_b128(
                    v_rs, v_in ? v_goff + (uint32_t)row0 * v_slb : kNoRow, 0, 0);
        };
        // (the maxima of a chunk's first block wait in registers: one reduction per chunk)
        float ma = 0.f, mb = 0.f, mv = 0.f;
        auto look_ahead = [&](const Raw &r, int k, int chunk, int hb) {
            ma = max_abs4(r.a, hb == 0 ? 0.f : ma), mb = max_abs4(r.b, hb == 0 ? 0.f : mb);
            if (hb == 0) mv = max_abs4(r.v, 0.f);
            else raise_slot(slots, k, chunk, ce, ma, mb, mv, lane);
        };
        auto cut = [&](const Raw &r, int buf, bool own, int hb) {
            lds_char *const pc = unit_pc + buf * kBufBytes;
            if (own) cut_quad_to_lds(r.a, ce.scale_a(), pc, kTileA, a_waddr);
            cut_quad_to_lds(r.b, ce.scale_b(), pc + kOffB, kTileA, b_waddr);
            if (hb == 0) cut_quad_to_lds(r.v, ce.scale_v(), pc + kOffV, kTileV, v_waddr);
            if (!own) asm volatile("" ::"v"(r.a));
        };
#pragma unroll
        for (int j = 0; j < PF; j++) fetch(raw[j], j, j % ND);
        wg_barrier();  // the slots are zero
        look_ahead(raw[0], S0, 0, 0);
        look_ahead(raw[1], S0, 0, 1);
        wg_barrier();  // the slot of the first chunk is complete
        // Barrier number k (k = 0: before the consumers' first position; k >= 1: in the
        // middle of position k - 1) finds position k cut and, where k is odd, the slot of the
        // chunk after it complete.  The last one finds a block of zeros.
        int buf = B0, slot = S0;
        auto step = [&](int v, int j, bool own, bool ahead, bool more) {
            const int hb = j % ND;
            if (hb == 0) read_slot(slots, slot, ce);
            if (ahead) look_ahead(raw[(j + ND) % PF], next_buf(slot), v / ND + 1, hb);
            cut(raw[j], buf, own, hb);
            if (more) fetch(raw[j], v + PF, hb);
            buf = next_buf(buf);
            if (hb == ND - 1) slot = next_buf(slot);
            wg_barrier();
            __builtin_amdgcn_sched_barrier(0);  // one position at a time, in this order
        };
        for (int v = 0; v < n1; v += PF) {
#pragma unroll
            for (int j = 0; j < PF; j++) step(v + j, j, false, true, true);
        }
        // (whole trips in the loop, the rest after it)
        int v = n1;
        for (; v + PF <= nwalk + 1; v += PF) {
#pragma unroll
            for (int j = 0; j < PF; j++) step(v + j, j, true, true, true);
        }
        // (what lies two positions on after the last but one of these is past the walk)
#pragma unroll
        for (int j = 0; j < PF - 1; j++) {
            if (v + j > nwalk) return;
            step(v + j, j, true, j + ND < PF, false);
        }
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
    uint32_t o_lane[2];
#pragma unroll
    for (int x = 0; x < 2; x++)
        o_lane[x] = (uint32_t)(16 * (x ^ ih) + ln) * o_slb + 4u * (16 * w + 4 * g);
    const bool o_in = 16 * w + 4 * g < fw;  // (columns beyond the width are not stored)

    f32x4 S[ND][4];  // the slab, block by block, in units of 2^Ucur
#pragma unroll
    for (int hb = 0; hb < ND; hb++)
#pragma unroll
        for (int dt = 0; dt < 4; dt++) S[hb][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    int Ucur = 0;
    constexpr int kPa[3] = {1, 0, 0}, kPb[3] = {0, 1, 0};  // piece products, smallest first
    auto state_row = [&](int dt, int r) -> int { return 32 * (dt / 2) + 8 * g + 4 * (dt % 2) + r; };
    const bool st_in = 16 * w + ln < fw;
    auto scale_block = [&](int hb, int e) {  // S <- S 2^e
#pragma unroll
        for (int dt = 0; dt < 2 * block_ks(hb); dt++)
#pragma unroll
            for (int r = 0; r < 4; r++) S[hb][dt][r] = __builtin_amdgcn_ldexpf(S[hb][dt][r], e);
    };
    auto add_caller_state = [&]() {  // in units of 2^Ucur
        const float *base =
            op.s0 + (int64_t)n * op.s0_sn + (int64_t)h * op.s0_sh + F * fb + 16 * w + ln;
#pragma unroll
        for (int hb = 0; hb < ND; hb++)
#pragma unroll
            for (int dt = 0; dt < 2 * block_ks(hb); dt++) {
                float x[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int d = D * hb + state_row(dt, r);
                    const bool in = st_in && d < Dw;
                    x[r] = *(in ? base + (int64_t)d * op.s0_sd : op.s0);
                    x[r] = in ? __builtin_amdgcn_ldexpf(x[r], -Ucur) : 0.f;
                }
                S[hb][dt] += f32x4{x[0], x[1], x[2], x[3]};
            }
    };

    Frag af[2][2][2], bfr[2][2], bt[4][2], vf[2];
    // row-major fragment number i of a position (12: b for the quadrant first, then a)
    auto rm_frag = [&](const lds_char *pc, int i, int hb) {
        const int k = i % 2, ks = (i / 2) % 2, x = i / 4;
        if (ks >= block_ks(hb)) return;
        if (x == 0)
            bfr[ks][k] = lds_frag8x2(pc + k * kTileA + b_addr[ks][0], pc + k * kTileA + b_addr[ks][1]);
        else
            af[x - 1][ks][k] = lds_frag16(pc + k * kTileA + a_addr[x - 1][ks]);
    };
    // position-major fragments: v (first blocks), number i of b^T (8, tile by tile)
    auto v_frag = [&](const lds_char *pc, int k) -> Frag {
        return lds_frag_tr(pc + k * kTileV + vt_addr[0], pc + k * kTileV + vt_addr[1]);
    };
    auto bt_frag_into = [&](Frag (&btx)[4][2], const lds_char *pc, int i, int hb) {
        const int dt = i / 2, k = i % 2;
        if (dt / 2 >= block_ks(hb)) return;  // tiles 2, 3: rows 32 .. 63 of the block
        btx[dt][k] = lds_frag_tr(pc + k * kTileA + bt_addr[dt][0], pc + k * kTileA + bt_addr[dt][1]);
    };
    wg_barrier();  // the slots are zero
    wg_barrier();  // the slot of the first chunk is complete
    wg_barrier();  // barrier 0: position 0 is cut
    read_slot(slots, S0, ce);
    Ucur = ce.state_exp();
    if (op.s0 && !exchange) add_caller_state();
    if (n1 > 0) {
        // ---- the first n1 positions of the walk: state update only, skewed by one position:
        // while the matrix instructions of position k - 1 run, the fragments of position k arrive ----
        int buf = B0, slot = S0;
        Frag bt2[4][2] = {}, vfs[2][2] = {};  // (the first round multiplies zeros)
        for (int c = 0; c < n1; c += PF) {
#pragma unroll
            for (int j = 0; j < PF; j++) {
                const lds_char *pc = unit_pc + buf * kBufBytes;
                const int q = (j / ND) % 2;
                if (j % ND == 0) {
                    read_slot(slots, slot, ce);  // the ceilings of this chunk, multiplied from the next position on
                } else if (ce.state_exp() != Ucur) {
                    const int e = Ucur - ce.state_exp();
                    scale_block(0, e), scale_block(1, e);
                    Ucur -= e;
                }
#pragma unroll
                for (int i = 0; i < 12; i++) {
                    if (j % ND == 0) {
                        if ((i % 4) / 2 < KS2)
                            S[1][i % 4] = mfma16h(bt2[i % 4][kPa[i / 4]], vfs[1 - q][kPb[i / 4]], S[1][i % 4]);
                        if (i < 2) vfs[q][i] = v_frag(pc, i);
                        else if (i < 10) bt_frag_into(bt, pc, i - 2, 0);
                    } else {
                        S[0][i % 4] = mfma16h(bt[i % 4][kPa[i / 4]], vfs[q][kPb[i / 4]], S[0][i % 4]);
                        if (i < 8) bt_frag_into(bt2, pc, i, 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                buf = next_buf(buf);
                if (j % ND == ND - 1) slot = next_buf(slot);
                wg_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the last of these positions (the second block of an odd chunk)
#pragma unroll
        for (int i = 0; i < 12; i++)
            if ((i % 4) / 2 < KS2)
                S[1][i % 4] = mfma16h(bt2[i % 4][kPa[i / 4]], vfs[1][kPb[i / 4]], S[1][i % 4]);
        read_slot(slots, 0, ce);  // the ceilings of our own first chunk
    }
    if (exchange) {
        // ---- the sum of this segment's rows goes out, the state before the segment comes in ----
        const uint32_t total_units = (uint32_t)p.total_waves;
        gfloat *const sums = (gfloat *)(hdr + kControlBytes / 4);
        StateExchange<ND, 1> xch(flags, sums, 4u * total_units,
                                (uint32_t)w * total_units + chain_id * nseg + (uint32_t)seg, seg,
                                (int)nseg, p.group, lane);
        f32x16 Sx[ND][1], X[ND][1];
#pragma unroll
        for (int hb = 0; hb < ND; hb++)
#pragma unroll
            for (int dt = 0; dt < 4; dt++)
#pragma unroll
                for (int r = 0; r < 4; r++) Sx[hb][0][4 * dt + r] = __builtin_amdgcn_ldexpf(S[hb][dt][r], Ucur);
        if (n1 > 0) xch.publish_sum(Sx);
        xch.gather(Sx, X);
        if (xch.failed && lane == 0)
            __hip_atomic_store(hdr + kHdrError, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // the units of the first chunk of the second pass (its ceilings are already known)
        Ucur = ce.state_exp();
#pragma unroll
        for (int hb = 0; hb < ND; hb++)
#pragma unroll
            for (int dt = 0; dt < 4; dt++)
#pragma unroll
                for (int r = 0; r < 4; r++) S[hb][dt][r] = __builtin_amdgcn_ldexpf(X[hb][0][4 * dt + r], -Ucur);
        if (op.s0) add_caller_state();
    }
    // (our own first chunk is cut)
#pragma unroll
    for (int i = 0; i < 12; i++) rm_frag(unit_pc, i, 0);
    // ---- the walk proper ----
    // `ce` holds the ceilings of the chunk at hand, Ucur the units of S.  dU < 0: the
    // state's units rise by -dU with this chunk (a block is rescaled once all of it has been cut).
    int dU = Ucur - ce.state_exp();
    int s = 0;  // S is cut as S 2^(dU - s)
    if (dU != 0) {
        scale_block(0, dU), scale_block(1, dU);
        Ucur -= dU;
        dU = 0;
    }
    {
        float m = 0.f;
#pragma unroll
        for (int t = 0; t < 4 * ND; t++) {
            const f32x4 x = S[t / 4][t % 4];
            m = fmaxf(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))), m);
        }
        while (s < 100 && __builtin_amdgcn_ballot_w64(m > pow2_field(127 + 14 + s)) != 0) s++;
    }
    float kappa = pow2_field(127 + dU - s);  // scale of the cut of S
    bool plain_cut = dU - s == 0;            // ... which is one as a rule: a cheaper cut
    int s_cut = s;                           // ... and the s that went into it
    float mS = 0.f;                          // largest |S| seen while cutting
    Frag sf[2][2];
    // tile 2 ks + u of block hb -> words 2 u, 2 u + 1 of the fragments of k-step ks (`track`: see
    // scan_tph_kernel; one chunk in three)
    auto cut_s = [&](int hb, int ks, int u, bool track) {
        const f32x4 x = S[hb][2 * ks + u];
        if (track)
            mS = fmaxf(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3]))), mS);
        if (plain_cut)
            cut_quad_f16_unscaled(x[0], x[1], x[2], x[3], sf[ks][0].w[2 * u], sf[ks][0].w[2 * u + 1],
                                  sf[ks][1].w[2 * u], sf[ks][1].w[2 * u + 1]);
        else
            cut_quad_f16(x[0], x[1], x[2], x[3], kappa, sf[ks][0].w[2 * u], sf[ks][0].w[2 * u + 1],
                         sf[ks][1].w[2 * u], sf[ks][1].w[2 * u + 1]);
    };
    cut_s(0, 0, 0, true);
    cut_s(0, 0, 1, true);

    // Ot_w of the chunk before in the units of that chunk (exponent Xo), and where its rows
    // go (before the first chunk: nowhere)
    f32x4 O[2];
#pragma unroll
    for (int x = 0; x < 2; x++) O[x] = f32x4{0.f, 0.f, 0.f, 0.f};
    int Xo = 0;
    uint32_t o_off = 0x80000000u;
    auto store_rows = [&](int x) {
        buffer_store4(o_rs, o_in ? o_off + o_lane[x] : kNoRow, __builtin_amdgcn_ldexpf(O[x][0], Xo),
                      __builtin_amdgcn_ldexpf(O[x][1], Xo), __builtin_amdgcn_ldexpf(O[x][2], Xo),
                      __builtin_amdgcn_ldexpf(O[x][3], Xo));
    };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 P = zero;  // the quadrant, summed over the blocks
    // One position: block HB of chunk c, in LDS buffer B, the chunk's slot and Pt tile number C
    // (compile-time numbers, as in scan_tph_kernel)
    auto position = [&](int c, auto buffer_number, auto block_number, auto chunk_number) {
        constexpr int B = decltype(buffer_number)::value, BN = (B + 1) % 3;
        constexpr int HB = decltype(block_number)::value, HN = 1 - HB;
        constexpr int C = decltype(chunk_number)::value, CN = (C + 1) % 3;
        constexpr bool last = HB == ND - 1;
        const lds_char *pc = unit_pc + B * kBufBytes;
        const lds_char *pn = unit_pc + BN * kBufBytes;
        lds_char *const ptc = pt_pc + C * (2 * kTileP);
        Frag pf[2][2];
        __builtin_amdgcn_sched_barrier(0);
        // phase 1: (1) the quadrant in turn with (2b) Ot_w += S_w^T a^T for rows 0 .. 31 of the
        // block; underneath: the rows of the chunk before go out, tiles 2, 3 of the block's
        // state are cut into pieces, position-major reads
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int m = i % 3, ks = i / 3, x = i % 2, mo = i / 2;
            if (HB == 0 && i < 2) store_rows(i);
            if (ks < block_ks(HB))
                P = mfma16h(bfr[ks][kPa[m]], af[0][ks][kPb[m]], i == 0 && HB == 0 ? zero : P);
            O[x] = mfma16h(sf[0][kPa[mo]], af[x][0][kPb[mo]], mo == 0 && HB == 0 ? zero : O[x]);
            if ((i == 1 || i == 3) && block_ks(HB) > 1) cut_s(HB, 1, i / 2, C == 0);
            if (HB == 0 && i < 2) vf[i] = v_frag(pc, i);
            if (i >= 2) bt_frag_into(bt, pc, i - 2, HB);
            __builtin_amdgcn_sched_barrier(0);
        }
        // all of the block is cut: it takes the units of this chunk; with the last one s follows
        // the state's size
        if (dU != 0) {
            scale_block(HB, dU);
            if (last) {
                mS = __builtin_amdgcn_ldexpf(mS, dU);
                s = max(0, s + min(dU, 0));
                Ucur -= dU;
            }
        }
        if (last && C == 0) {
            while (s < 100 && __builtin_amdgcn_ballot_w64(mS > pow2_field(127 + 14 + s)) != 0) s++;
            mS = 0.f;
        }
        __builtin_amdgcn_sched_barrier(0);
        // phase 2: (2b) for rows 32 .. 63 in turn with (3) S_w += b^T v_w for tiles 0 and 1;
        // underneath: b^T of tiles 2 and 3 and, with the last block, the quadrant is masked, cut
        // and handed to the others
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int x = i % 2, m = i / 2;
            if (block_ks(HB) > 1) O[x] = mfma16h(sf[1][kPa[m]], af[x][1][kPb[m]], O[x]);
            S[HB][i % 2] = mfma16h(bt[i % 2][kPa[m]], vf[kPb[m]], S[HB][i % 2]);
            if (i < 4) bt_frag_into(bt, pc, 4 + i, HB);
            if (i == 1 && last) {
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
        wg_barrier();
        // The next position is cut; with the last block all of Pt is in LDS and the next chunk's
        // slot complete.
        // phase 3: (3) for tiles 2 and 3, then (2a) Ot_w += v_w^T Pt; underneath: the next
        // position's row-major fragments and tiles 0, 1 of its block of S_w cut into pieces
        u32x4 slot_next = {0, 0, 0, 0};
        int Xc = 0;
        if (last) {
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int k = 0; k < 2; k++) pf[x][k] = lds_frag16(ptc + k * kTileP + pt_raddr[x]);
            Xc = ce.out_exp();
            slot_next = *(const lds_vec4 *)(slots + 4 * CN);
            if (s_cut != 0) {  // (rare: the state has grown beyond 2^14 units)
                const float r_cut = pow2_field(127 + s_cut);
                O[0] *= r_cut;
                O[1] *= r_cut;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int m = i / 2;
            if (block_ks(HB) > 1) S[HB][2 + i % 2] = mfma16h(bt[2 + i % 2][kPa[m]], vf[kPb[m]], S[HB][2 + i % 2]);
            rm_frag(pn, 2 * i, HN);
            rm_frag(pn, 2 * i + 1, HN);
            if (!last && (i == 1 || i == 3)) cut_s(HN, 0, i / 2, C == 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (!last) return;
        // the ceilings of the next chunk
        ce.Ea = max(kExpFloor, (uint32_t)__builtin_amdgcn_readfirstlane(slot_next.x) & 0xffu);
        ce.Wb = max(ce.Wb, (uint32_t)__builtin_amdgcn_readfirstlane(slot_next.y));
        ce.Wv = max(ce.Wv, (uint32_t)__builtin_amdgcn_readfirstlane(slot_next.z));
        // (dU > 0: small values after nothing but zeros; the state's units fall, so s rises)
        dU = Ucur - ce.state_exp();
        s += max(dU, 0);
        kappa = pow2_field(127 + dU - s);
        plain_cut = dU - s == 0;
        s_cut = s;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 6; i++) {
            const int x = i % 2, m = i / 2;
            O[x] = mfma16h(vf[kPa[m]], pf[x][kPb[m]], O[x]);
            if (i == 1 || i == 3) cut_s(0, 0, i / 2, CN == 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        o_off = (uint32_t)chunk_row0(c) * o_slb;
        Xo = Xc;
    };
    auto chunk = [&](int c, auto number) {
        constexpr int C = decltype(number)::value;
        position(c, std::integral_constant<int, 2 * C % 3>(), std::integral_constant<int, 0>(), number);
        position(c, std::integral_constant<int, (2 * C + 1) % 3>(), std::integral_constant<int, 1>(), number);
    };
    {
        int c = c0;
        for (; c + 3 <= nchunks; c += 3) {
            chunk(c, std::integral_constant<int, 0>());
            chunk(c + 1, std::integral_constant<int, 1>());
            chunk(c + 2, std::integral_constant<int, 2>());
        }
        if (c < nchunks) chunk(c++, std::integral_constant<int, 0>());
        if (c < nchunks) chunk(c++, std::integral_constant<int, 1>());
    }
    store_rows(0);
    store_rows(1);
    if (op.s_out && seg == (int)nseg - 1) {
        float *base =
            op.s_out + (int64_t)n * op.so_sn + (int64_t)h * op.so_sh + F * fb + 16 * w + ln;
#pragma unroll
        for (int hb = 0; hb < ND; hb++)
#pragma unroll
            for (int dt = 0; dt < 2 * block_ks(hb); dt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int d = D * hb + state_row(dt, r);
                    if (st_in && d < Dw) base[(int64_t)d * op.so_sd] = __builtin_amdgcn_ldexpf(S[hb][dt][r], Ucur);
                }
    }
    // the last consumer of the launch leaves the control block zeroed
    if (exchange) {
        const uint32_t total_units = (uint32_t)p.total_waves;
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

}  // namespace mfma
}  // namespace ftc
