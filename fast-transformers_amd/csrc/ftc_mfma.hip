// Host side of the MFMA scan (kernel: ftc_mfma_kernel.h): which scans qualify, how L is cut
// into segments, workspace size, and the launch.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdlib>

#include "ftc_wg_kernel.h"

namespace ftc {
using namespace mfma;
namespace {

struct MfmaPlan {
    int nseg, seg_len;
    int64_t waves, workspace_bytes;
};

// all-fp32 scans of these widths run as workgroups of F / 32 wavefronts (ftc_wg_kernel.h)
bool use_wg_kernel(int64_t D, int64_t F, int nscans, int64_t L, bool all_f32) {
    if (!all_f32 || !scan_wg_covers((int)D, (int)F)) return false;
    if (tuning().wg >= 0) return tuning().wg != 0;  // tuning aid
    // Measured: a single scan over long chains (the forward) is 2-7 % faster in workgroup
    // form (cfg3 forward 331 us against 349, N=8, H=16, L=4096: 164 against 177); launches of
    // three scans and short chains are faster with one wavefront per segment.
    return nscans == 1 && L >= 128 * kChunk && D == 64 && F == 64;
}

// Row widths that the chain-parallel kernel takes (ftc_tp_kernel.h): states of 16 x 16 to
// 128 x 128, walked in blocks of 64 rows, with one workgroup per block of 64 output columns;
// widths that are multiples of 4 (a lane's 16 bytes lie wholly inside a row or wholly outside).
// (`forced`: a part of a scan that the caller has split because only this kernel takes it;
// then any multiple of 4 will do)
// `odd`: fp32 rows of any width on 4-byte boundaries, which the kernels read and write where they lie: the
// fp16-piece kernel with states of up to 64 rows, the one on three bf16 pieces (`forced`) of up to 128.
bool tp_widths(int64_t D, int64_t F, bool forced = false, bool odd = false) {
    if (odd) return D >= 8 && D <= (forced ? 128 : 64) && F >= 8 && F <= 512;
    const int64_t least = forced ? 4 : 16;
    return D >= least && D <= 128 && F >= least && F <= 512 && D % 4 == 0 && F % 4 == 0;
}
int64_t tp_fblocks(int64_t F) { return (F + 63) / 64; }

// whether the kernels that split L take fp32 rows of these widths (as column slices, if need be)
bool mfma_scan_supported_widths(int64_t D, int64_t F) {
    int widths[kMfmaMaxSlices];
    return mfma_slice_widths(D, F, widths) > 0;
}

// segments that a chain may be cut into without an exchange: as many as one round of workgroups has room for, up to four
int64_t round_segments(int64_t units) { return std::max<int64_t>(1, std::min<int64_t>(4, 256 / units)); }
// ... which have to fill half the GPU where other kernels take the widths as well
constexpr int64_t kHalfTheGpu = 128;

// all-fp32 scans can run one workgroup per chain (and block of 64 output columns) with no
// split of L (ftc_tp_kernel.h).  `units`: chains x scans x column blocks; `wide`: a state
// other than 64 x 64, for which the kernels that split L are half as fast as for 64 x 64;
// `others`: one of those kernels takes this shape (else the choice is the VALU kernel).
// Returns the number of segments per chain (0: another kernel takes the launch).
int tp_kernel_segments(int64_t units, int64_t L, bool wide, bool others, bool long_chains = false,
                       bool cut_long = false, int64_t most_units = 512, int64_t brief_chunks = 0) {
    // a chain is walked by one workgroup from end to end: beyond 256 chunks the split of L
    // of the other kernels is faster, and its segment sums also keep the rounding of a long
    // running state in check (`long_chains`: the caller knows better, see tp_plan_compute)
    if (L > (long_chains ? 1024 : 256) * kChunk) return 0;
    // One workgroup per CU at a time.  A workgroup that takes a whole chain reads every row
    // once; with fewer chains than CUs a chain is cut into up to four segments whose
    // workgroups each rebuild the state before their segment by themselves (a state-only
    // chunk costs a bit more than half of a full one), as long as that fills at least half the GPU.
    const int64_t total_chunks = (L + kChunk - 1) / kChunk;
    int nseg = (int)std::max<int64_t>(1, std::min(round_segments(units), total_chunks));
    if (tuning().tp_segs >= 0) nseg = std::max(1, std::min(tuning().tp_segs, 16));  // tuning aid
    if (tuning().tp >= 0) return tuning().tp != 0 ? nseg : 0;                       // tuning aid
    // Measured (forward, us, N=10 H=8): cfg2 (L=1000) 30 against 42 for the kernels that split
    // L and exchange states; L=3000: 75 against 84; L=4096: 100 against 108; L=8192: 201
    // against 201 -- cut chains pay off while the chunks that a workgroup walks for its
    // state alone are few.
    if (nseg > 1 && total_chunks > 128) {
        if (!wide && !long_chains) return 0;
        if (!wide) nseg = 1;
        // (`cut_long`: shapes that never exchange keep their cuts: 32 x 128, 64 chains, L=8192,
        // forward: 190 us in two segments against 219 whole and 206 on the kernels that split L)
        if (!cut_long) nseg = 1;
    }
    // (wide states: the other kernels run them as column slices that each repeat the chunk
    // product, and lose at any number of rounds; on a quarter of the CUs they still win, N=1,
    // H=8, L=2048, 128 x 128 forward: 52 against 91 us.  The VALU kernel loses always.)
    // (chains of up to `brief_chunks` chunks at any number, see tp_plan_compute)
    const bool brief = total_chunks <= brief_chunks;
    if (wide) return !others || brief || units * nseg >= kHalfTheGpu ? nseg : 0;
    // Beyond `most_units` workgroups the other kernels win again (short chains: there every
    // chain has its own wavefront, all resident at once, and nothing is split either).
    return (brief || units * nseg >= (long_chains ? 112 : kHalfTheGpu)) && units <= most_units ? nseg : 0;
}

// Plans depend on the sizes alone and a caller repeats the same sizes call after call (the
// segment search walks up to 4096 candidates for a long sequence): the last plans of every
// thread are kept, keyed by their arguments and by the generation of the tuning variables.
template <typename Value>
struct PlanMemo {
    static constexpr int kEntries = 32;
    struct Entry {
        int64_t key[8];
        uint64_t generation;
        Value value;
    };
    Entry entry[kEntries] = {};
    template <typename Compute>
    Value get(const int64_t (&key)[8], Compute compute) {
        uint64_t h = 1469598103934665603ull;
        for (int64_t k : key) h = (h ^ (uint64_t)k) * 1099511628211ull;
        Entry &e = entry[h % kEntries];
        const uint64_t generation = tuning().generation;
        bool hit = e.generation == generation;
        for (int i = 0; i < 8 && hit; i++) hit = e.key[i] == key[i];
        if (!hit) {
            e.value = compute();
            for (int i = 0; i < 8; i++) e.key[i] = key[i];
            e.generation = generation;
        }
        return e.value;
    }
};

// Where to cut a chain of `chunks` chunks into (at most) `nseg` segments for the
// chain-parallel kernel.  The workgroup of a segment first rebuilds the state before its
// segment from the chunks in front of it, so later segments are made shorter until all
// workgroups finish together: the starts (multiples of `step` chunks) that minimise the longest
// workgroup.  `state_only`: the time of a chunk walked for its state alone, against one that also
// produces rows.
// Returns the number of segments; start[0 .. n] filled (start[n] = chunks).
int tp_segment_starts(int64_t chunks, int nseg, int32_t *start, int step, double state_only) {
    const int groups = (int)((chunks + step - 1) / step);
    nseg = std::max(1, std::min(std::min(nseg, groups), kMaxTpSegments));
    if (tuning().tp_ratio >= 0) state_only = tuning().tp_ratio;  // tuning aid
    auto chunk = [&](int g) -> int { return (int)std::min<int64_t>(step * g, chunks); };
    // best[s][g]: smallest achievable longest time of segments s .. nseg-1 when segment s
    // starts at group g (dynamic programme from the last segment back)
    constexpr int kMaxGroups = 64;
    if (groups > kMaxGroups || nseg == 1) {
        start[0] = 0, start[1] = (int32_t)chunks;
        return 1;
    }
    double best[kMaxTpSegments + 1][kMaxGroups + 1];
    int next[kMaxTpSegments + 1][kMaxGroups + 1];
    for (int s = 0; s <= nseg; s++)
        for (int g = 0; g <= groups; g++) best[s][g] = 1e30, next[s][g] = groups;
    best[nseg][groups] = 0.0;
    for (int s = nseg - 1; s >= 0; s--)
        for (int g = s; g < groups; g++)
            for (int e = g + 1; e <= groups - (nseg - 1 - s); e++) {
                const double own = state_only * chunk(g) + (chunk(e) - chunk(g));
                if (own >= best[s][g]) break;  // (it grows with e)
                const double t = std::max(own, best[s + 1][e]);
                if (t < best[s][g]) best[s][g] = t, next[s][g] = e;
            }
    int g = 0;
    for (int s = 0; s < nseg; s++) {
        start[s] = chunk(g);
        g = next[s][g];
    }
    start[nseg] = (int32_t)chunks;
    return nseg;
}

// The cuts of a launch of the chain-parallel kernel with a state of D rows.  `scaled`: on two fp16
// pieces, where a chunk walked for its state alone takes 0.6 of the others (0.75 against 1.3 us with
// every workgroup streaming rows); on three bf16 pieces 0.45 where a state of 33 to 64 rows writes fp32
// results, 0.55 otherwise and for two segments of odd widths or of bf16 rows (128 chains, L=1088, forward
// 25.2 against 26.0 at 0.45).  Three pieces of fp32 rows may start half of what the producers request
// ahead (kTpAhead) further on (kHalfTrips; up to 64 chunks, a longer search for a smaller share of a
// segment beyond).  Measured against 0.6 and steps of kTpAhead for all, whose last one counted as whole, 22
// shapes drawn for each, geometric means of the time: fused attention of 64 x 64 0.928 (at 0.55: 0.940),
// odd widths 0.936; 80 chains, L=1000, fused: 38.5 -> 35 us; bf16 rows forward, 64 chains, L=1000: 17.6 ->
// 16.8, 49, L=1588: 23.7 -> 21.7; backward, 20 chains, L=900: 20.5 -> 19.2, 31, L=407: 15.0 -> 13.0.
// (Kept like the plans: the search takes the host up to 2 us.)
struct TpCuts {
    int nseg;
    int32_t start[kMaxTpSegments + 1];
};
TpCuts tp_cuts(int64_t D, bool scaled, bool fp32_rows, bool fp32_results, bool fused, int nseg, int64_t chunks) {
    const int step = !scaled && fp32_rows && chunks <= 64 ? kTpAhead / 2 : kTpAhead;
    const bool light = D > 32 && D <= 64 && fp32_results && (fused || nseg > 2);
    const int percent = scaled ? 60 : light ? 45 : 55;
    static thread_local PlanMemo<TpCuts> memo;
    const int64_t key[8] = {chunks, nseg, step, percent, 0, 0, 0, 0};
    return memo.get(key, [&]() {
        TpCuts c = {};
        c.nseg = tp_segment_starts(chunks, nseg, c.start, step, 0.01 * percent);
        return c;
    });
}

// Longer chains on few CUs: the chain-parallel kernel with an exchange of segment sums.  A
// chain is cut into as many equal segments as fill the GPU (one workgroup each); a workgroup
// walks its own chunks twice, first for their state alone.  Returns the number of chunks per
// segment (0: not this way) and the number of segments in *nseg.
// (`most_fours`: the workgroups up to which a chain has a segment for every four chunks, see below)
int tp_exchange_segments(int64_t units, int64_t L, bool wide, int64_t most_fours, int *nseg) {
    const int64_t total_chunks = (L + kChunk - 1) / kChunk;
    *nseg = 0;
    if (tuning().tpx == 0) return 0;  // tuning aid
    // Up to 64 chunks the cut chains without an exchange are as fast (cfg2: 30 us either way)
    // and need no workspace -- unless the chains are so few that four or more segments of each
    // fit one round of workgroups: those win from 24 chunks on, also against the kernels that
    // split L (64 x 64 forward, us, this way / before: 16 chains, L=2048: 28 / 44, L=1024:
    // 21 / 28; 8 chains, L=2048: 23 / 31; 32 chains, L=2048: 34 / 42; backward of 8 chains,
    // L=2048: 31 / 38, of 4: 26 / 37; 128 x 128 forward, 16 chains, L=2048: 50 / 81).
    const bool force = tuning().tpx_segs >= 2;  // tuning aid: also where the rules below say no
    const bool brief = total_chunks <= 64;
    // (not for one or two workgroups' worth of chains, 22 against 21 us, and from 33 on only
    // from 48 chunks: backward of 16 chains, L=1024: 34 against 26 cut in five without an exchange)
    if (!force && (units < 1 || total_chunks < 24)) return 0;
    if (!force && brief && (units < 3 || units > 64 || (units > 32 && total_chunks < 48))) return 0;
    // (more workgroups than CUs: only where chains are too long to walk whole)
    if (!force && units > 128 && total_chunks <= 256) return 0;
    int64_t want = 256 / units;
    // the number of segments with the shortest estimated time, rounds x (a segment walked
    // twice + the exchange and the start, in chunks' time)
    // (wide states: twelve chunks' time for those -- with six, 128 x 128 backward of 16 chains,
    // L=4096, went into three rounds of 16-chunk segments, 202 us, where two segments take 185)
    auto shortest = [&](double twice, double fixed) {
        double best = 1e30;
        for (int64_t n = std::max<int64_t>(2, (total_chunks + 255) / 256); n <= 64; n++) {
            const int64_t c = ((total_chunks + n - 1) / n + kTpAhead - 1) / kTpAhead * kTpAhead;
            const int64_t rounds = (units * ((total_chunks + c - 1) / c) + 255) / 256;
            const double t = (double)rounds * (twice * (double)c + fixed);
            if (t < best - 1e-9) best = t, want = n;
        }
    };
    if (wide) {
        // workgroups that do not fill whole rounds of 256 (the first walk at 0.4 of the cost)
        if (units * want != 256) shortest(1.4, 12.0);
    } else if (want < 2 || (total_chunks + want - 1) / want > 256) {
        // 64 x 64 with no single round of segments of at most 256 chunks: a few rounds still
        // beat the kernels that split L while those have no more than a wavefront or two per
        // SIMD to run (backward, ms, this way with the segments chosen here / split L:
        // N*H = 16, L=65536: 0.71 / 0.79; 32, L=32768: 0.72 / 0.82; 64, L=16384: 0.80 / 0.91;
        // 128, L=16384: 1.36 / 1.56; but 256, L=16384: 2.70 / 2.60.  Ten segments at N*H = 16
        // against 8: 0.83, 11: 0.82, 16: 0.79 -- the last round wants to be full).
        if (!force && units > 384) return 0;
        shortest(1.0, 40.0);
    }
    // Two segments of up to 64 chunks lose to chains cut in two without an exchange, whose
    // first workgroup walks its part once (forward, 96 chains, L=4096: 117 against 100 us; 128
    // chains: 145 against 128; backward of 32 chains: 110 against 95); with three segments the
    // exchange wins again (backward of 24 chains: 83 against 86; forward of 64: 73 against 88).
    // Wider states the same (64 x 128 forward, 64 chains, L=4096: 116 against 104; 128 x 128
    // backward of 16 chains: 204 against 186).
    if (!force && want == 2 && total_chunks <= 128) return 0;
    // segments of at least four chunks (one or two chains, L=4096: 32 segments 21.5 us, 16: 25.1), the last one
    // of what is left (forward, us, as many segments as there are whole fours of chunks, which makes eight of the four
    // a segment / this way: 8 chains, L=800 20.7 / 17.9, 1 chain, L=6150 24.8 / 19.9; backward of 4, L=1600 31 / 24).
    // Not where that were more than `most_fours` workgroups, which wait for each other longer than they walk: a state of
    // up to 64 rows 192 of them, whichever kernel and widths (eight chunks a segment / four: 64 x 64, 101 chunks, 208
    // workgroups 24.8 / 25.0, 234 25.9 / 26.5, but 156 24.1 / 22.5; 64 x 128, 10 chains, L=1463 25.2 / 25.7, 4, L=4000 26.7 /
    // 27.9; 25 x 33, 28 chains, L=1100 23.3 / 25.0; 48 x 48 backward, 9, L=1100 24.1 / 25.3; from 110 calls on either
    // side of the line 0.88 to 0.97 of the time below it, 1.00 to 1.06 above); several scans of such a state on
    // three bf16 pieces 240 (32 x 64 backward, 6 chains, L=1600, 234 of them 0.99, 2, L=5154, 246 1.05); wider ones any number
    // (128 x 128, 8 chains, L=4000 0.89, 245 of 250 calls 0.73 to 0.93), and fused attention as well, whose chunks take
    // longer (8 chains, L=3111, 200 of them 31.2 / 28.5, 12, L=2335, 228 32.0 / 29.7).
    const int64_t fours = (total_chunks + 3) / 4;
    want = std::min<int64_t>(want, units * fours <= most_fours ? fours : total_chunks / 4);
    if (tuning().tpx_segs >= 0) want = std::max(1, tuning().tpx_segs);  // tuning aid
    if (want < 2) return 0;
    const int64_t seg_chunks = ((total_chunks + want - 1) / want + kTpAhead - 1) / kTpAhead * kTpAhead;
    const int64_t n = (total_chunks + seg_chunks - 1) / seg_chunks;
    // a workgroup walks at most 256 chunks with one running state (rounding), a chain has
    // at most 64 x 64 steps (flags of a group are watched by one wavefront), and every
    // consumer of every segment has a flag word
    if (n < 2 || seg_chunks > 256 || n > 4096 || 4 * units * n > kMaxWaves) return 0;
    *nseg = (int)n;
    return (int)seg_chunks;
}

// The chain-parallel kernel's plan for `nscans` scans of a D x F state over chains x L rows:
// *seg_chunks > 0: an exchange with *nseg segments of that many chunks; else *nseg > 0: chains
// cut into *nseg segments that need no exchange; both 0: another kernel takes the launch.
// (fp32 rows; those with bf16 among them have a plan of their own, mixed_plan_compute)
void tp_plan_compute(int64_t D, int64_t F, int64_t chains, int nscans, int64_t L, int *nseg,
                     int *seg_chunks, bool forced, bool odd, bool normed) {
    *nseg = *seg_chunks = 0;
    if (!tp_widths(D, F, forced, odd)) return;
    const bool wide = D != 64 || F != 64 || forced || odd;
    const bool others = !forced && !odd && mfma_scan_supported_widths(D, F);
    const int64_t units = chains * nscans * tp_fblocks(F);
    // Shapes of the other kernels with 32 rows or columns (a workgroup here has half of its
    // matrix work or half of its consumers to spare for them): measured at N=8, H=16, L=4096,
    // forward + backward, 32 x 128 0.62 against 0.80 ms and 128 x 32 0.76 against 0.78 on whole
    // chains, but 32 x 32 0.34 against 0.28, and with an exchange (N=4, H=16, L=16384)
    // 128 x 32 1.73 against 1.58 and 32 x 128 1.70 against 1.59: those stay where they were.
    const bool narrow = others && (D <= 32 || F <= 32);
    // Chains too short for an exchange (fewer than 24 chunks) run here on any number of
    // workgroups: the kernels that split L pay more for their exchange than a workgroup for
    // walking the chain (64 x 64 forward, 8 chains, L=640: 19 against 27 us; 128 x 128 backward, 4
    // chains, L=512: 29 against 62).  A single scan on the bf16-piece kernel, and its scans with
    // half of the consumers idle, only up to 8 chunks (128 x 128 forward, 2 chains, L=256: 16
    // against 17, L=512: 22 against 17; 128 x 32 forward, 8 chains, L=512: 27 against 20); of that kernel's with
    // more than 32 columns up to 10, from eight workgroups' worth on up to 13 and from twenty on up to 23 (128 x 128
    // forward, us, the kernels that split L / this one: 2 chains, L=270 17.2 / 14.4, L=390 18.8 / 18.3; 4, L=390 20.1 / 18.3, L=500
    // 20.9 / 22.0; 12, L=500 27.3 / 22.0, L=700 30.3 / 27.9; 128 x 96, 10 chains, L=736 28.4 / 30.1, 12 30.7 / 30.0; 128 x 64, 20 chains, L=610 29.7 / 25.8; 96 x 96, 12, L=390 20.2 /
    // 17.2; errors against float64 0.6 to 0.7 of theirs).
    const int64_t brief_chunks = D <= 64 || (F > 32 && nscans >= 2) ? 23 : F <= 32 ? 8 : units >= 20 ? (D > 96 && F > 64 && F <= 96 && units < 24 ? 20 : 23) : units >= 8 ? 13 : 10;
    if (narrow && D <= 32 && F <= 32) return;
    // Thousands of chains of one or two chunks with a state of at most 64 x 64 go to those kernels too,
    // where a workgroup's start costs more than its chunks (8192 chains, L=64: 32 x 128 1.17
    // against 0.60 ms, 20 x 20 0.63 against 0.46 on padded copies), and 32-wide shapes on more
    // than two rounds of workgroups, as for 64 x 64.
    // (four rounds for a state of 32 rows on chains of 32 chunks or more: 32 x 128 forward, 384
    // chains, L=1024: 113 against 174 us; 512 chains, L=2048: 277 against 344; 1024 chains: 293 / 279)
    if (narrow && units > (D <= 32 && L >= 32 * kChunk ? 1024 : 512) && tuning().tp < 0) return;
    // ... and 32-wide shapes on few workgroups: a workgroup of this kernel walks its chunks at
    // 1.1 to 1.7 us each whatever else the GPU does, the kernels that split L spread them over
    // all CUs (forward, us, this kernel / those: 32 x 128, 32 chains, L=4096: 83 / 62; 16 chains:
    // 78 / 54; 64 chains, 128 workgroups: 94 / 106.  128 x 32, 32 chains, L=4096: 152 / 69; 64
    // chains: 170 / 103; 128 chains: 227 / 204, L=2048: 107 / 101; 256 chains: 317 / 383).  Short
    // chains stay (32 x 128, 32 chains, L=1024: 29 / 39; 128 x 32, 64 chains, L=512: 32 / 36),
    // and 64 x 32 on the fp16-piece kernel needs 128 workgroups like 32 x 64 (128 chains,
    // L=2048: 51 / 57, L=8192: 210 / 229; 64 chains, L=1024: 28 / 32, L=2048: 47 / 41).
    if (narrow && tuning().tp < 0) {
        const int64_t total_chunks = (L + kChunk - 1) / kChunk;
        // a single scan on the bf16-piece kernel with half of its consumers without columns
        const bool lone_slab = F <= 32 && D > 64 && nscans == 1;
        int64_t least = 64, brief = lone_slab ? 16 : 32;
        // (the kernels that split L run 96 columns as slices: 32 x 96, 16 chains, L=2048: 44 / 73)
        if (D <= 32 && F == 96) least = 32, brief = 64;
        if (total_chunks > brief_chunks && units < (lone_slab ? 256 : 128) &&
            !(units >= least && total_chunks <= brief))
            return;
    }
    if (!forced && D <= 64 && F <= 64 && units > 512 && L <= 2 * kChunk) return;
    // fp32 64 x 64 chains of 257 to 1024 chunks on 112 workgroups or more are walked whole: a
    // running fp32 state of that length is what the reference keeps too (L=32768 against float64:
    // scale errors 1.8e-6 forward and 3e-6 backward where the reference's own order has 1.1e-6 and
    // 4e-6), and a workgroup per chain and scan reads every row once where an exchange reads it
    // twice and the kernels that split L more often (us, whole / before: forward, 256 chains,
    // L=16384: 883 / 1061; 128 chains: 485 / 537; backward of 64 chains: 559 / 704; of 256: 2082
    // / 2626; of 256 at L=32768: 4134 / 5290; of 36 chains, 108 workgroups: 466 / 419).
    // The same for the other states that the fp16-piece kernel takes, from 192 workgroups on, 128
    // beyond 512 chunks (64 x 128 forward, 128 chains, L=16384: 662 against 1049 us; 64 chains,
    // L=32768: 910 against 1083, L=16384: 458 against 452; 48 x 80, 64 chains, L=16384: 470 / 405).  Not for the bf16-piece kernel: 128 x 128 walked whole at L=12000 is outside the
    // element-wise bound 2.8 times as often as the reference's own order, where twice is the bar.
    // (32-wide states included: 32 x 128 forward, 128 chains, L=16384: 553 against 756; 64 x 32
    // backward, 256 chains, L=12000: 1404 against 1825)
    const bool walk_long = D <= 64 && !(odd && forced) && L > 256 * kChunk && L <= 1024 * kChunk &&
                           units >= (!wide ? 112 : L > 512 * kChunk ? 128 : 192);
    const int64_t most_fours = D > 64 || normed ? INT64_MAX : forced && nscans > 1 ? 240 : 192;
    if (!narrow && !walk_long) *seg_chunks = tp_exchange_segments(units, L, wide, most_fours, nseg);
    // fp32 rows, 64 x 64: any number of chains of 16 chunks or more (the fp16-piece kernel walks
    // them faster than the kernels that split L stream them: backward, 256 chains, L=4096: 528
    // against 694 us; 768 chains, L=2048: 784 against 1013; forward, 1536 chains, L=1024: 309
    // against 376); from 8 chunks on three rounds of workgroups for a single scan and nine for
    // the three of a backward call (L=256: backward of 384 chains 71 against 82, of 768 chains
    // 136 against 146, of 2048 chains 327 against 295; forward of 768 chains 50 against 50, of
    // 1024 chains 65 against 56), two below that (256 chains, L=128: 31 against 27)
    const int64_t chunks = (L + kChunk - 1) / kChunk;
    const int64_t most_units = chunks >= 16  ? INT64_MAX
                               : chunks >= 8 ? (nscans == 3 ? 2304 : 768)
                                             : 512;
    if (*seg_chunks == 0)
        *nseg = tp_kernel_segments(units, L, wide, others, walk_long, narrow, most_units, brief_chunks);
}

// Scans with bf16 rows among them: where the kernels that split L, which multiply such rows as they are
// too, are faster.  Measured over 4860 launches (the widths 32, 64, 96 and 128, forward, dV alone, dQ with
// dK, all three; 1 to 2048 chains of 64 to 32768 positions), each in whole and cut chains and with
// exchanges (us, split L / here):
//   wide: 64 x 64 forward, 1024 chains, L=64 12.3 / 17.9, L=256 32 / 40, but 512 chains, L=512 49 / 35;
//   backward, 768 chains, L=128 57 / 67, but 384 chains 45 / 36; 128 x 128 forward, 1 chain, L=1000 18 / 21,
//   but 4 chains, L=2048 47 / 26; 96 x 96 forward, 48 chains, L=8192 179 / 194, but 4 chains, L=2048 32 / 21;
//   32 rows or columns, several scans: dQ and dK of 32 x 128, 768 chains, L=128 47 / 60, but 256 chains 32 / 21,
//   128 chains, L=16384 1118 / 897, 48 chains, L=8192 223 / 264; 32 x 32 backward, 48 chains, L=8192 135 / 157,
//   but 16 chains 92 / 64 and L=65536 336 / 397;
//   single ones: 32 x 32, 16 chains, L=4096 17 / 22, 256 chains, L=1000 43 / 30; 128 x 32, 64 chains,
//   L=4096 66 / 74, 256 chains 236 / 165; 32 x 128 forward, 128 chains, L=8192 262 / 209, 64 chains 141 / 166
//   and L=16384 277 / 313, where its fp32 rows have to be exchanged.
// ... of them the short chains of wide states (more than 32 rows and columns): a round of workgroups takes
// 4.7 us here however short its chains, so those kernels win from some number of workgroups on, which grows
// with the chunks.  Measured: 128 to 2048 chains of 20 to 512 positions, split L / here: 64 x 64 forward, 684
// chains, L=126 20 / 26; 512 chains, L=512 49 / 35; 128 x 64, 768 chains, L=64 1.37 of the time here.
bool short_chains_split(int64_t D, int64_t F, int64_t units, bool single, int64_t chunks) {
    if (chunks > 16) return false;
    constexpr int16_t kAny = INT16_MAX;
    // the most workgroups for chains of 1, 2, 3, 4, 6, 8, 12 and 16 chunks
    struct Row {
        int d, f;
        int16_t most[8];
    };
    static constexpr Row kSingle[] = {
        {64, 64, {256, 256, 256, 256, 416, 512, 512, 512}},    {64, 96, {512, 650, 720, 720, 1024, 1216, 1300, kAny}},
        {64, 512, {256, 256, 256, 256, 512, 512, 512, 512}},   {96, 64, {256, 256, 256, 256, 800, 800, kAny, kAny}},
        {96, 96, {256, 256, 256, 256, 256, 256, kAny, kAny}},  {96, 512, {256, 256, 256, 256, kAny, kAny, kAny, kAny}},
        {128, 512, {256, kAny, kAny, kAny, kAny, kAny, kAny, kAny}}};
    static constexpr Row kSeveral[] = {
        {64, 64, {900, 1280, 1600, 1700, 1900, 2000, kAny, kAny}},
        {64, 96, {1200, 1500, 1700, 2048, 2100, 2400, kAny, kAny}},
        {64, 512, {600, 800, 880, 1060, 1100, 1160, 1160, kAny}}, {96, 64, {750, kAny, kAny, kAny, kAny, kAny, kAny, kAny}},
        {96, 96, {1000, 3000, 3300, 3300, 3300, 3300, kAny, kAny}}, {96, 512, {600, 3500, kAny, kAny, kAny, kAny, kAny, kAny}},
        {128, 64, {kAny, kAny, kAny, kAny, kAny, kAny, kAny, kAny}}, {128, 96, {800, 3500, kAny, kAny, kAny, kAny, kAny, kAny}},
        {128, 512, {2000, kAny, kAny, kAny, kAny, kAny, kAny, kAny}}};
    const int bucket = chunks <= 4 ? (int)chunks - 1 : chunks <= 6 ? 4 : chunks <= 8 ? 5 : chunks <= 12 ? 6 : 7;
    const Row *row = single ? kSingle : kSeveral;
    while (D > row->d || F > row->f) row++;
    // (96 x 96, a single scan: a last round less than four fifths full)
    if (single && D > 64 && D <= 96 && F > 64 && F <= 96 && units > 256 && (units + 255) / 256 * 205 > units) return true;
    // (many rounds of longer chains: both keep the memory busy)
    const int64_t again = chunks <= 8 || D > 64 || (F > 64 && F <= 96) ? INT64_MAX
                          : single ? (F > 64 ? 1100 : chunks <= 12 ? 1200 : 850)
                                   : 2300;
    return row->most[bucket] != kAny && units > row->most[bucket] && units < again;
}
bool mixed_splits(int64_t D, int64_t F, int64_t units, int nscans, int64_t chunks, bool bf16_results) {
    // (widths that those kernels take as padded copies only)
    if (!mfma_scan_supported_widths(D, F)) return D <= 64 && F <= 64 && units > (nscans == 1 ? 512 : 1400) && chunks <= 2;
    const bool single = nscans == 1;
    // (a last round of workgroups that is nearly empty)
    const bool uneven = units > 256 && (units + 255) / 256 * 256 * 7 > units * 10;
    if (D > 32 && F > 32) {
        if (short_chains_split(D, F, units, single, chunks)) return true;
        if (!single || D <= 64) return false;
        if (D <= 96 && F > 64 && F <= 96 && chunks > 48 && units >= (bf16_results ? 12 : 20) && units < (bf16_results ? 176 : 128))
            return true;
        // (128 x 128, us, split L / here: 3 chains, L=390 15.0 / 13.0, 6, L=610 20.8 / 17.2, L=760 23.3 / 19.3, but 3, L=500 15.0 / 15.2;
        // errors against float64 half of theirs.  bf16 results, dV of a backward call and the call: 128 x 64, 1 chain, L=416
        // 25.8 / 26.8, 3, L=380 25.7 / 27.1, but 10, L=410 0.95 of the time; 128 x 96, 7 chains, L=430 0.94, but L=760 46.9 / 49.1)
        const int64_t brief = bf16_results && units < 8 ? 11 : 13;
        const int64_t many = bf16_results && F > 64 && F <= 96 && chunks > 16 ? 16 : 12;
        return chunks > brief && chunks < (units <= 1 ? 128 : units <= 3 ? 96 : units <= 7 ? 48 : units < many ? 28 : 0);
    }
    if (!single) {
        if (D <= 32 && F <= 32) {
            // (bf16 results: whole chains take a time per round of 256 workgroups, split L a time per chain, so whole ones
            // where the rounds are 70 to 77 % full on average, or where chains are short or few enough for an exchange.
            // us, split L / here: 64 chains, L=4128 124 / 86, 85 chains, L=16384 448 / 305, but 86 chains 469 / 549, and 60
            // chains, L=7000 144 / 127, but L=14385 248 / 254; two rounds: 128 chains, L=4128 163 / 150, L=8192 284 / 287, 120
            // chains 274 / 288, L=14385 517 / 498; three: 180 chains, L=5154 261 / 271, L=8192 426 / 422, 200 chains 278 /
            // 273 and 460 / 427; 40 chains, L=6000 113 / 98, 20 chains, L=11000 116 / 92, 32 chains, L=11000 157 / 173)
            if (bf16_results && chunks > 128 && chunks <= 1024) {
                const int64_t rounds = (units + 255) / 256;
                const int64_t least = rounds == 1   ? (chunks > 320 ? 72 : 70)
                                      : rounds == 2 ? (chunks > 344 ? 70 : 75)
                                                    : (chunks > 224 ? 70 : 77);
                const bool full = 100 * units >= rounds * 256 * least;
                const bool brief = units <= 256 && chunks <= 192;
                const bool few = units <= 48 || (units <= 60 && chunks <= 512) || (units <= 84 && chunks <= 344);
                return !full && !brief && !few;
            }
            if (chunks > 128) return units > (chunks > 1024 ? 24 : 48);
            return chunks <= 64 && units > (chunks <= 4 ? 1024 : chunks <= 8 ? 1100 : 1536);
        }
        if (F <= 32 && chunks >= 192 && ((units > 64 && units < 144) || uneven)) return true;
        if (F <= 32 && chunks > 512) return units > 16;
        if (chunks > 64) return false;
        if (F > 64 && F <= 96 && chunks <= 12) return units > (chunks == 1 ? 1200 : chunks <= 3 ? 1450 : chunks <= 4 ? 1750 : 2150);
        if (F > 64) return units > (chunks <= 8 ? 1024 : 2048);
        return chunks <= 2 ? units > 512 : chunks <= 8 ? units > 768 : F <= 32 && units > 1024;
    }
    if (F > 64) {  // 32 rows
        if (F <= 96 && chunks <= 12) return units > (chunks == 1 ? 600 : chunks <= 2 ? 800 : chunks <= 4 ? 900 : 1150);
        if (chunks <= 64) return units > (chunks <= 2 ? 512 : chunks <= 8 ? 768 : 1024);
        if (chunks < 192) return false;
        if (bf16_results) return uneven || (units > 32 && units < 160);
        return units > 512 || uneven || (units > 32 && (chunks > 256 || units < 192));
    }
    if (F > 32) {
        if (chunks <= 24) return units > (chunks <= 4 ? (bf16_results ? 256 : 384) : chunks <= 8 ? 448 : bf16_results ? 512 : INT64_MAX);
        return chunks >= 48 && chunks <= 256 && units > 4 && units < (chunks <= 72 ? 48 : bf16_results ? 112 : 64);
    }
    // 32 columns
    if (chunks <= 2) return D <= 64 || units > 256;
    if (chunks <= 8) return units > (chunks > 4 && !bf16_results ? 320 : 256);
    if (chunks > 12 && uneven) return true;
    if (D > 64 && D <= 96 && chunks <= 24 && units > 256) return true;
    if (D > 64) {
        if (chunks <= 48) return units < (chunks <= 16 ? 32 : 16) || (bf16_results && units > 512);
        if (chunks <= 96) return !((units >= 8 && units <= 32) || units >= 112);
        return !(units <= (bf16_results && chunks > 256 ? 8 : 16) || (units >= 168 && chunks <= 256) ||
                 (units >= 112 && units <= 144 && chunks <= 128));
    }
    if (chunks <= 24) return units > 512;
    if (chunks <= 48) return units < 48 || (units > 512 && (bf16_results || (D <= 32 && units < 900)));
    if (bf16_results) return chunks > 256 || units < (D <= 32 ? (chunks <= 72 ? 176 : 224) : chunks <= 96 ? 112 : 176) || units > 512;
    // Forward, measured on 24 to 512 chains of 1600 to 32768 positions, with inputs from memory and with inputs that the
    // kernel before left in the caches (us, split L / here, the latter in parentheses).  Where all rows fit the Infinity Cache
    // split L reads them faster from there, and the lines are where both ways meet; else memory bounds split L.
    const bool cached = units * chunks * (int64_t)(kChunk * (4 * D + 6 * F)) <= (int64_t)256 << 20;
    if (D <= 32) {
        // Two segments a chain on up to 128 chains: 96 chains, L=1600 27.6 / 26.4 (25.1 / 22.7), 128, L=2500 43.9 / 40.4
        // (35.1 / 32.3).  Whole chains on more: 144, L=1600 34.4 / 29.8 (29.0 / 28.8), but 160, L=2500 51 / 44 (37.8 / 42.9);
        // 208, L=2900 72 / 50 (49.3 / 48.3), but 192 71 / 55 (46.0 / 48.5).  Beyond the caches 160, L=6000 107 / 96 (98 / 96),
        // L=8192 133 / 128, 208, L=4700 116 / 79 (106 / 78).  Longer ones are not walked whole.
        if (chunks > 256) return true;
        if (units <= 128) return units < (chunks <= 56 ? 96 : chunks <= 88 ? 128 : INT64_MAX);
        return units < (!cached ? 160 : chunks <= 56 ? 144 : chunks <= 72 ? 176 : 208);
    }
    // 64 rows.  Cut up to 128 chunks: 80 chains, L=2500 43.3 / 38.5 (36.4 / 31.5), 128, L=3778 83 / 63 (66 / 54); whole: 152, L=4000
    // 102 / 82 (93 / 81), but 136, L=3778 88 / 78 (70 / 77).
    if (chunks <= 72) return units < 64;
    if (chunks <= 128) return units < 80 || (chunks > 96 && units > 128 && units < 152);
    // Whole up to 256 chunks, on more than 128 chains: 152, L=5154 122 / 104, 136, L=6000 124 / 120.
    if (units >= 160 && chunks <= 256) return false;
    if (units > 128 && chunks <= 256) return cached;
    // With an exchange where the segments of all chains fill a round of 256 workgroups, two for more than 128 chains, to
    // seven eighths: 120, L=6000 126 / 113, 64, L=16384 153 / 135, 160, L=11000 254 / 244; but 96, L=9000 134 / 144, 136, L=8224
    // 165 / 188, 200 233 / 252 (within 1.03 elsewhere: 112, L=20000 322 / 332).  In the caches few long chains gain either way
    // (28, L=11000 65 / 59 (53 / 52)), five segments on 48 to 51 where rows come from memory, L=6000 59 / 55 (47 / 51); more
    // stay, 64 71 / 66 (57 / 60), 80 85 / 79 (66 / 73).
    const int64_t room = units <= 128 ? 256 : 512, groups = units * (room / units);
    if (units > 512 || 8 * groups < 7 * room) return true;
    if (!cached) return units < (chunks <= 320 ? 48 : 24);
    return chunks > 320 ? units < 24 || units > 32 : chunks <= 160 || units < 48 || units > 51;
}

// The plan of scans with bf16 rows among them on the chain-parallel kernel (three pieces for the state and
// fp32 rows, bf16 rows multiplied as they are, scan_tp_bf16_kernel): whichever is estimated shorter of
// whole or cut chains and an exchange of segment sums.  The estimates are fitted to 15650 launches (within
// 8 and 6 %): a chunk takes a workgroup 0.48, 0.65, 0.98 or 1.12 us with a state of up to 32, 64, 96 or 128
// rows, 1.25 times that where one operand is fp32, a round of workgroups 4.7 us besides; both walks of an
// exchange 1.55 times as long, and the exchange what a round's workgroups wait for each other.
// Chains are walked whole up to 256 chunks, and up to 1024 where the results are bf16, which makes the
// rounding of a long running state a non-issue.
// `stateful`: a state is handed in or out.
void mixed_plan_compute(int64_t D, int64_t F, int64_t chains, int nscans, int64_t L, bool bf16_results, bool stateful,
                        int *nseg, int *seg_chunks) {
    *nseg = *seg_chunks = 0;
    if (!tp_widths(D, F) || tuning().tp == 0) return;
    const int64_t units = chains * nscans * tp_fblocks(F), chunks = (L + kChunk - 1) / kChunk;
    // (FTC_TP=1, FTC_TPX=0: tuning aids)
    if (tuning().tp < 0 && mixed_splits(D, F, units, nscans, chunks, bf16_results)) return;
    // A state that a few chains of 9 or 13 chunks hand out: the kernels that split L add it up in sums of a few chunks, a
    // chain walked whole in one, which leaves it 1.05 times as far from float64 (0.99 at 10 to 12 chunks, where they
    // have longer sums).  Sums of four chunks, exchanged, leave it 0.96 times as far, and the rows 0.53 times either way.
    // 128 x 128, us, split L / exchanged / whole: 1 chain, L=270 20.2 / 16.4 / 12.8, 4, L=400 23 / 17.9 / 15.2.
    if (stateful && nscans == 1 && D > 96 && F > 32 && (chunks == 9 || chunks == 13) && units < 16 && tuning().tp < 0 &&
        tuning().tpx != 0 && mfma_scan_supported_widths(D, F)) {
        *seg_chunks = kTpAhead;
        *nseg = (int)((chunks + kTpAhead - 1) / kTpAhead);
        return;
    }
    const double chunk_us = (D <= 32 ? 0.48 : D <= 64 ? 0.65 : D <= 96 ? 0.98 : 1.12) * (bf16_results ? 1.25 : 1.0);
    double least = 1e30;
    if (chunks <= (bf16_results ? 1024 : 256)) {
        // (priced at 0.6 in steps of kTpAhead, as fitted, and not as tp_cuts has them launched: at the launch's price
        // bf16 forwards of 20 to 60 chunks on few chains would be cut instead of exchanging sums, 160 of 9053
        // launches in 0.95 of their time, but their sums run over longer segments, 1.08e-7 from float64 for
        // 1.00e-7; backward calls would take 1.03 times as long)
        int32_t start[kMaxTpSegments + 1];
        int n = chunks <= 128 ? (int)std::max<int64_t>(1, std::min(round_segments(units), chunks)) : 1;
        n = tp_segment_starts(chunks, n, start, kTpAhead, 0.6);
        double longest = (double)chunks;
        if (n > 1) {
            longest = 0;
            for (int i = 0; i < n; i++) longest = std::max(longest, 0.6 * start[i] + (double)(start[i + 1] - start[i]));
        }
        least = (double)((units * n + 255) / 256) * (longest * chunk_us + 4.7) + 0.5;
        *nseg = n;
    }
    // (not below 24 chunks, 28 of wide states: 16 of them, 1 chain of 64 x 64 backward 14.4 us against 13.5 cut in
    // four; 25, 12 chains of 128 x 64 backward 46 against 42)
    for (int64_t n = 2; n <= 64 && n <= chunks / 4 && chunks >= (D > 64 ? 28 : 24) && tuning().tpx != 0; n++) {
        const int64_t c = ((chunks + n - 1) / n + kTpAhead - 1) / kTpAhead * kTpAhead, segs = (chunks + c - 1) / c;
        if (c > 256 || segs < 2 || 4 * units * segs > kMaxWaves) continue;
        const double filled = std::min(1.0, (double)(units * segs) / 256.0);
        const double us = (double)((units * segs + 255) / 256) * (1.55 * (double)c * chunk_us + 0.3 + 9.9 * filled) +
                          5.7 + 0.13 * (double)std::min<int64_t>(segs, 16) + 0.9 * std::sqrt((double)segs);
        if (us < least - 1e-9) least = us, *nseg = (int)segs, *seg_chunks = (int)c;
    }
}

// workspace of the exchange: control block, then two state slots (own sum, group total) of
// D x 16 floats (D rounded up to whole blocks of 64 rows) per consumer, four consumers per segment
int64_t tp_exchange_workspace_bytes(int64_t units, int nseg, int64_t D) {
    return kControlBytes + 2 * 4 * units * nseg * (int64_t)((D + 63) / 64 * 64 * 16 * 4);
}

// `wg`: the plan is for workgroups of F / 32 wavefronts (each has its own flag words);
// `norm`: for their fused attention form, with one more wavefront and state slab per unit
MfmaPlan make_plan_compute(int64_t N, int64_t H, int64_t L, int64_t D, int64_t F, int nscans,
                           bool wg, bool norm) {
    MfmaPlan pl;
    const int64_t flags_per_unit = wg ? F / 32 + (norm ? 1 : 0) : 1;
    const int64_t chains = std::max<int64_t>(1, N * H);
    const int64_t total_chunks = (L + kChunk - 1) / kChunk;
    // Resident at a time: 1024 wavefronts (one per SIMD: register footprint), or one workgroup
    // per CU with 4 / (F / 32) segments each.  Pick the segment
    // length (in chunks) that minimises an estimate of the makespan: rounds of resident
    // wavefronts times the work of one wavefront (pass 1 costs about half of pass 2, the
    // exchange of segment sums about three chunks).
    const int64_t slots = wg ? 256 * scan_wg_units_per_block((int)F, norm) : 1024;
    int64_t best_c = total_chunks;
    double best_cost = (double)total_chunks * (double)((chains * nscans + slots - 1) / slots);
    for (int64_t c = 1; c < total_chunks && c <= 4096; c++) {
        const int64_t nseg = (total_chunks + c - 1) / c;
        const int64_t waves = chains * nseg;
        if (waves * nscans * flags_per_unit > kMaxWaves || nseg > 4096) continue;  // <= 64 groups of 64 steps
        const double rounds = (double)((waves * nscans + slots - 1) / slots);
        // (the exchange: a step reads the sums of its group and the totals of the groups before
        // it one after the other, about a chunk and a half's time each beyond the first four;
        // bf16 forward, 32 chains, L=1024: segments of 1 / 2 / 4 / 8 chunks 34 / 23 / 23 / 29 us)
        double reads = (double)(nseg - 1);
        if (nseg > 5) {
            int64_t g = 1;
            while (g * g < nseg) g++;
            reads = (double)((g - 1) + ((nseg + g - 1) / g - 1));
        }
        // (states of up to 64 x 64 only: on wider ones a chunk takes longer and the reads weigh
        // less -- 128 x 32, 8 chains, L=4096: segments of 4 chunks 51 us, of 8 chunks 69)
        const double look_back = D <= 64 && F <= 64 ? 1.6 * std::max(0.0, reads - 4.0) : 0.0;
        const double per_wave = nseg > 1 ? c * 1.5 + 3.0 + look_back : (double)c;
        const double cost = rounds * per_wave;
        if (cost < best_cost - 1e-9) {
            best_cost = cost;
            best_c = c;
        }
    }
    // tuning aid: FTC_SEG_CHUNKS=<n> forces segments of n chunks
    if (tuning().seg_chunks >= 0) {
        const int64_t forced = tuning().seg_chunks;
        if (forced >= 1 && forced <= total_chunks) {
            const int64_t nseg = (total_chunks + forced - 1) / forced;
            if (chains * nseg * nscans * flags_per_unit <= kMaxWaves && nseg <= 4096) best_c = forced;
        }
    }
    pl.seg_len = (int)(best_c * kChunk);
    pl.nseg = (int)((L + pl.seg_len - 1) / pl.seg_len);
    pl.waves = chains * pl.nseg;
    pl.workspace_bytes = 0;
    if (pl.nseg > 1)
        pl.workspace_bytes = kControlBytes + 2 * nscans * pl.waves * D * (F + (norm ? 32 : 0)) *
                                                 (int64_t)sizeof(float);
#ifdef FTC_TIMELINE
    pl.workspace_bytes += nscans * pl.waves * 128;  // time stamps (ftc_wg_kernel.h)
#endif
    return pl;
}

struct TpPlan {
    int nseg, seg_chunks;
};
void tp_plan(int64_t D, int64_t F, int64_t chains, int nscans, int64_t L, int *nseg, int *seg_chunks,
             bool forced = false, bool odd = false, bool normed = false) {
    static thread_local PlanMemo<TpPlan> memo;
    const int64_t key[8] = {D, F, chains, nscans, L, forced ? 1 : 0, odd ? 1 : 0, normed ? 1 : 0};
    const TpPlan pl = memo.get(key, [&]() {
        TpPlan p;
        tp_plan_compute(D, F, chains, nscans, L, &p.nseg, &p.seg_chunks, forced, odd, normed);
        return p;
    });
    *nseg = pl.nseg, *seg_chunks = pl.seg_chunks;
}
void mixed_plan(int64_t D, int64_t F, int64_t chains, int nscans, int64_t L, bool bf16_results, bool stateful, int *nseg,
                int *seg_chunks) {
    static thread_local PlanMemo<TpPlan> memo;
    const int64_t key[8] = {D, F, chains, nscans, L, bf16_results ? 1 : 0, stateful ? 1 : 0, 0};
    const TpPlan pl = memo.get(key, [&]() {
        TpPlan p;
        mixed_plan_compute(D, F, chains, nscans, L, bf16_results, stateful, &p.nseg, &p.seg_chunks);
        return p;
    });
    *nseg = pl.nseg, *seg_chunks = pl.seg_chunks;
}
MfmaPlan make_plan(int64_t N, int64_t H, int64_t L, int64_t D, int64_t F, int nscans, bool wg,
                   bool norm = false) {
    static thread_local PlanMemo<MfmaPlan> memo;
    const int64_t key[8] = {N, H, L, D, F, nscans, wg ? 1 : 0, norm ? 1 : 0};
    return memo.get(key, [&]() { return make_plan_compute(N, H, L, D, F, nscans, wg, norm); });
}

// every row must start on a 16-byte boundary (16-byte loads and stores)
bool aligned16(const void *ptr, int64_t s0, int64_t s1, int64_t s2, int dtype) {
    const int per16 = dtype == FTC_F32 ? 4 : 8;
    return ((uintptr_t)ptr % 16 == 0) && s0 % per16 == 0 && s1 % per16 == 0 && s2 % per16 == 0;
}

// what the chain-parallel kernel asks of rows: fp32 rows on 16-byte boundaries, bf16 rows (which
// it reads and writes four values at a time) on 8-byte boundaries
bool aligned_quads(const void *ptr, int64_t s0, int64_t s1, int64_t s2, int dtype) {
    if (dtype == FTC_F32) return aligned16(ptr, s0, s1, s2, dtype);
    return ((uintptr_t)ptr % 8 == 0) && s0 % 4 == 0 && s1 % 4 == 0 && s2 % 4 == 0;
}

// element-type combinations with a compiled kernel: (a, b, v, out)
enum Combo { kNone = 0, kFFFF, kBBBF, kFBBB, kBFBB, kBBFB };
Combo combo_of(const ScanDesc &sd) {
    const int a = sd.a.dtype, b = sd.b.dtype, v = sd.v.dtype, o = sd.out.dtype;
    const int F32 = FTC_F32, B16 = FTC_BF16;
    if (a == F32 && b == F32 && v == F32 && o == F32) return kFFFF;  // every fp32 scan
    if (a == B16 && b == B16 && v == B16 && o == F32) return kBBBF;  // bf16 forward
    if (a == F32 && b == B16 && v == B16 && o == B16) return kFBBB;  // bf16 dQ (a = grad_out)
    if (a == B16 && b == F32 && v == B16 && o == B16) return kBFBB;  // bf16 dK (b = grad_out)
    if (a == B16 && b == B16 && v == F32 && o == B16) return kBBFB;  // bf16 dV (v = grad_out)
    return kNone;
}

// chain-parallel scans of states of up to 64 rows run on the fp16 matrix path
// (ftc_tph_kernel.h: two scaled fp16 pieces per value), wider ones on three bf16 pieces
bool tph_takes_rows(int64_t D) {
    return D <= 64 && tuning().tph != 0;  // (FTC_TPH=0: tuning aid)
}

// rows must not overlap (the descriptor's end marks the first row outside the segment) and
// row strides must keep a segment's byte extent inside a 32-bit buffer descriptor
bool stride_ok(int64_t stride_l, int width) { return stride_l >= width && stride_l <= (1 << 16); }

}  // namespace

int mfma_slice_widths(int64_t D, int64_t F, int (&widths)[kMfmaMaxSlices]) {
    // the widest state a wavefront holds is 4096 values
    const int widest = D == 32 ? 128 : D == 64 ? 64 : (D == 96 || D == 128) ? 32 : 0;
    if (widest == 0 || F < 32 || F % 32 != 0) return 0;
    int n = 0;
    for (int64_t left = F; left > 0;) {
        int w = widest;
        while (w > left) w /= 2;
        if (n == kMfmaMaxSlices) return 0;
        widths[n++] = w;
        left -= w;
    }
    return n;
}

ScanDesc mfma_slice(const ScanDesc &scan, int col0, int width) {
    ScanDesc s = scan;
    const int vb = scan.v.dtype == FTC_F32 ? 4 : 2, ob = scan.out.dtype == FTC_F32 ? 4 : 2;
    s.v.ptr = (const char *)scan.v.ptr + (int64_t)col0 * vb;
    s.v.width = width;
    s.out.ptr = (char *)scan.out.ptr + (int64_t)col0 * ob;
    s.out.width = width;
    if (s.initial.ptr) s.initial.ptr += col0;
    if (s.final_.ptr) s.final_.ptr += col0;
    return s;
}

bool mfma_scan_same_launch(const ScanDesc &x, const ScanDesc &y) {
    return combo_of(x) == combo_of(y) && x.a.width == y.a.width && x.v.width == y.v.width;
}

bool mfma_operand_in_place(const void *ptr, int64_t stride_n, int64_t stride_h, int64_t stride_l,
                           int dtype, int width, int64_t L) {
    return (L <= 1 || stride_ok(stride_l, width)) && aligned16(ptr, stride_n, stride_h, stride_l, dtype);
}

bool mfma_scan_supported(const ScanDesc &sd, int64_t L) {
    const Operand &a = sd.a, &b = sd.b, &v = sd.v;
    const OperandOut &out = sd.out;
    const int D = a.width, F = v.width;
    const bool shape_ok = (D == 64 && F == 64) || (D == 32 && F == 128) || (D == 128 && F == 32) ||
                          (D == 32 && F == 32) || (D == 32 && F == 64) || (D == 64 && F == 32) ||
                          (D == 96 && F == 32);
    if (!shape_ok) return false;
    if (combo_of(sd) == kNone) return false;
    if (L > 1 && !(stride_ok(a.stride_l, D) && stride_ok(b.stride_l, D) &&
                   stride_ok(v.stride_l, F) && stride_ok(out.stride_l, F)))
        return false;
    return aligned16(a.ptr, a.stride_n, a.stride_h, a.stride_l, a.dtype) &&
           aligned16(b.ptr, b.stride_n, b.stride_h, b.stride_l, b.dtype) &&
           aligned16(v.ptr, v.stride_n, v.stride_h, v.stride_l, v.dtype) &&
           aligned16(out.ptr, out.stride_n, out.stride_h, out.stride_l, out.dtype);
}

int64_t mfma_scan_workspace_bytes(int64_t N, int64_t H, int64_t L, int64_t D, int64_t F,
                                  int nscans) {
    // whichever kernel the element types will select
    int64_t bytes = std::max(make_plan(N, H, L, D, F, nscans, false).workspace_bytes,
                             make_plan(N, H, L, D, F, nscans, true).workspace_bytes);
    return std::max(bytes, mfma_tp_workspace_bytes(N, H, L, D, F, nscans));
}

int64_t mfma_tp_workspace_bytes(int64_t N, int64_t H, int64_t L, int64_t D, int64_t F, int nscans,
                                bool forced, bool odd) {
    int nseg = 0, seg_chunks = 0;
    const int64_t chains = std::max<int64_t>(1, N * H);
    if (forced && odd) F = 64;  // (`nscans` blocks of columns, see column_blocks)
    tp_plan(D, F, chains, nscans, L, &nseg, &seg_chunks, forced, odd);
    return seg_chunks > 0 ? tp_exchange_workspace_bytes(chains * nscans * tp_fblocks(F), nseg, D) : 0;
}

bool mfma_scan_clips(int64_t D, int64_t F, int nscans, int64_t L) {
    int widths[kMfmaMaxSlices];
    return D <= 64 && !(D == 32 && F == 32) && mfma_slice_widths(D, F, widths) == 1 && tuning().dma != 0 &&
           !use_wg_kernel(D, F, nscans, L, true);
}

bool has_state(const ScanDesc *scans, int nscans) {
    for (int i = 0; i < nscans; i++)
        if (scans[i].initial.ptr || scans[i].final_.ptr) return true;
    return false;
}

// the widest rows of a launch (they differ between scans only where `odd` allows it)
void widest_rows(const ScanDesc *scans, int nscans, int *D, int *F) {
    *D = *F = 0;
    for (int i = 0; i < nscans; i++) *D = std::max(*D, scans[i].a.width), *F = std::max(*F, scans[i].v.width);
}

// blocks of 64 output columns in all
int64_t column_blocks(const ScanDesc *scans, int nscans) {
    int64_t n = 0;
    for (int i = 0; i < nscans; i++) n += tp_fblocks(scans[i].v.width);
    return n;
}

bool mfma_tp_takes(const ScanDesc *scans, int nscans, int64_t N, int64_t H, int64_t L, bool forced,
                   bool odd) {
    if (nscans < 1 || nscans > kMaxScans) return false;
    int D, F;
    widest_rows(scans, nscans, &D, &F);
    if (!tp_widths(D, F, forced, odd)) return false;
    if (odd && !forced && !tph_takes_rows(D)) return false;
    int64_t widest_stride = 0;
    const bool stateful = has_state(scans, nscans);
    bool mixed = false;
    for (int i = 0; i < nscans; i++) {
        const ScanDesc &sd = scans[i];
        const Combo combo = combo_of(sd);
        mixed = mixed || combo != kFFFF;
        // (rows with bf16 among them: not as parts of wider scans, whose results are added up in fp32)
        if (combo == kNone || (combo != kFFFF && (forced || tuning().tph == 0))) return false;
        // (odd widths: scans of any widths side by side, where pieces are scaled as long as none has a
        // second block of columns)
        if ((sd.a.width != D || sd.v.width != F) && !(odd && (forced || F <= 64))) return false;
        if (odd && (combo != kFFFF || sd.a.width < 8 || sd.v.width < 8)) return false;
        if (L > 1 && !(stride_ok(sd.a.stride_l, sd.a.width) && stride_ok(sd.b.stride_l, sd.a.width) &&
                       stride_ok(sd.v.stride_l, sd.v.width) && stride_ok(sd.out.stride_l, sd.v.width)))
            return false;
        if (odd) {
            if (((uintptr_t)sd.a.ptr | (uintptr_t)sd.b.ptr | (uintptr_t)sd.v.ptr | (uintptr_t)sd.out.ptr) % 4)
                return false;
        } else if (!(aligned_quads(sd.a.ptr, sd.a.stride_n, sd.a.stride_h, sd.a.stride_l, sd.a.dtype) &&
              aligned_quads(sd.b.ptr, sd.b.stride_n, sd.b.stride_h, sd.b.stride_l, sd.b.dtype) &&
              aligned_quads(sd.v.ptr, sd.v.stride_n, sd.v.stride_h, sd.v.stride_l, sd.v.dtype) &&
              aligned_quads(sd.out.ptr, sd.out.stride_n, sd.out.stride_h, sd.out.stride_l, sd.out.dtype)))
            return false;
        widest_stride = std::max(widest_stride, std::max(std::max(sd.a.stride_l, sd.b.stride_l),
                                                         std::max(sd.v.stride_l, sd.out.stride_l)));
    }
    // the chain-parallel kernel addresses a whole chain through one 32-bit descriptor
    if ((L + 2 * kChunk) * std::max<int64_t>(widest_stride, std::max(D, F)) * 4 >= 0x7fffffffLL)
        return false;
    int nseg = 0, seg_chunks = 0;
    const int64_t chains = std::max<int64_t>(1, N * H);
    // (fp32 states of more than 64 rows that are handed in or out stay with the kernels that split L, whose sums are
    // shorter, over 9 to 23 chunks where the chains' segments do not fill half the GPU: 128 x 128, 8 chains, L=400 39.0 us
    // for 22.1, but the state is 1.25e-7 from float64 there and 3.5e-7 here; the rows are 1.9e-7 and 1.3e-7.
    // Those that are only handed in as well: rows are the same whether the state is asked for or not.
    // So do bf16 rows with 65 to 96 state rows over 9, 12 and 13 chunks: 96 x 96, 1 to 7 chains, 9 and 13 the state 1.05
    // times as far, 12 13.6 us for 14.7; see mixed_plan_compute)
    const int64_t chunks = (L + kChunk - 1) / kChunk, units = chains * tp_fblocks(F);
    if (stateful && !forced && !odd && nscans == 1 && D > 64 && F > 32 && chunks > 8 && tuning().tp < 0 &&
        mfma_scan_supported_widths(D, F)) {
        if (mixed ? D <= 96 && units < 16 && (chunks == 9 || chunks == 12 || chunks == 13)
                  : chunks < 24 && units * round_segments(units) < kHalfTheGpu)
            return false;
    }
    if (mixed)
        mixed_plan(D, F, chains, nscans, L, scans[0].out.dtype != FTC_F32, stateful, &nseg, &seg_chunks);
    else if (odd && forced)
        tp_plan(D, 64, chains, (int)column_blocks(scans, nscans), L, &nseg, &seg_chunks, forced, odd);
    else
        tp_plan(D, F, chains, nscans, L, &nseg, &seg_chunks, forced, odd);
    return nseg > 0;
}

int64_t mfma_tp_mixed_workspace_bytes(int64_t N, int64_t H, int64_t L, int64_t D, int64_t F, int nscans,
                                      bool may_have_state) {
    const int64_t chains = std::max<int64_t>(1, N * H);
    int64_t bytes = 0;
    for (const bool bf16_results : {false, true})
        for (const bool stateful : {false, may_have_state}) {
            int nseg = 0, seg_chunks = 0;
            mixed_plan(D, F, chains, nscans, L, bf16_results, stateful, &nseg, &seg_chunks);
            if (seg_chunks > 0)
                bytes = std::max(bytes, tp_exchange_workspace_bytes(chains * nscans * tp_fblocks(F), nseg, D));
        }
    return bytes;
}

// (a chunk of a state of more than 64 rows takes 1.7 times as long; `forced`: on three bf16 pieces, `nscans` blocks)
double mfma_tp_odd_chunks(int64_t D, int64_t F, int64_t N, int64_t H, int nscans, int64_t L, bool forced) {
    int nseg = 0, seg_chunks = 0;
    if (forced) F = 64;  // (`nscans` blocks of columns)
    const int64_t chains = std::max<int64_t>(1, N * H), units = chains * nscans * tp_fblocks(F);
    tp_plan(D, F, chains, nscans, L, &nseg, &seg_chunks, forced, true);
    if (nseg == 0) return 1e30;
    // (fitted to segments of whole fours of chunks, eight of them where a chain is no multiple of four.  Priced as the four that
    // are launched, backward calls would be two launches instead of one: 75 x 10, 8 chains, L=989 37.7 -> 49.1 us,
    // L=2900 61 -> 66, 99 x 101, 4 chains, L=4000 68 -> 85.  Others would gain, 32 chains, L=989, 75 x 10 62 -> 56 and
    // 120 x 31 70 -> 59, with dQ and dK 1.5 times as far from float64, and 120 x 31, 7 to 20 chains, L=1463 0.87 to 0.92 of
    // the time, 0.5 to 0.7 times as far)
    const int64_t chunks = (L + kChunk - 1) / kChunk;
    if (seg_chunks == kTpAhead && chunks % kTpAhead) {
        seg_chunks = 2 * kTpAhead;
        nseg = (int)((chunks + seg_chunks - 1) / seg_chunks);
    }
    const int64_t rounds = (units * nseg + 255) / 256;
    double longest = 0.0;
    if (seg_chunks > 0) {
        longest = 1.6 * seg_chunks + 4.0;
    } else {
        // (at the price of tp_cuts more scans of two shapes would share a launch, 43 calls of 18106 in 0.88 of their
        // time, but 31 x 120 came out 3.5e-7 from float64 for 2.1e-7 and 75 x 10 2.5e-7 for 1.6e-7)
        int32_t start[kMaxTpSegments + 1];
        nseg = tp_segment_starts(chunks, nseg, start, kTpAhead, 0.6);
        for (int s = 0; s < nseg; s++)
            longest = std::max(longest, 0.6 * start[s] + (double)(start[s + 1] - start[s]));
    }
    return (double)rounds * ((D > 64 ? 1.7 : 1.0) * longest + 4.0);
}

// (rows of 128 values: the chain-parallel kernel alone)
bool fused_wide(int64_t D, int64_t F) { return D > 64 || F > 64; }

// (the attention's gradients with an exchange: another tile of state for the sums of rows)
constexpr int64_t kGradStateRows = 128;

bool fused_attention_supported(const ScanDesc &sd, int64_t L) {
    if (combo_of(sd) != kFFFF || sd.reverse || sd.initial.ptr || sd.final_.ptr) return false;
    if (!fused_wide(sd.a.width, sd.v.width))
        return scan_wg_norm_covers(sd.a.width, sd.v.width) && mfma_scan_supported(sd, L);
    for (const Operand *t : {&sd.a, &sd.b, &sd.v})
        if (!mfma_operand_in_place(t->ptr, t->stride_n, t->stride_h, t->stride_l, t->dtype, t->width, L)) return false;
    const OperandOut &o = sd.out;
    return mfma_operand_in_place(o.ptr, o.stride_n, o.stride_h, o.stride_l, o.dtype, o.width, L);
}

// (the exchange of the chain-parallel fused form: another tile of state for its denominators)
int64_t fused_tp_state_rows(int64_t D) { return (D + 63) / 64 * 64 + 64; }

// The fused attention launch on the chain-parallel kernel: its plan is that of a single 64 x 64
// scan whatever the widths (a chunk costs the same).  Returns false: the workgroup form, whose
// units split L and which carries two units of 32 value columns per workgroup.  The lines are where the
// two cross; this way / the workgroup form, time, on both sides of them: 64 x 64, 16 chunks, 4 chains 0.98; 21
// chunks, 20 chains 0.96, 16 chains 1.00; 24 chunks, 20 chains 0.97, 16 chains 1.00; 32 chunks, 36 chains 0.93, 32 (there
// and below with an exchange) 0.98; 36 chunks, 40 chains 0.92; 42 chunks, 40 chains 0.95, 36 chains 1.00; 48 chunks,
// 36 chains 0.93, 28 chains 0.97; 64 chunks, 24 chains 0.91, 20 chains 0.98; far from them 64 chains, 10, 24, 42
// and 64 chunks 0.54, 0.68, 0.80 and 0.85.  With an exchange up to 6 chains from 28 chunks on, up to 12 from
// 37, where the workgroup form's segments grow (us, workgroup form / this way: 3 chains, 28 chunks 21.5 / 20.2, 4, 50
// chunks 27.3 / 21.6, 1, 101 chunks 30.2 / 22.9, 256 chunks 37.6 / 25.4; 8, 37 chunks 25.1 / 21.7, 128 chunks
// 36.7 / 32.7; 12, 50 chunks 29.9 / 25.1; but 3 to 8 chains, 25 chunks 19.3 / 20.0); 8 chains, 22.5 / 21.1 at 32
// chunks, and 16, 23.5 / 22.3 at 28 and 41.7 / 39.3 at 128, stay.  64 x 32: 16 chunks, 8 chains 0.89; 24 chunks, 40 chains 0.84; 32 chunks,
// 40 chains 0.95; 40 chunks, 56 chains 0.90, 48 chains 0.96; 48 chunks, 80 chains 0.89, 64 chains 1.02.  32 x 64: 10
// chunks, 16 chains 0.94, 8 chains 1.00; 16 chunks, 24 chains 0.96, 16 chains 1.06; 24 chunks, 40 chains 0.91, 32
// chains 1.11; 32 chunks, 56 chains 0.94, 48 chains 1.00; 40 chunks, 64 chains 0.93; 48 chunks, 80 chains 0.92, 64 chains
// 1.08.  32 x 32 stays: 1000 positions 31.7 / 31.3 us the other way round.  One width of 32 on more than a round of
// workgroups, or with an exchange, stays too: 102 / 116 and 95.7 / 106 us.
// Chains of more than 256 chunks are not walked whole on three bf16 pieces (tp_plan_compute).
//
// Rows of 128 have no other fused form: the plan is that of such a scan where the chain-parallel kernel
// has to take it.  Measured, 128 x 128 (us, two scans with the element-wise passes around them / this
// way): 8 chains, L=2000 122 / 47; 80 chains, L=300 102 / 34; 128 chains, L=856 260 / 90; 256 chains,
// L=1000 476 / 208; 70 chains, L=8192 1335 / 715.
bool fused_tp_plan(int64_t D, int64_t F, int64_t chains, int64_t L, int *nseg, int *seg_chunks) {
    *nseg = *seg_chunks = 0;
    if (fused_wide(D, F)) {
        tp_plan(D, F, chains, 1, L, nseg, seg_chunks, true, false, true);
        return *nseg > 0;
    }
    if (tuning().wg > 0) return false;
    const int64_t chunks = (L + kChunk - 1) / kChunk;
    tp_plan(64, 64, chains, 1, L, nseg, seg_chunks, false, false, true);
    if (*nseg > 0 && *seg_chunks == 0 && chunks > 256) *nseg = 0;
    if (*nseg == 0 || tuning().wg == 0) return *nseg > 0;  // (FTC_WG=0: tuning aid)
    // the fewest chains without an exchange, where the two cross
    const bool square = D == 64 && F == 64;
    int64_t least;
    if (square)
        least = chunks <= 16 ? 4 : chunks <= 24 ? 20 : chunks <= 32 ? 36 : 40;
    else if (D == 64)
        least = chunks <= 10 ? 4 : chunks <= 16 ? 8 : chunks <= 24 ? 32 : chunks <= 32 ? 40 : chunks <= 44 ? 56 : 80;
    else
        least = chunks <= 4    ? INT64_MAX
                : chunks <= 7  ? 8
                : chunks <= 10 ? 16
                : chunks <= 16 ? 24
                : chunks <= 24 ? 40
                : chunks <= 28 ? 48
                : chunks <= 32 ? 56
                : chunks <= 44 ? 64
                               : 80;
    const bool take = *seg_chunks > 0 ? square && (chains <= 6 ? chunks >= 28 : chains <= 12 ? chunks >= 37 : chains >= (chunks >= 64 ? 24 : 36) && chunks >= 44)
                                      : (square || ((D == 64 || F == 64) && chains <= 256 && chunks <= 60)) && chains >= least;
    if (!take) *nseg = *seg_chunks = 0;
    return take;
}

int64_t fused_attention_workspace_bytes(int64_t N, int64_t H, int64_t L, int64_t D, int64_t F) {
    int nseg, seg_chunks;
    int64_t bytes = fused_wide(D, F) ? 0 : make_plan(N, H, L, D, F, 1, true, true).workspace_bytes;
    const int64_t chains = std::max<int64_t>(1, N * H);
    if (fused_tp_plan(D, F, chains, L, &nseg, &seg_chunks) && seg_chunks > 0)
        bytes = std::max(bytes, tp_exchange_workspace_bytes(chains * tp_fblocks(F), nseg, fused_tp_state_rows(D)));
    return bytes;
}

bool fused_attention_wide_covers(int64_t N, int64_t H, int64_t L, int64_t D, int64_t F) {
    int nseg, seg_chunks;
    return fused_tp_plan(D, F, std::max<int64_t>(1, N * H), L, &nseg, &seg_chunks);
}

bool attention_gradients_take(const ScanDesc *scans, int nscans, const AttentionGradients &grads, int64_t N,
                              int64_t H, int64_t L) {
    if (!tph_takes_rows(64) || nscans < 1 || nscans > kMaxScans) return false;
    // (a whole chain is addressed through one 32-bit descriptor)
    auto in_place = [&](const void *ptr, int64_t sn, int64_t sh, int64_t sl, int dtype, int width) {
        return dtype == FTC_F32 && width == 64 && mfma_operand_in_place(ptr, sn, sh, sl, dtype, width, L) &&
               (L + 2 * kChunk) * std::max<int64_t>(sl, 64) * 4 < 0x7fffffffLL;
    };
    for (int i = 0; i < nscans; i++) {
        for (const Operand *t : {&scans[i].a, &scans[i].b, &scans[i].v, &grads.rows[i]})
            if (!in_place(t->ptr, t->stride_n, t->stride_h, t->stride_l, t->dtype, t->width)) return false;
        const OperandOut &o = scans[i].out;
        if (!in_place(o.ptr, o.stride_n, o.stride_h, o.stride_l, o.dtype, o.width)) return false;
    }
    int nseg = 0, seg_chunks = 0;
    // (where the planner has those scans on the kernels that split L they stay there: they hold every value exactly,
    // and chains of one to four chunks are faster so, N=32, H=32, L=64, forward and backward 133 us against 168)
    tp_plan(64, 64, std::max<int64_t>(1, N * H), nscans, L, &nseg, &seg_chunks);
    return nseg > 0;
}

int64_t attention_gradients_workspace_bytes(int64_t N, int64_t H, int64_t L, int nscans) {
    int nseg = 0, seg_chunks = 0;
    const int64_t chains = std::max<int64_t>(1, N * H);
    tp_plan(64, 64, chains, nscans, L, &nseg, &seg_chunks);
    return seg_chunks > 0 ? tp_exchange_workspace_bytes(chains * nscans, nseg, kGradStateRows) : 0;
}

int mfma_scan(const ScanDesc *scans, int nscans, int64_t N, int64_t H, int64_t L,
              void *workspace, size_t workspace_bytes, hipStream_t stream,
              const FusedAttention *fused, bool may_chain_parallel, bool forced, bool odd,
              const AttentionGradients *grads, bool clipped) {
    if (nscans < 1 || nscans > kMaxScans) return fail(FTC_ERR_INVALID, "bad scan count");
    int D, F;
    widest_rows(scans, nscans, &D, &F);
    auto tiles = [clipped](int width) { return clipped ? (width + 31) / 32 * 32 : width; };
    D = tiles(D), F = tiles(F);
    const Combo combo = combo_of(scans[0]);
    if (fused && (nscans != 1 || !fused_attention_supported(scans[0], L)))
        return fail(FTC_ERR_UNSUPPORTED, "no fused attention kernel for this shape or layout");
    const int64_t chains = std::max<int64_t>(1, N * H);
    int tpx_nseg = 0, tpx_seg_chunks = 0, tp_nseg = 0;
    int64_t widest = 0;
    for (int64_t l : {scans[0].a.stride_l, scans[0].b.stride_l, scans[0].v.stride_l, scans[0].out.stride_l})
        widest = std::max(widest, l);
    // (a whole chain is addressed through one 32-bit descriptor; a caller whose workspace is that of the
    // workgroup form gets the workgroup form)
    bool fused_tp = fused && (L + 2 * kChunk) * std::max<int64_t>(widest, 64) * 4 < 0x7fffffffLL &&
                          fused_tp_plan(D, F, chains, L, &tpx_nseg, &tpx_seg_chunks);
    const bool wide_rows = fused && fused_wide(D, F);
    if (wide_rows && !fused_tp)
        return fail(FTC_ERR_UNSUPPORTED, "no fused attention kernel for this shape or layout");
    if (fused_tp && !wide_rows && tpx_seg_chunks > 0 && !plan_only() &&
        (int64_t)workspace_bytes < tp_exchange_workspace_bytes(chains, tpx_nseg, fused_tp_state_rows(D)))
        fused_tp = false, tpx_nseg = tpx_seg_chunks = 0;
    if (grads && !attention_gradients_take(scans, nscans, *grads, N, H, L))
        return fail(FTC_ERR_UNSUPPORTED, "no kernel takes these gradients straight from their inputs");
    const bool tp_shape = grads || (!fused && may_chain_parallel && mfma_tp_takes(scans, nscans, N, H, L, forced, odd));
    const int64_t fblocks = tp_shape || wide_rows ? tp_fblocks(F) : 1;
    const int64_t blocks = odd && forced ? column_blocks(scans, nscans) : nscans * fblocks;
    if (fused_tp && tpx_seg_chunks == 0) tp_nseg = tpx_nseg, tpx_nseg = 0;
    if (tp_shape) {
        if (combo != kFFFF)
            mixed_plan(D, F, chains, nscans, L, scans[0].out.dtype != FTC_F32, has_state(scans, nscans), &tpx_nseg,
                       &tpx_seg_chunks);
        else if (odd && forced)
            tp_plan(D, 64, chains, (int)blocks, L, &tpx_nseg, &tpx_seg_chunks, forced, odd);
        else
            tp_plan(D, F, chains, nscans, L, &tpx_nseg, &tpx_seg_chunks, forced, odd);
        if (tpx_seg_chunks == 0) tp_nseg = tpx_nseg, tpx_nseg = 0;
    }
    const bool tp = tp_nseg > 0 || tpx_seg_chunks > 0;
    if (clipped ? tp || !mfma_scan_clips(D, F, nscans, L) : !tp && !mfma_scan_supported(scans[0], L))
        return fail(FTC_ERR_UNSUPPORTED, "no MFMA kernel takes a %d x %d state here", D, F);
    const bool wg = !fused_tp && !clipped && (fused || use_wg_kernel(D, F, nscans, L, combo == kFFFF));
    MfmaPlan pl = wide_rows ? MfmaPlan{} : make_plan(N, H, L, D, F, nscans, wg, fused != nullptr);
    int32_t tp_start[kMaxTpSegments + 1] = {0};
    if (tpx_seg_chunks > 0) {  // one workgroup per chain segment, segment sums exchanged
        pl.nseg = tpx_nseg;
        pl.seg_len = tpx_seg_chunks * kChunk;
        pl.waves = chains * pl.nseg;
        pl.workspace_bytes = tp_exchange_workspace_bytes(chains * blocks, pl.nseg,
                                                         fused_tp ? fused_tp_state_rows(D) : grads ? kGradStateRows : D);
    } else if (tp) {  // one workgroup per chain segment, nothing to exchange
        const bool scaled = tph_takes_rows(D) && !(odd && forced) && !fused && combo == kFFFF;  // (scan_tph_kernel)
        const TpCuts cuts = tp_cuts(D, scaled, combo == kFFFF, scans[0].out.dtype == FTC_F32, fused != nullptr, tp_nseg,
                                    (L + kChunk - 1) / kChunk);
        pl.nseg = cuts.nseg;
        for (int i = 0; i <= pl.nseg; i++) tp_start[i] = cuts.start[i];
        pl.seg_len = (int)L;
        pl.waves = chains * pl.nseg;
        pl.workspace_bytes = 0;
    }
    if (!plan_only()) {
        if (pl.workspace_bytes > 0 && (!workspace || workspace_bytes < (size_t)pl.workspace_bytes))
            return fail(FTC_ERR_WORKSPACE, "workspace of %lld bytes needed, %zu given",
                        (long long)pl.workspace_bytes, workspace_bytes);
        if (pl.workspace_bytes > 0 && (uintptr_t)workspace % 256 != 0)
            return fail(FTC_ERR_WORKSPACE, "workspace must be 256-byte aligned");
    }

    ScanArgs args;
    int64_t max_stride = 0;
    for (int i = 0; i < kMaxScans; i++) {
        const ScanDesc &sd = scans[i < nscans ? i : 0];
        ScanOperands &o = args.scan[i];
        o.a = sd.a.ptr, o.b = sd.b.ptr, o.v = sd.v.ptr;
        o.out = sd.out.ptr;
        // With a single position the row stride addresses nothing, but the kernels still
        // step over the 31 absent rows of the chunk with it: those must fall outside the
        // one-row descriptor, so a stride below the row width is replaced by the width.
        auto row_stride = [L](int64_t stride_l, int width) {
            return L == 1 ? std::max<int64_t>(stride_l, width) : stride_l;
        };
        o.d = sd.a.width, o.f = sd.v.width;
        o.a_sn = sd.a.stride_n, o.a_sh = sd.a.stride_h, o.a_sl = row_stride(sd.a.stride_l, o.d);
        o.b_sn = sd.b.stride_n, o.b_sh = sd.b.stride_h, o.b_sl = row_stride(sd.b.stride_l, o.d);
        o.v_sn = sd.v.stride_n, o.v_sh = sd.v.stride_h, o.v_sl = row_stride(sd.v.stride_l, o.f);
        o.o_sn = sd.out.stride_n, o.o_sh = sd.out.stride_h, o.o_sl = row_stride(sd.out.stride_l, o.f);
        o.rev = sd.reverse ? 1 : 0;
        // (element types of the rows, for the kernel that takes them scan by scan)
        o.pad = (sd.a.dtype == FTC_BF16 ? kRowsBf16A : 0) | (sd.b.dtype == FTC_BF16 ? kRowsBf16B : 0) |
                (sd.v.dtype == FTC_BF16 ? kRowsBf16V : 0) | (sd.out.dtype == FTC_BF16 ? kRowsBf16Out : 0);
        o.s0 = sd.initial.ptr;
        o.s0_sn = sd.initial.stride_n, o.s0_sh = sd.initial.stride_h, o.s0_sd = sd.initial.stride_d;
        o.s_out = sd.final_.ptr;
        o.so_sn = sd.final_.stride_n, o.so_sh = sd.final_.stride_h, o.so_sd = sd.final_.stride_d;
        if (fused && fused->denominators)  // (the fused form has no state to hand out)
            o.s_out = fused->denominators, o.so_sn = fused->den_sn, o.so_sh = fused->den_sh, o.so_sd = 0;
        if (grads) {  // (nor have these)
            const Operand &t = grads->rows[i < nscans ? i : 0];
            o.pad = grads->kinds[i < nscans ? i : 0];
            o.s0 = (const float *)t.ptr, o.s0_sn = t.stride_n, o.s0_sh = t.stride_h, o.s0_sd = row_stride(t.stride_l, o.f);
        }
        max_stride = std::max(max_stride, std::max(std::max(sd.a.stride_l, sd.b.stride_l),
                                                   std::max(sd.v.stride_l, sd.out.stride_l)));
    }
    // buffer descriptors address a segment with 32-bit byte offsets
    if ((int64_t)((tp ? L : (int64_t)pl.seg_len) + 2 * kChunk) * max_stride * 4 >= 0x7fffffffLL)
        return fail(FTC_ERR_UNSUPPORTED, "segment too long for 32-bit offsets");
    args.L = L;
    args.eps = fused ? fused->eps : 0.f;
    args.key_len = fused ? fused->key_lengths : grads ? grads->key_lengths : nullptr;
    args.row_dd = grads ? grads->dd : nullptr, args.row_rden = grads ? grads->rden : nullptr;
#ifdef FTC_TIMELINE
    if (tp && !fused && !grads)  // tuning aid: where the chain-parallel kernel writes its time stamps
        if (const char *env = getenv("FTC_STAMP_PTR"))  // (a build for measurements only)
            args.key_len = (const int64_t *)(uintptr_t)strtoull(env, nullptr, 0);
#endif
    args.H = (int32_t)H;
    args.seg_len = pl.seg_len;
    for (int i = 0; i <= kMaxTpSegments; i++) args.tp_start[i] = tp_start[i];
    args.tp_exchange = tpx_seg_chunks > 0 ? 1 : 0;
    args.tp_seg_chunks = tpx_seg_chunks;
    args.nseg = pl.nseg;
    args.waves_per_scan = (int32_t)pl.waves;
    args.total_waves = (int32_t)(pl.waves * blocks);
    args.tp_d = D, args.tp_fblocks = (int32_t)fblocks;
    for (int i = 0; i < kMaxScans; i++) args.tp_first[i] = (int32_t)column_blocks(scans, std::min(i, nscans));
    // very short chains: one level (every step adds the sums of all steps before it);
    // otherwise groups of about sqrt(nseg) steps, which moves fewer states per step
    args.group = pl.nseg;
    if (pl.nseg > 5) {
        args.group = 1;
        while (args.group * args.group < pl.nseg) args.group++;
    }
    // tuning aid: FTC_GROUP=<n> forces groups of n steps
    if (tuning().group >= 0) args.group = std::max(1, tuning().group);
    // a wavefront watches one flag per lane: at most 64 steps per group and 64 groups
    args.group = std::min(args.group, 64);
    while ((pl.nseg + args.group - 1) / args.group > 64) args.group++;

    const bool half_pieces = tp && tph_takes_rows(D) && !(odd && forced);
    bool mixed = false;  // rows with bf16 among them
    const bool rows_as_they_are = tp && combo != kFFFF;
    for (int i = 0; i < nscans; i++) {
        mixed = mixed || combo_of(scans[i]) != kFFFF;
        if ((!rows_as_they_are && combo_of(scans[i]) != combo) ||
            (!(tp && odd) && (tiles(scans[i].a.width) != D || tiles(scans[i].v.width) != F)))
            return fail(FTC_ERR_INVALID, "scans of one launch must share widths and dtypes");
    }
    // fp32 states of up to 64 rows: the kernel that feeds its fragments from LDS tiles
    bool dma = D <= 64 && combo == kFFFF;
    if (tuning().dma >= 0) dma = dma && tuning().dma != 0;  // tuning aid
    note_kernel(fused_tp ? (tpx_seg_chunks > 0 ? "scan_tp_kernel<NORM> (exchange)" : "scan_tp_kernel<NORM>")
                : rows_as_they_are ? (tpx_seg_chunks > 0 ? "scan_tp_bf16_kernel (exchange)" : "scan_tp_bf16_kernel")
                : tp ? (half_pieces ? (tpx_seg_chunks > 0 ? "scan_tph_kernel (exchange)" : "scan_tph_kernel")
                                  : (tpx_seg_chunks > 0 ? "scan_tp_kernel (exchange)" : "scan_tp_kernel"))
                : wg ? (fused ? "scan_wg_kernel<NORM>" : "scan_wg_kernel")
                : dma ? "scan_dma_kernel" : "scan_mfma_kernel");
    if (plan_only()) {
        char cuts[160] = "";
        if (tp && tpx_seg_chunks == 0)
            for (int i = 0, at = 0; i <= pl.nseg && at < 140; i++)
                at += snprintf(cuts + at, sizeof(cuts) - at, "%s%d", i ? "," : ", cuts at chunks ",
                               (int)args.tp_start[i]);
        note_plan("%s: %d scan%s (%s), state %d x %d, %lld chains, %d segment%s of %d rows%s, "
                  "%lld workgroups or wavefronts, workspace %lld bytes",
                  ftc_last_kernel(), nscans, nscans == 1 ? "" : "s",
                  scans[0].reverse ? "first one reverse" : "first one forward", D, F,
                  (long long)chains, (int)pl.nseg, pl.nseg == 1 ? "" : "s", (int)pl.seg_len, cuts,
                  (long long)args.total_waves, (long long)pl.workspace_bytes);
        return FTC_OK;
    }
    if (tp) {
        if (fused)
            launch_scan_tp_norm(workspace, args, stream);
        else if (mixed)
            launch_scan_tp_mixed(workspace, args, stream);
        else if (grads)
            launch_scan_tph_gradients(workspace, args, stream);
        else if (half_pieces)
            launch_scan_tph(workspace, args, odd, stream);
        else
            launch_scan_tp(workspace, args, odd, stream);
    } else if (wg) {
        launch_scan_wg_ffff(D, F, fused != nullptr, workspace, args, stream);
    } else if (dma) {
        launch_scan_dma_ffff(D, F, workspace, args, stream, clipped);
    } else switch (combo) {
        case kFFFF: launch_scan_ffff(D, F, workspace, args, stream); break;
        case kBBBF: launch_scan_bbbf(D, F, workspace, args, stream); break;
        case kFBBB: launch_scan_fbbb(D, F, workspace, args, stream); break;
        case kBFBB: launch_scan_bfbb(D, F, workspace, args, stream); break;
        case kBBFB: launch_scan_bbfb(D, F, workspace, args, stream); break;
        default: return fail(FTC_ERR_UNSUPPORTED, "no MFMA kernel for this dtype combination");
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess)
        return fail(FTC_ERR_HIP, "MFMA scan launch failed: %s", hipGetErrorString(err));
    return FTC_OK;
}

}  // namespace ftc
