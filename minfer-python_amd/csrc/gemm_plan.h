// Which kernel of the GEMM family takes a call, in which tiles and in how many K slices: the rules on sizes, types and alignment, with
// what was measured on both sides of each line.  Host code only, without a GPU header, so that the rules can be run on their own.
#pragma once

#include <math.h>
#include <stdint.h>

#include <algorithm>

namespace minfer_attn {

constexpr int kBK = 64;                     // K values of a step of the tiled kernels
constexpr int kRowsSeg = 128;               // ... of a segment of gemm_rows_lds_kernel
constexpr int kStripeSeg = 256;             // ... of the stripe kernels
constexpr int kGemvSegHalfs = 4096;         // ... of gemv_kernel
constexpr int kGemvMaxKHalfs = 16384;       // the longest activation row that gemv_kernel keeps in LDS: 32 KiB

// The tiled kernel's shapes: 32 m16 x 32 n16, ns stages, occ workgroups to a unit (GemmShape).  The more there are the closer a
// problem's tiles come to whole rounds of the chip (plan_tiles); of the 26 from 128 to 256 in steps of 32 these lose 0.3 % to all
// over random shapes (256 x 192 takes 4096 x 6144 x 4096 in two rounds: 163.8 us, the others 167.8 at best).  A [K, N] weight is
// staged in sub-tiles of 128 columns and takes those whose n16 is a multiple of 4.
struct GemmTile { int m16, n16, ns, occ; };
constexpr GemmTile kGemmTiles[] = {
    {8, 8, 2, 1}, {8, 7, 2, 1}, {7, 8, 2, 1}, {6, 8, 2, 1}, {5, 8, 3, 1}, {4, 8, 3, 1}, {7, 6, 3, 1}, {6, 6, 3, 1},
    {4, 6, 3, 1}, {5, 7, 3, 1}, {7, 4, 3, 1}, {6, 4, 3, 1}, {5, 4, 3, 1}, {4, 4, 3, 1}, {4, 4, 2, 2}, {8, 6, 2, 1}};
constexpr int kGemmTileCount = sizeof(kGemmTiles) / sizeof(kGemmTiles[0]);

// ---- few rows against an [N, K] weight -----------------------------------------------------------------------

// gemm_rows_lds_kernel: four waves that take a segment each.
inline bool rows_lds_takes(int64_t M, int64_t K) { return M <= 16 && K % (4 * kRowsSeg) == 0; }
// gemv_kernel: one to four rows that its LDS area holds.
inline bool gemv_takes(int64_t M, int64_t K) { return M >= 1 && M <= 4 && K <= kGemvMaxKHalfs && (M == 1 || (K > kGemvSegHalfs && M * K <= 2 * kGemvMaxKHalfs)); }
// gemm_stripe_kernel.  Which widths it takes (in stripes of 64 columns; weights coming from memory): from 96 on every row count that reaches
// it (14336 x 4096 at 2-32 rows 21.6-22.4 us, the 16-column kernels 23.2-40.5); an output head from 5 rows on (128256 x 4096 at 8
// rows 164 against 182, 57344 x 8192 160 against 186; at 2-4 rows the kernels that keep more workgroups on a compute unit
// were ahead, 166-170 against 176-178, and on another chip behind, 165-169 against 161-163); narrower ones down to 32 stripes from 5 rows on, up to 8 when their rows are long enough to matter, against the 16-column
// and few-row kernels (us: 2048 x 4096 at 16 / 17 / 64 rows 9.6 / 7.8, 14.0 / 8.6, 21.5 / 14.0; 5120 x 5120 at 5 / 16 rows 14.9 / 12.9,
// 20.4 / 14.5; 3072 x 8192 at 8 / 32 rows 14.9 / 12.8, 29.8 / 17.2; 4096 x 14336 at 8 / 64 rows 24.3 / 22.8, 70.8 / 44.1).
inline bool stripe_takes(int64_t M, int64_t stripes, int64_t K) {
    if (M < 1 || M > 64 || K % kStripeSeg != 0) return false;
    if (stripes > 640) return M >= 5;
    return stripes >= 96 || (stripes >= 80 && M >= 8) || (stripes >= 32 && M >= 5 && (M > 8 || K >= 2560));
}
// Where it is also ahead of its K slices, whose workgroups copy less each but leave partial sums to be added up (us, slices / whole rows;
// weights from memory: calls cycling over 640 MiB of copies, half of which and less the last-level cache would serve, 3584 x 8192 at 32 rows 17.7 or 13.5 for
// whole rows; without C, which costs slices 0.1 and whole rows 0.3 up to 16 rows, 0.6 to 1.4 from 17 on).
// By the rows a unit copies, (NB + MB) x 16 of K values, the narrower the weight the fewer, since below 48 stripes a quarter of the units and
// more have no column block, and from 65 to 79 a few units have two where the others have one: 4096 x 14336 at 9 / 16 rows 23.6 / 22.9, 24.1 / 24.3; 3584 x 8192
// at 16 15.1 / 13.9; 2560 x 5120 at 16 10.2 / 10.2; 2048 x 8192 at 5 10.2 / 12.0, 2048 x 4096 at 32 / 33 10.1 / 9.8, 10.4 / 10.5; 4608 x 4096 at 33 / 48 / 64
// 14.3 / 13.8, 14.9 / 15.2, 15.7 / 17.2; 5632 x 4096 at 33 / 64 15.8 / 14.2, 18.1 / 17.7; 6144 x 4096 at 64 18.5 / 17.8.
// From 17 rows on, where gemm_reduce_kernel adds up, the rows themselves count and up to 64 stripes the line is lower, in proportion to the units that have a
// block: 2560 x 5120 at 28 / 32 rows 11.4 / 12.2, 11.7 / 13.1; 3072 x 4096 at 40 / 48 11.9 / 11.5, 12.2 / 12.3; 4096 x 4096 at 48 / 56 / 64 13.1 / 12.7, 13.5 / 14.1,
// 13.8 / 14.6 (62 and 63 stripes alike); 4096 x 6144 at 32 / 36 15.2 / 14.9, 16.1 / 16.3; 3584 x 6144 at 28 / 32 14.1 / 13.9, 14.3 / 14.6.  Rows of 8192 values
// keep whole rows longer: 4096 x 8192 at 24 / 28 / 32 17.7 / 16.2, 17.9 / 16.9, 17.9 / 18.0; 3584 x 8192 at 20 / 24 15.8 / 15.1, 15.8 / 16.0.
// Over 1500 sizes of 32 to 64 stripes, 2560 to 14336 values and 17 to 64 rows the choice is 0.3 % behind the better one.
inline bool stripe_blocks_pay(int64_t M, int64_t stripes, int64_t K) {
    if (!stripe_takes(M, stripes, K)) return false;
    if (stripes >= 96) return true;
    if (M > 16 && stripes <= 64 && (16 + M) * K > std::max<int64_t>(224000, (K >= 8192 ? 5800 : 4800) * stripes)) return false;
    const int64_t most = stripes < 48 ? 16000 : stripes <= 64 || stripes >= 80 ? 25000 : 22000;
    return ((stripes > 64 ? 2 : 1) + (M + 15) / 16) * K <= most;
}
// A weight of fewer than 192 stripes: with a workspace, K slices bring the workgroups up to the chip's 256 compute units
// (every slice four segments at least); the slices' sums are added up by finish_slices or gemm_reduce_kernel (slices_meet).
// 1 = no slices.
inline int stripe_slices(int64_t M, int64_t N, int64_t K) {
    const int64_t stripes = (N + 63) / 64;
    if (M < 1 || M > 64 || K % kStripeSeg != 0 || N % 8 != 0 || stripes >= 192) return 1;
    return (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(256 / stripes, K / kStripeSeg / 4), 16));
}

// ---- few rows against a [K, N] weight ------------------------------------------------------------------------

// [K, N] weights of up to 64 rows: slices of K bring the column tiles up to the chip's 256 compute units, every slice two
// steps of 64 at least; from 17 rows on four and at most 32 slices, since the sums grow with the rows.  The workspace is for these; a call that
// has it takes 8 or 16 of them at most.
constexpr int64_t kKnRows = 64;
inline int kn_slices(int64_t M, int64_t N, int64_t K) {
    if (M < 1 || M > kKnRows || K % kBK != 0 || K < 8 * kBK || N % 8 != 0) return 1;
    const int64_t tiles = (N + 127) / 128;
    return (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(256 / tiles, K / kBK / (M <= 16 ? 2 : 4)), M <= 16 ? 64 : 32));
}

// ---- who adds the K slices up ----------------------------------------------------------------------------------
// Whether the slices of stripe_slices or kn_slices meet inside the launch (finish_slices; where the stream has counters): up to kMeetRows
// rows, which is what its threads have pieces for.  Both rules stay at 256 workgroups, so two slices and more are of at most kMeetTiles tiles and
// the sums are 2 MiB at most.  Written through to where every XCD sees them they are as fast as a second launch or faster up to 1 MiB, and level or behind
// above it (us, weights from memory, in a loop of calls, inside / second launch: `[K, N]` 4 x 4096 x 4096, 0.5 MiB, 10.5 / 10.9; 8 x 4096 x 4096, 1 MiB, 11.0 / 11.0; 16 x 2048 x
// 8192, 2 MiB in 16 slices, 12.9 / 12.2; 16 x 8192 x 4096, 2 MiB in four, 17.0 / 17.1; `[N, K]` 9 x 2048 x 8192 10.4 / 10.8, 16 x 1024 x 14336 in 14 slices 12.0 / 11.1; Q8_0 8 x
// 8192 x 8192 18.3 / 18.8), but the launch is 2.7 us of the host's, which bounds the steps of so few rows.  The slices of gemm_kernel go to a second launch, which
// spreads over the chip what its tiles' last workgroups would add up (17 x 528 x 1152 9.5 / 8.7, 40 x 808 x 1600 13.3 / 9.8, 24 x 3424 x 1408 11.3 / 9.7).
constexpr int kMeetRows = 16, kMeetTiles = 128;
inline bool slices_meet(int64_t M) { return M <= kMeetRows; }

// ---- which tiles, how many K slices --------------------------------------------------------------------------
inline int64_t tile_count(int64_t M, int64_t N, int64_t bm, int64_t bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); }
// Microseconds of a launch of `tiles` tiles in `slices` K slices each, weights from memory: whole rounds of the chip, the last,
// partly filled one at 0.76 + 0.24 of its share (its units run faster), a round its K steps at 20 ns per pair of 16-row blocks (two
// workgroups on a unit 1.84 of one; with two stages a step that is shorter than the largest tile's does not cover its copies) and
// 3.8 us of first and last copies and results; the copies of all tiles at 31 TB/s and the weight at 7 TB/s, which are hidden behind
// that in part: the three add up as their squares; past one round, where the clock has come down to what the power budget leaves, the
// more the more a tile copies per flop (3072 x 8192 x 4096: 128 x 256 tiles 177.7 us, 192 x 256 167.1, without this estimated 171.7 and
// 172.9; 4096 x 5120 x 4096 150.9 and 137.0); 3.6 us around it, 0.9 more for the launch that adds the slices up, and 0.29 us
// per MB of sums.  Fitted to 4700 timed calls (150 shapes of 65 to 7000 rows, both layouts, up to 40 choices each), whose sums were added up by
// one load after the other: the choice it made was 1.0 % behind the best one on average, fixed rules for 128 x 128 and 128 x 256 slices and a
// table of rounds 6 %.  With gemm_reduce_kernel as it is, 100 shapes for which slices and whole rows are estimated to be close (70 of them within 12 %), ten
// choices each, weights from memory: 2.4 % behind the best one without C and 2.1 % with it, 10 of the 100 in slices where whole rows are faster and 9 the other way
// round, so the line has no side that it leans to; the constants of the sums that would be best for these alone (1.7 us, 0.20 us per MB) are 1.8 % behind.
inline double plan_cost(const GemmTile& t, int64_t tiles, int slices, int64_t M, int64_t N, int64_t K, int cus) {
    const double steps = (double)((K / kBK + slices - 1) / slices), area = t.m16 * t.n16;
    const double step = (0.0201 * area + 0.0738) * (t.occ == 2 ? 1.84 : 1.0) + (t.ns == 2 && t.occ == 1 ? 0.0147 + 0.0076 * (64 - area) : 0.0);
    const int64_t wgs = tiles * slices, per = (int64_t)cus * t.occ, full = wgs / per, rest = wgs % per;
    const double rounds = (double)full + (rest ? 0.76 + 0.24 * (double)rest / (double)per : 0.0);
    const double power = wgs > per ? 1.0 + ((t.m16 + t.n16) / area - 0.25) : 1.0;
    const double compute = rounds * (step * steps + 3.8) * power, weight = (double)N * (double)K * 2 / 7.0e6;
    const double copies = (double)tiles * (double)(K / kBK) * (t.m16 + t.n16) * 4096 / 31.3e6;
    const double launch = 3.6 + sqrt(compute * compute + copies * copies + weight * weight);
    return slices > 1 ? launch + 0.9 + 0.286e-6 * slices * (double)M * (double)N * 4 : launch;
}
// The cheapest tile shape and number of slices, up to max_slices of them (what a workspace holds): slices that bring the
// workgroups to one or two rounds of the chip or just below, 3 steps long at least, with 64 MiB of sums at most.
constexpr int64_t kMostSlices = 32;
struct TilePlan { int tile, slices; };
inline TilePlan plan_tiles(int64_t M, int64_t N, int64_t K, bool nt, int64_t max_slices, int cus) {
    const int64_t room = std::min<int64_t>(std::min<int64_t>(kMostSlices, max_slices), std::min<int64_t>(K / kBK / 3, (INT64_C(16) << 20) / (M * N)));
    TilePlan best{0, 1};
    double cost = 0;
    for (int i = 0; i < kGemmTileCount; ++i) {
        const GemmTile& t = kGemmTiles[i];
        if (!nt && t.n16 % 4 != 0) continue;
        const int64_t tiles = tile_count(M, N, 32 * t.m16, 32 * t.n16), fill = (int64_t)cus * t.occ / tiles;
        if (t.occ == 2 && tiles * std::max<int64_t>(room, 1) <= cus) continue;   // one workgroup to a unit: the other entry's three stages
        const int64_t options[5] = {1, fill, fill - 1, fill * 3 / 4, 2 * fill};
        for (int o = 0; o < 5; ++o) {
            if (options[o] > room && options[o] != 1) continue;
            if (options[o] < 1 || (o > 0 && options[o] == 1)) continue;
            const double c = plan_cost(t, tiles, (int)options[o], M, N, K, cus);
            if (cost == 0 || c < cost) { cost = c; best = {i, (int)options[o]}; }
        }
    }
    return best;
}
// plan_tiles, remembered: estimating takes a microsecond and more, and a call asks twice (for the workspace and to launch), as does every
// next token or chunk for all the projections of a layer.  The last 16 plans of a thread, looked through from one end to the other
// (4 to 10 ns): a place by some hash of the sizes is shared sooner or later by the projections of one model, which then push each other out.  A
// plan depends on nothing but what it is looked up by.
constexpr int kPlansKept = 16;
inline TilePlan tile_plan(int64_t M, int64_t N, int64_t K, bool nt, int64_t max_slices, int cus) {
    struct Entry { int64_t M, N, K, max_slices; int nt, cus; TilePlan plan; };
    static thread_local Entry kept[kPlansKept];
    static thread_local unsigned oldest = 0;
    max_slices = std::min<int64_t>(max_slices, kMostSlices);
    for (const Entry& e : kept)
        if (e.M == M && e.N == N && e.K == K && e.max_slices == max_slices && e.nt == (int)nt && e.cus == cus) return e.plan;
    Entry& e = kept[oldest];
    oldest = (oldest + 1) % kPlansKept;
    e = Entry{M, N, K, max_slices, (int)nt, cus, plan_tiles(M, N, K, nt, max_slices, cus)};
    return e.plan;
}
// Slices that a workspace is sized for: the plan's, and no fewer than bring 128 x 128 tiles to one round of the chip (to two while
// a slice stays 16 steps long), four steps long at least: the size has been that, and callers may keep a workspace by it.
inline int gemm_slices(int64_t M, int64_t N, int64_t K, bool nt, int cus) {
    if (K <= 0 || K % kBK != 0 || N % 8 != 0) return 1;
    int64_t s = 1;
    const int64_t tiles = tile_count(M, N, 128, 128), kt = K / kBK;
    if (tiles <= 256 && kt >= 8) {
        s = std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(256 / tiles, kt / 4), 32));
        if (tiles >= 64 && tiles * s <= 256 && kt / (2 * s) >= 16 && (s >= 2 || kt >= 192)) s *= 2;
    }
    return std::max((int)s, tile_plan(M, N, K, nt, kMostSlices, cus).slices);
}

// ---- the dispatch ----------------------------------------------------------------------------------------------
// Which kernel, and for the sliced ones (stripe_slices, kn_rows, tiles) in how many K slices; `tile` is an index of kGemmTiles.
enum class GemmKernel { plain, gemv, rows_lds, skinny, stripe, stripe_slices, kn_rows, tiles };
struct GemmRoute { GemmKernel kernel; int slices, tile; };

// `fast`: sizes, strides and alignment are those of the kernels that move 16-byte pieces and whole K steps.  `fit`: slices of M x N fp32
// sums that the workspace holds.  `units`: says how many compute units the chip has.
//
// A decode step's few tokens against an [N, K] weight: stream the weight once.  Which kernel does that best was
// measured with the calls cycling over copies of the weight, 640 MiB in all: a weight of up to 256 MiB called again
// and again is served by the chip's last-level cache, where the order of the kernels is a different one (14336 x
// 4096 at one row: stripes 18.0 us against 19.5 for whole rows per wave from the cache, 21.7-24.2 against 21.7-21.9 from memory).
// These calls are bound by the host: no rule for up to 16 rows asks for a plan of tiles.
inline GemmRoute gemm_route(int64_t M, int64_t N, int64_t K, bool nt, bool fast, int64_t fit, int (*units)()) {
    if (!fast) return {GemmKernel::plain, 1, 0};
    if (nt && M <= 64) {
        const int64_t stripes = (N + 63) / 64;
        const bool rows_takes = rows_lds_takes(M, K);
        // one row: whole weight rows per wave (14336 x 4096: 21.7-21.9 us, the 16-column kernel 23.2-23.6, stripes 21.7-24.2; 28672 x 8192:
        // 75-76 / 91 / 81-97); a weight under 32 M values goes to the 16-column kernel when it takes it (4096 x 4096: 8.4 against 10.6)
        if (M == 1 && K <= kGemvMaxKHalfs && (N * K >= (INT64_C(1) << 25) || !rows_takes)) return {GemmKernel::gemv, 1, 0};
        // two to four rows against long rows of a wide weight go the same way, every weight piece multiplied with the same
        // piece of each activation row (28672 x 8192 at 2-4 rows: 77.5-82.6 us against 92-95 for the 16-column kernel, 10240 x
        // 8192 at 2-3 rows 32.1-34.6 against 36.3-38.8; 8192 x 8192 29.2-33.9 against 29.2-30.9, and rows of 4096 values gain nothing)
        if (M >= 2 && gemv_takes(M, K) && K >= 8192 && N >= 10240 && (M <= 3 || N >= 16384)) return {GemmKernel::gemv, 1, 0};
        // up to 4 rows (8 where stripe_takes says no) against fewer than 96 stripes, and up to 4 against an output head: the 16-column
        // kernel (128256 x 4096 at 2-4 rows 166-170 against 176-178, on another chip 165-169 against 161-163; 28672 x 4096 at 2-8 rows 41.6-44.8 against 38.5-39.1 and 14336 x
        // 4096 23.2-25.6 against 21.7-21.8: those go on)
        const bool rows_first = rows_takes && ((M <= 8 && stripes < 96 && !stripe_takes(M, stripes, K)) || (M <= 4 && stripes > 640));
        const int slices = stripe_slices(M, N, K);
        const bool sliceable = slices > 1 && fit >= slices;
        // ... except long rows of a narrow weight when a workspace allows K slices: one wave per 16 columns walks a whole row
        // by itself (1024 x 14336 at 2-8 rows 16.5-20.8 us, in slices 10.5-10.9; 1536 x 8960 15.1-17.4 and 9.3-9.8; 2048 x
        // 8192 at 5-8 rows 12.4-13.4 and 10.2-10.3.  The lines are those of slices that took a second launch; now that they meet inside it 2048 x 8192 at
        // 2-4 rows, 11.4-12.0 and 10.1, and rows of 6144 values, 1536 x 6144 at 2-8 rows 8.8-10.4 and 8.4-8.8, would gain as well)
        const bool long_rows_few_stripes = K >= 8192 && ((M >= 5 && stripes <= 32) || (M >= 2 && stripes <= 24));
        if (rows_first && !(sliceable && long_rows_few_stripes)) return {GemmKernel::rows_lds, 1, 0};
        // with a workspace, K slices of the stripes, from 9 rows on, where whole rows are not ahead (stripe_blocks_pay): up to 16 rows only for 25 M
        // weight values or rows of 6144 values and more (2048 x 8192 at 9-16 rows 10.5-11.0 against 13.9-16.7 for the 16-column kernel, 1024 x 14336 11.3-12.1 against
        // 21.6-26.9), from 17 rows on for 8 M values (1536 x 5632 and the like: gemm_skinny_kernel is the other choice)
        const bool slices_pay = !stripe_blocks_pay(M, stripes, K) && (long_rows_few_stripes || (M >= 9 && (N * K >= INT64_C(25000000) || K >= 6144 || (M >= 17 && N * K >= (INT64_C(1) << 23)))));
        if (sliceable && slices_pay) return {GemmKernel::stripe_slices, slices, 0};
        if (stripe_takes(M, stripes, K)) return {GemmKernel::stripe, 1, 0};
        if (rows_takes) return {GemmKernel::rows_lds, 1, 0};
        if (M == 1 && K <= kGemvMaxKHalfs) return {GemmKernel::gemv, 1, 0};
        if (M <= 16) return {GemmKernel::skinny, 1, 0};
        if ((M <= 32 || N * K <= (INT64_C(1) << 25)) && !(fit > 1 && tile_plan(M, N, K, nt, kMostSlices, units()).slices > 1)) return {GemmKernel::skinny, 1, 0};
    }
    if (!nt && M <= kKnRows) {
        // eight slices at most, 16 for rows of 80 K steps and more, and for up to 1024 columns from 17 rows on (eight / 16: 512 x 4096 at 17 / 64 rows 8.9 / 7.8,
        // 10.6 / 9.5; 1024 x 4096 9.2 / 8.5, 11.3 / 11.0; 1536 x 4096 at 17 / 64 9.5 / 9.0, 12.2 / 12.4; 2048 x 4096 at 40 11.1 / 11.8): further ones save less streaming than their sums
        // cost (us, weights from memory, as many as fill the chip / these: 1000 x 4096 at 1 / 9 / 16 rows 10.4 / 7.7, 13.2 / 8.9, 15.1 / 9.6; 2560 x 2560 at 12 10.1 / 8.2;
        // 1024 x 14336 at 9 / 40 15.2 / 12.8, 14.3 / 14.6; 512 x 8192 at 9 16.6 / 9.8; minfer_gemm_workspace_bytes stays that of filling it)
        const int most = std::min(kn_slices(M, N, K), K >= 80 * kBK || (M > 16 && N <= 1024) ? 16 : 8);   // a smaller workspace: as many of these as it holds (40 x 4096 x 4096: none 31.7 us, two 20.9, four 14.6, all eight 12.6)
        return {GemmKernel::kn_rows, std::max((int)std::min<int64_t>(most, fit), 1), 0};
    }
    TilePlan plan = tile_plan(M, N, K, nt, kMostSlices, units());
    if (plan.slices > std::max<int64_t>(fit, 1)) plan = tile_plan(M, N, K, nt, std::max<int64_t>(fit, 1), units());
    return {GemmKernel::tiles, plan.slices, plan.tile};
}

// ---- weights stored as Q8_0 blocks -----------------------------------------------------------------------------
constexpr int64_t kQ8SkinnyRows = 64;       // up to here the kernels that stream the blocks; above, dequantise once and run the tiles
constexpr int kGemvMaxK = 16384;            // the longest activation row that gemv_q8_kernel keeps in LDS: 32 KiB

// the streaming kernel takes up to 64 rows, needs weight rows that are multiples of 4 bytes (an even number of blocks)
// and stores 8-byte pieces of D (N a multiple of 4); every other shape goes through the dequantised weight
inline bool q8_streams(int64_t M, int64_t N, int64_t K) { return M <= kQ8SkinnyRows && (K / 32) % 2 == 0 && N % 4 == 0; }
// Where gemm_stripe_q8_kernel over whole rows is ahead of its K slices and of gemm_skinny_q8_kernel on a weight of fewer than 192 stripes: rows of up to 4096 values, by the rows a
// unit copies, (NB + MB) x 16 of K values (us, the other / it: 8192 x 4096 at 2 / 16 / 32 rows 11.8 / 11.0, 12.7 / 11.1, 14.9 / 12.8;
// 6144 x 4096 at 16 / 24 / 40 rows 12.3 / 11.0, 14.1 / 12.1, 15.2 / 15.4; 6144 x 2048 at 16 rows 9.1 / 6.7; 5120 x 4096 at 24 / 40 12.6 /
// 12.0, 14.0 / 15.1; 4096 x 4096 at 16 / 64 9.7 / 8.2, 13.9 / 13.2; 4096 x 2048 at 8 / 16 / 64 5.4 / 5.9, 8.7 / 5.5, 11.7 / 8.6; 2048 x 4096
// at 16 / 24 / 40 8.8 / 8.0, 9.9 / 9.6, 10.7 / 11.2; 5120 x 5120 at 16 rows 12.1 / 12.7).  64 stripes are 253 to 256 column blocks, one to a unit
// with no unit idle, and have a line of their own: 4096 x 4096 still gains at 64 rows, 20480 by this count.
inline bool q8_blocks_pay(int64_t M, int64_t N, int64_t K) {
    const int64_t stripes = (N + 63) / 64, rows = (stripes > 64 ? 2 : 1) + (M + 15) / 16;
    if (K > 4096 || M < 2 || M > 64 || stripes < 32 || stripes >= 192) return false;
    if (stripes >= 96) return rows * K <= 17000 && (M >= 8 || N * K >= INT64_C(20000000));
    return M >= 16 && rows * K <= (stripes < 64 ? 12500 : stripes == 64 ? 20500 : 17000);
}
// K slices of gemm_stripe_q8_kernel for a weight of fewer than 192 stripes when a workspace is given (1 = none): 256 / stripes workgroups
// per chunk of four blocks, full chunks whatever the width (weights coming from memory: 4096 x 14336 at 16 / 32 / 64 rows
// 19.0 / 21.8 / 26.4 us against 29.6 / 43.0 / 68.4 for gemm_skinny_q8_kernel, 8192 x 8192 at 2-64 rows 19.6-28.5 against
// 23.7-40.3, 6144 x 4096 12.4-17.7 against 12.7-22.2; 4096 x 4096 up to 8 rows 10.2 against 7.7-8.3: two launches, so a
// weight of 16 M values or fewer only from 16 rows on, or from 8 when its rows are 6144 values and longer, or from 2
// when they are 8192 values and longer and the stripes 24 at most, as for the 16-bit weights).
inline int q8_slices(int64_t M, int64_t N, int64_t K) {
    if (M < 2 || M > 64 || K % kStripeSeg != 0 || N % 8 != 0) return 1;
    const bool long_rows = (K >= 6144 && M >= 8) || (K >= 8192 && N <= 24 * 64);
    if (N * K <= (INT64_C(1) << 24) && M < 16 && !long_rows) return 1;
    return stripe_slices(M, N, K);
}
// gemm_stripe_q8_kernel.  Which calls it takes: 2-64 rows, whole segments of 8 blocks, rows that start on 16-byte boundaries, and a weight wide
// enough for two and a half blocks per workgroup, or two from 16 rows, or one and a half above 32 (weights coming from memory:
// 14336 x 4096 at 2-16 rows 16.7-16.9 us against 20.8-26.8 for gemm_skinny_q8_kernel, 64 rows 23.4 against 50.9; 28672 x
// 4096 29.7-43.4 against 36.8-97.7), or q8_blocks_pay.  Chunks of as many blocks as a workgroup has, as for the 16-bit weights (11008 x 4096
// at 2 / 24 / 64 rows 15.4 -> 13.3, 18.4 -> 15.6, 23.3 -> 20.6; 18944 x 3584 at 2 / 40 rows 25.6 -> 21.6, 34.1 -> 31.3): all of a
// chunk's blocks are dequantised and multiplied, there or not (skipping the missing ones of four by a branch cost the full chunks a
// third).
inline bool q8_stripe_ok(int64_t M, int64_t N, int64_t K, bool aligned) {
    return M >= 2 && M <= 64 && K % kStripeSeg == 0 && aligned &&
           (N >= 10240 || (N >= 8192 && M >= 16) || (N >= 6144 && M > 32) || q8_blocks_pay(M, N, K));
}

// Which of the kernels that stream the blocks takes a call that q8_streams.  `aligned`: the weight starts on a 16-byte boundary (its rows
// of whole segments, 272 bytes each, then do too); `fit` as in gemm_route.
enum class Q8Kernel { gemv, stripe, stripe_slices, skinny };
struct Q8Route { Q8Kernel kernel; int slices; };
inline Q8Route q8_route(int64_t M, int64_t N, int64_t K, bool aligned, int64_t fit) {
    // one row of whole segments: whole weight rows per wave
    if (M == 1 && K % 256 == 0 && K <= kGemvMaxK && aligned) return {Q8Kernel::gemv, 1};
    const int slices = aligned && !q8_blocks_pay(M, N, K) ? q8_slices(M, N, K) : 1;
    if (slices > 1 && fit >= slices) return {Q8Kernel::stripe_slices, slices};
    return {q8_stripe_ok(M, N, K, aligned) ? Q8Kernel::stripe : Q8Kernel::skinny, 1};
}

// More rows than the kernels that stream the blocks take: the rows of each of the calls of theirs in which a product goes all
// the same (the last one takes what remains; M: none, the weight is dequantised).  Dequantising writes and reads back twice the blocks' bytes; a second call reads the blocks again,
// from the last-level cache mostly (us, weights from memory, dequantised / in parts): 65 rows x 14336 x 4096 64.0 / 39.4, 4096 x 14336
// 61.7 / 42.3, 128256 x 4096 488 / 288, 6144 x 4096 32.8 / 28.6, 4096 x 4096 24.4 / 21.8; 128 rows 72.1 / 46.3, 70.3 / 49.7, 496 / 337,
// 37.3 / 34.8, 26.3 / 27.0; 160 rows in three 76.2 / 64.9, 73.9 / 69.8, 507 / 483, 40.4 / 48.1; 192 28672 x 4096 124 / 128.
// Judged by the parts as they run, the shorter last one too: every one has to be a product that a kernel streams (a part that is not
// dequantises the weight by itself), and the stripe kernels have to take it, or else the dequantised weight is one that
// the tiled kernel does not take (N no multiple of 8: 65 x 4100 x 4096 3645 us, in parts through gemm_skinny_q8_kernel 40).
inline int64_t q8_part_rows(int64_t M, int64_t N, int64_t K, bool aligned) {
    if (M <= kQ8SkinnyRows || M > 160 || N * K < (M <= 96 ? INT64_C(16000000) : M <= 128 ? INT64_C(20000000) : INT64_C(50000000))) return M;
    const int64_t parts = (M + kQ8SkinnyRows - 1) / kQ8SkinnyRows, rows = ((M + parts - 1) / parts + 15) / 16 * 16;
    for (const int64_t r : {rows, M - (parts - 1) * rows}) {
        // (the room of the dequantised weight holds the slices of a part)
        if (!q8_streams(r, N, K) || (N % 8 == 0 && q8_route(r, N, K, aligned, kMostSlices).kernel == Q8Kernel::skinny)) return M;
    }
    return rows;
}

}  // namespace minfer_attn
