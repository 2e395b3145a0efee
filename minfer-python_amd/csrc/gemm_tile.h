// The tiled kernel of the GEMM family (from 65 rows on) and its launch; compiled once per element type (gemm_tile_f16.hip,
// gemm_tile_bf16.hip).
#pragma once

#include <algorithm>

#include "gemm_common.h"

namespace minfer_attn {

typedef s16x8 __attribute__((aligned(8))) s16x8_a8;

// Tile shapes: four waves (2 x 2), a wave owning M16 x N16 blocks of 16 x 16; NS stages of the K ring in LDS (NS - 1 steps in
// flight while one is multiplied), OCC waves per SIMD.
template <int M16_, int N16_, int NS_, int OCC_ = 1> struct GemmShape {
    static constexpr int M16 = M16_, N16 = N16_, NS = NS_, OCC = OCC_, WAVES = 4;
    static constexpr int BM = 32 * M16, BN = 32 * N16;
    static constexpr int A_PANEL = BM * 128, B_PANEL = BN * 128, STAGE = A_PANEL + B_PANEL;   // bytes of one K step
    static constexpr int A_COPIES = M16, B_COPIES = N16;   // wave-wide copies (1 KiB) per wave and K step
};

// The tiled kernel: a workgroup of four waves (2 x 2) owns a BM x BN tile of D, wave (wm, wn) 16 M16 rows x 16 N16 columns of it.
// What bounds it: from a round of the largest tiles on the power budget (4096 x 14336 x 4096 and 4096^3 run at 1.6-1.7 GHz of
// 2.4 with the matrix pipes busy 74 and 76 % of the cycles, whatever the order of the instructions), below that what a wave issues between its
// MFMAs and the copies.  Four waves rather than eight read a third fewer LDS bytes per flop (a fragment feeds M16 or N16 MFMAs), and
// with one wave per SIMD everything has to fit in the 12 clocks that an MFMA leaves the issue port: a K step is one basic block, a
// copy three instructions, and reads and copies share no slot.  Eight waves (2 x 4 or 4 x 2, a copy of seven instructions, results
// stored from the registers) and seven sizes against these (clocks settled, us): 600 x 14336 x 4096 74.8 -> 66.8, 1777 x 4096 x 4096
// [K, N] 63.0 -> 55.3, 1777 x 6144 x 4096 82.5 -> 75.3, 4096^3 109 -> 101; 50 random products of 513 to 8192 rows 13 % on average,
// 70 of 65 to 600 rows (with plan_tiles) 14-18 %.
//
// [N, K] weights (NT) come as a group of up to three (the QKV projection): their columns are numbered through as one wide matrix
// of p.N columns and tiled without regard to where one weight ends (grp.end = cumulative column counts, multiples of 8): every
// copied piece of 8 weight rows and every stored piece of 8 columns lies inside one weight, which is looked up once per piece.
template <class T> MA_DEV void mfma_acc(f32x4& acc, s16x8 a, s16x8 b);
template <> MA_DEV void mfma_acc<F16>(f32x4& acc, s16x8 a, s16x8 b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
template <> MA_DEV void mfma_acc<BF16>(f32x4& acc, s16x8 a, s16x8 b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// What follows each MFMA of a slice: how many of the NR fragment reads, NC copies and NP pointer steps have been issued after
// MFMA i.  Reads lie in groups 1 .. N16 - 2; copies and pointer steps (which are in different slices) in the slots of groups
// 1 .. N16 - 1 that have no read, as evenly as these allow.
template <int M16, int N16, int NR, int NC, int NP> struct SliceOrder {
    static constexpr int S = M16 * N16, LO = M16, MID = (N16 - 2) * M16;
    int reads[S + 1], copies[S + 1], steps[S + 1];
    constexpr SliceOrder() : reads{}, copies{}, steps{} {
        int free_slots = 0;
        bool has_read[S] = {};
        for (int r = 0; r < NR; ++r) has_read[LO + r * MID / NR] = true;
        for (int i = LO; i < S; ++i) free_slots += !has_read[i];
        int r = 0, c = 0, s = 0, f = 0;
        for (int i = 0; i < S; ++i) {
            if (i >= LO) {
                while (r < NR && LO + r * MID / NR <= i) ++r;
                if (!has_read[i]) {
                    while (c < NC && c * free_slots / NC <= f) ++c;
                    while (s < NP && s * free_slots / NP <= f) ++s;
                    ++f;
                }
            }
            reads[i + 1] = r; copies[i + 1] = c; steps[i + 1] = s;
        }
    }
};

// Waits until the copies of all but the `later` most recent steps have landed, NC copies each; more than MAX of them are none.
template <int MAX, int NC> MA_DEV void wait_steps(int later) {
    if constexpr (MAX <= 0) wait_vmcnt<0>();
    else if (later >= MAX) wait_vmcnt<MAX * NC>();
    else wait_steps<MAX - 1, NC>(later);
}

template <class T, bool NT, class SH>
__global__ __launch_bounds__(SH::WAVES * 64, SH::OCC) void gemm_kernel(const GemmParams p) {
    static_assert(NT || SH::BN % 128 == 0, "a [K, N] weight is staged in sub-tiles of 128 columns");
    constexpr int kBM = SH::BM, kBN = SH::BN, NW = SH::WAVES, CA = SH::A_COPIES, CB = SH::B_COPIES, NC = CA + CB, NS = SH::NS;
    constexpr int M16 = SH::M16, N16 = SH::N16;
    __shared__ __attribute__((aligned(1024))) char lds[NS * SH::STAGE];   // stage: the A panel, then the B panel

    const int lane = threadIdx.x & 63, w = wave_id();
    const int wm = w & 1, wn = w >> 1;

    // ---- which tile ----------------------------------------------------------------------------------
    // Workgroup ids are dealt round-robin to the 8 XCDs; each gets a run of consecutive units.  The units of one K slice follow each
    // other, so that an XCD's tiles read the same part of A's and B's rows (with the slices of one tile on consecutive ids instead: 136 x 1480 x
    // 11072 23.6 -> 18.4 us, 486 x 1536 x 8960 27.1 -> 23.4, 183 x 4096 x 4096 20.6 -> 17.2).
    const bool split = p.splits > 1;
    const int tiles = p.tiles_m * p.tiles_n;
    const int unit = (int)(blockIdx.x & 7) * p.per_xcd + (int)(blockIdx.x >> 3);
    const int slice = split ? unit / tiles : 0;
    const int t = unit - slice * tiles;
    if (split ? slice >= p.splits : t >= tiles) return;
    // Tiles are numbered down bands of kGroupM tile rows, so that the tiles an XCD runs at one time form a block that
    // shares A row panels as well as B column panels in its L2 (row-major numbering made every XCD read all of B).
    constexpr int kGroupM = 4;
    const int band = t / (kGroupM * p.tiles_n), in_band = t % (kGroupM * p.tiles_n);
    const int first_m = band * kGroupM, gm = min(kGroupM, p.tiles_m - first_m);
    const int m0 = (first_m + in_band % gm) * kBM;
    const int n0 = (in_band / gm) * kBN;

    // ---- global -> LDS copies: lane offsets (bytes) from the panel's (B as [N, K]: the piece's) first element ----
    // A wave-wide copy moves a piece of 1 KiB; piece q = j*NW + w of a panel lands at 1024 q and holds
    //   A (and B as [N, K]): rows 8q .. 8q+7 of 128 bytes each;
    //   B as [K, N]:         k rows 4*(q%16) .. +3 of sub-tile q/16 (64 k rows of 256 bytes, 128 columns).
    uint32_t a_off[CA], b_off[CB];
    const short* b_src[NT ? CB : 1];   // wave-uniform
    const int kt_all = p.K / kBK;           // K steps of this workgroup: all of them, or its slice
    const int kt_first = split ? (int)((int64_t)slice * kt_all / p.splits) : 0;
    const int KT = split ? (int)((int64_t)(slice + 1) * kt_all / p.splits) - kt_first : kt_all;
    const short* a_src = (const short*)p.A + (int64_t)m0 * p.lda + (int64_t)kt_first * kBK;
#pragma unroll
    for (int j = 0; j < CA; ++j) {
        const int row = 8 * (j * NW + w) + (lane >> 3), pg = lane & 7;
        a_off[j] = (uint32_t)((int64_t)(min(m0 + row, p.M - 1) - m0) * p.lda + 8 * (pg ^ swz_row_tile(row))) * 2u;
    }
    if (!NT) b_src[0] = (const short*)p.B + (int64_t)kt_first * kBK * p.ldb + n0;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const int q = j * NW + w;
        if (NT) {
            int local;
            const int sg = group_of_unit(p.grp, min(n0 + 8 * q, p.N - 8), local);   // (past the last weight: its last rows)
            const int64_t ldj = sg == 0 ? p.grp.ldb[0] : sg == 1 ? p.grp.ldb[1] : p.grp.ldb[2];
            b_src[j] = (const short*)(sg == 0 ? p.grp.B[0] : sg == 1 ? p.grp.B[1] : p.grp.B[2]) + (int64_t)local * ldj + (int64_t)kt_first * kBK;
            const int row = lane >> 3, pg = lane & 7;
            b_off[j] = (uint32_t)((int64_t)row * ldj + 8 * (pg ^ swz_row_tile(8 * q + row))) * 2u;
        } else {
            const int sub = q >> 4, row = 4 * (q & 15) + (lane >> 4), pg = lane & 15;
            const int col = min(n0 + 128 * sub + 8 * (pg ^ swz_col_tile(row)), p.N - 8) - n0;
            b_off[j] = (uint32_t)((int64_t)row * p.ldb + col) * 2u;
        }
    }
    const int64_t b_step = NT ? kBK : (int64_t)kBK * p.ldb;   // elements from one K step to the next
    const uint32_t dst0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_addr(lds) + w * 1024));
    // copy c of a step (the wave's A copies, then its B copies) into the stage whose part for this wave is at dst
    auto copy_one = [&](uint32_t dst, auto c_tag) __attribute__((always_inline)) {
        constexpr int c = decltype(c_tag)::value;
        if constexpr (c < CA) copy16_global_to_lds_at<c * NW * 1024>(a_src, a_off[c], dst);
        else copy16_global_to_lds_at<SH::A_PANEL + (c - CA) * NW * 1024>(b_src[NT ? c - CA : 0], b_off[c - CA], dst);
    };
    // The sources of the next step's copies: pointer 0 is A's, the others B's.
    constexpr int NP = 1 + (NT ? CB : 1);
    auto advance = [&](int s) __attribute__((always_inline)) {
        if (s == 0) a_src += kBK; else b_src[s - 1] += b_step;
    };

    // ---- per-lane LDS read addresses (stage 0; block offsets are immediates) --------------------------------
    // The matrix instruction is v_mfma_f32_16x16x32 (on random fp16 operands the chip sustains 1.80-1.90 PFLOP/s of it and
    // 1.56-1.62 of v_mfma_f32_32x32x16).  It computes D^T = B^T A^T, so that a lane holds 4 consecutive n of one row m.  A K step
    // is two slices of 32 values; a fragment is 16 rows x 32 k, lane (l16, quad) holding row l16, k = 8 quad + 0..7 of the slice:
    // 16 bytes at granule (4 slice + quad) ^ swizzle of the row, which is the same for rows 16 b + l16.
    constexpr int BLK = 16 * 128;
    const int l16 = lane & 15, quad = lane >> 4;
    uint32_t m_rd[2], n_rd[NT ? 2 : N16];
    {
        const int sw = swz_row_tile(l16);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const uint32_t o = lds_addr(lds) + l16 * 128 + 16 * ((4 * ks + quad) ^ sw);
            m_rd[ks] = o + M16 * wm * BLK;
            if (NT) n_rd[ks] = o + SH::A_PANEL + N16 * wn * BLK;    // n fragments: as the m fragments
        }
        if (!NT) {
            // n fragments through transpose reads of the [k][n] sub-tile: the 16-lane group `quad` addresses k rows
            // 8 quad + 0..3 (second read: + 4) of the slice, 16 columns, and lane l16 receives column l16
            const int krow = 8 * quad + (l16 >> 2);
            const int swv = swz_col_tile(krow);
#pragma unroll
            for (int nb = 0; nb < N16; ++nb) {
                const int n = 16 * (N16 * wn + nb), col = (n & 127) + 4 * (l16 & 3);
                n_rd[nb] = lds_addr(lds) + SH::A_PANEL + (n >> 7) * kColTile + krow * 256 + 16 * ((col >> 3) ^ swv) + 2 * (col & 7);
            }
        }
    }
    // (the address of a stage is made opaque: otherwise the compiler keeps one register per block and adds the stage to each)
    auto at_stage = [&](uint32_t addr, uint32_t so) __attribute__((always_inline)) -> uint32_t {
        uint32_t x = addr + so;
        asm("" : "+v"(x));
        return x;
    };
    uint32_t m_at, n_at[NT ? 1 : N16];   // of the stage and slice that is being read
    auto read_from = [&](uint32_t so, int ks) __attribute__((always_inline)) {
        m_at = at_stage(m_rd[ks], so);
        if (NT) n_at[0] = at_stage(n_rd[ks], so);
        else if (ks == 0) {
#pragma unroll
            for (int nb = 0; nb < (NT ? 0 : N16); ++nb) n_at[nb] = at_stage(n_rd[nb], so);
        }
    };
    auto read_n = [&](int ks, int nb) __attribute__((always_inline)) -> s16x8 {
        if (NT) return lds_read_b128(n_at[0], nb * BLK);
        const s16x4 t0 = lds_read_tr16(n_at[nb], (32 * ks) * 256);
        const s16x4 t1 = lds_read_tr16(n_at[nb], (32 * ks + 4) * 256);
        return s16x8{t0[0], t0[1], t0[2], t0[3], t1[0], t1[1], t1[2], t1[3]};
    };
    auto read_m = [&](int mb) __attribute__((always_inline)) -> s16x8 { return lds_read_b128(m_at, mb * BLK); };

    // The accumulators live in the accumulation registers and are named there by the asm statement of every MFMA: left to the
    // allocator, 256 of them (and the phis of a loop with branches) spill.  What the compiler cannot see into it cannot keep the
    // distance to either: nothing but MFMAs touches them until the epilogue, which starts with the wait states (build.py looks).
    f32x4 acc[N16][M16];
#pragma unroll
    for (int nb = 0; nb < N16; ++nb)
#pragma unroll
        for (int mb = 0; mb < M16; ++mb) acc[nb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};

    // ---- main loop ---------------------------------------------------------------------------------------
    // A slice is N16 groups of M16 MFMAs (group nb: n fragment nb against every m fragment).  Both kinds of fragments are
    // double-buffered: the next slice's are read during groups 1 .. N16-2, the m fragments first.  The workgroup's only
    // barrier per K step sits after group 0 of the step's second slice: by then every read of the stage has returned, and the
    // wave's share of the next stage's copies, issued NS - 1 steps before, has landed; what follows the barrier reads the next
    // stage and copies step kt + NS into the stage just vacated.  Every MFMA, read and copy is pinned where it is written
    // (scheduling barriers): left alone the compiler moves reads down to just before their use.
    static constexpr SliceOrder<M16, N16, N16 + M16, NC, NP> order{};
    s16x8 nf[2][N16], mf[2][M16];
    auto pin = [&]() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
#pragma unroll
    for (int st = 0; st < NS; ++st) {
        if (st >= KT) break;
        if (st > 0) {
#pragma unroll
            for (int s = 0; s < NP; ++s) advance(s);
        }
        for_range<0, NC>([&](auto c) __attribute__((always_inline)) { copy_one(dst0 + st * SH::STAGE, c); });
    }
    wait_steps<NS - 1, NC>(KT - 1);   // the copies of step 0 retire first
    __syncthreads();
    read_from(0, 0);
#pragma unroll
    for (int mb = 0; mb < M16; ++mb) mf[0][mb] = read_m(mb);
#pragma unroll
    for (int nb = 0; nb < N16; ++nb) nf[0][nb] = read_n(0, nb);
    uint32_t so = 0;
    // COPY: the step that issues the copies of step kt + NS; the last NS steps have none to issue.
    auto step = [&](auto copy_tag, int in_flight) __attribute__((always_inline)) {
        constexpr bool COPY = decltype(copy_tag)::value;
        uint32_t dst = dst0 + so;
        asm("" : "+s"(dst));
        const uint32_t next = so == (NS - 1) * SH::STAGE ? 0u : so + SH::STAGE;
        for_range<0, 2 * M16 * N16>([&](auto i_tag) __attribute__((always_inline)) {
            constexpr int ks = decltype(i_tag)::value / (M16 * N16), i = decltype(i_tag)::value % (M16 * N16), nb = i / M16, mb = i % M16;
            if (i == 0) pin();
            mfma_acc<T>(acc[nb][mb], nf[ks][nb], mf[ks][mb]);
            pin();
            for_range<order.reads[i], order.reads[i + 1]>([&](auto r_tag) __attribute__((always_inline)) {
                constexpr int r = decltype(r_tag)::value;
                if constexpr (r == 0) read_from(ks == 0 ? so : next, ks ^ 1);
                if constexpr (r < M16) mf[ks ^ 1][r] = read_m(r);
                else nf[ks ^ 1][r - M16] = read_n(ks ^ 1, r - M16);
            });
            if constexpr (COPY && ks == 0) for_range<order.steps[i], order.steps[i + 1]>([&](auto s) __attribute__((always_inline)) { advance(decltype(s)::value); });
            if constexpr (COPY && ks == 1) for_range<order.copies[i], order.copies[i + 1]>([&](auto c) __attribute__((always_inline)) { copy_one(dst, c); });
            pin();
            if constexpr (ks == 1 && i == M16 - 1) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this wave has read everything it needs from this stage
                if constexpr (COPY || NS == 2) wait_vmcnt<COPY ? (NS - 2) * NC : 0>();   // and its share of the next stage has landed
                else wait_steps<NS - 2, NC>(in_flight);
                __syncthreads();
                pin();
            }
        });
        so = next;
    };
    int kt = 0;
    for (; kt + NS < KT; ++kt) step(std::true_type{}, 0);
    for (; kt < KT; ++kt) step(std::false_type{}, KT - 2 - kt);   // (what the last step reads of a next one is not used)

    // ---- epilogue: D = alpha * acc + beta * C.  Register e of a block is n = 4 quad + e, m = l16: stored from the registers an
    // instruction would write 32 bytes to each of 16 rows.  A block row of 16 rows goes through the wave's own part of the LDS
    // (rows padded by 16 bytes: no bank conflicts with N16 = 8, 4 N16 clocks a block row,
    // 0.5 % of the kernel, with 6 and 7) and leaves in 16-byte pieces of whole rows, C coming in the same way.
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");        // the last MFMAs' results
    __syncthreads();
    constexpr int ROW = N16 * 64 + 16, ITEMS = 32 * N16, IT = (ITEMS + 63) / 64;   // bytes of a padded row; pieces of 8 columns
    static_assert(NW * 16 * ROW <= NS * SH::STAGE, "the waves' areas fit the stages");
    const uint32_t area = lds_addr(lds) + w * 16 * ROW;
    int i_row[IT], i_n[IT];
    bool i_on[IT];
    short* d_col[IT];
    int64_t i_ldd[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int idx = 64 * it + lane, g = idx % (2 * N16);
        i_row[it] = idx / (2 * N16);
        i_n[it] = n0 + 16 * N16 * wn + 8 * g;
        i_on[it] = idx < ITEMS && i_n[it] < p.N;
        d_col[it] = (short*)p.D + i_n[it];
        i_ldd[it] = p.ldd;
        if (NT) {
            int local;
            const int sg = group_of_unit(p.grp, i_n[it], local);
            d_col[it] = (short*)(sg == 0 ? p.grp.D[0] : sg == 1 ? p.grp.D[1] : p.grp.D[2]) + local;
            i_ldd[it] = sg == 0 ? p.grp.ldd[0] : sg == 1 ? p.grp.ldd[1] : p.grp.ldd[2];
        }
    }
    typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
    // A block row's pieces of C are requested CD block rows before they are added (rows and columns past the end read the last ones, and the
    // lanes without a piece, an eighth of them with N16 = 7, the next rows'; giving those the last piece's place is 68 instructions more and no faster):
    // waited for as soon as requested, as they were, every one of a wave's 4 to 8 block rows costs the latency of memory, 3 to 12 us a
    // tile (with C, us, before / after: 4096^3 `[N, K]` 123.3 / 110.5, 8192 x 4096 x 4096 243.5 / 218.3, 600 x 14336 x 4096 75.1 / 67.6,
    // 1777 x 4096 x 4096 `[K, N]` 58.0 / 54.8, without C 51.4).
    auto block_rows = [&](auto c_tag) __attribute__((always_inline)) {
        constexpr bool HAS_C = decltype(c_tag)::value;
        static_assert(M16 >= 4, "block rows to request C ahead of");
        constexpr int CD = HAS_C ? 4 : 1;
        s16x8 c[CD][IT];
        auto load_c = [&](int mb) __attribute__((always_inline)) {
            const int mw = m0 + 16 * (M16 * wm + mb);
#pragma unroll
            for (int it = 0; it < IT; ++it)
                c[mb % CD][it] = *reinterpret_cast<const s16x8_a8*>((const short*)p.C + (int64_t)min(mw + i_row[it], p.M - 1) * p.ldc + min(i_n[it], p.N - 8));
        };
        if constexpr (HAS_C) {
#pragma unroll
            for (int mb = 0; mb < CD; ++mb) load_c(mb);
        }
#pragma unroll
        for (int mb = 0; mb < M16; ++mb) {
            const int mw = m0 + 16 * (M16 * wm + mb);
            if (mw >= p.M) break;
#pragma unroll
            for (int nb = 0; nb < N16; ++nb) *(lds_f32x4*)(uintptr_t)(area + l16 * ROW + 16 * (4 * nb + quad)) = acc[nb][mb];
            wave_lds_order();
#pragma unroll
            for (int it = 0; it < IT; ++it) {
                const int m = mw + i_row[it];
                if (!i_on[it] || m >= p.M) continue;
                const uint32_t at = area + (uint32_t)i_row[it] * ROW + 32 * (uint32_t)((64 * it + lane) % (2 * N16));
                const f32x4 x0 = *(const lds_f32x4*)(uintptr_t)at, x1 = *(const lds_f32x4*)(uintptr_t)(at + 16);
                if (!HAS_C && split) {   // the slice's raw sums
                    float* dst = p.part + ((int64_t)slice * p.M + m) * p.N + i_n[it];
                    *reinterpret_cast<f32x4*>(dst) = x0;
                    *reinterpret_cast<f32x4*>(dst + 4) = x1;
                    continue;
                }
                float v[8];
#pragma unroll
                for (int e = 0; e < 4; ++e) { v[e] = p.alpha * x0[e]; v[4 + e] = p.alpha * x1[e]; }
                if constexpr (HAS_C) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] += p.beta * T::to_float(c[mb % CD][it][e]);
                }
                uint4 pk;
                pk.x = T::pack2(v[0], v[1]); pk.y = T::pack2(v[2], v[3]); pk.z = T::pack2(v[4], v[5]); pk.w = T::pack2(v[6], v[7]);
                *reinterpret_cast<s16x8_a8*>(d_col[it] + (int64_t)m * i_ldd[it]) = __builtin_bit_cast(s16x8, pk);
            }
            wave_lds_order();
            if constexpr (HAS_C) if (mb + CD < M16) load_c(mb + CD);
        }
    };
    if (split || p.beta == 0.f) block_rows(std::false_type{});
    else block_rows(std::true_type{});
}

// ---- launch ------------------------------------------------------------------------------------------------
template <class T, int I> static int launch_tile(GemmParams p, bool nt, hipStream_t stream) {
    constexpr GemmTile t = kGemmTiles[I];
    using SH = GemmShape<t.m16, t.n16, t.ns, t.occ>;
    p.tiles_m = (p.M + SH::BM - 1) / SH::BM;
    p.tiles_n = (p.N + SH::BN - 1) / SH::BN;
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n;
    p.per_xcd = (int)((tiles * std::max(p.splits, 1) + 7) / 8);
    const dim3 grid((unsigned)p.per_xcd * 8), block(SH::WAVES * 64);
    if (nt) {
        if (p.grp.end[0] == 0) {   // a weight by itself is a group of one
            p.grp.B[0] = p.B; p.grp.D[0] = p.D; p.grp.ldb[0] = p.ldb; p.grp.ldd[0] = p.ldd;
            p.grp.N[0] = p.grp.end[0] = p.grp.end[1] = p.grp.end[2] = p.N;
        }
        hipLaunchKernelGGL((gemm_kernel<T, true, SH>), grid, block, 0, stream, p);
    } else {
        if constexpr (t.n16 % 4 == 0) hipLaunchKernelGGL((gemm_kernel<T, false, SH>), grid, block, 0, stream, p);
        else return fail(MINFER_ATTN_EINVAL, "gemm_kernel: a [K, N] weight takes tiles of 128 or 256 columns");
    }
    return check_launch("gemm_kernel");
}
template <class T, int... I> static int launch_tile_of(const GemmParams& p, bool nt, int tile, hipStream_t stream, std::integer_sequence<int, I...>) {
    int rc = MINFER_ATTN_OK;
    (void)((I == tile && (rc = launch_tile<T, I>(p, nt, stream), true)) || ...);
    return rc;
}
template <class T> static int launch_gemm_tile(const GemmParams& p, bool nt, int tile, hipStream_t stream) {
    return launch_tile_of<T>(p, nt, tile, stream, std::make_integer_sequence<int, kGemmTileCount>{});
}

}  // namespace minfer_attn
