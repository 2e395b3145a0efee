// Half-precision GEMM for gfx950: D = alpha * A x B + beta * C with fp32 accumulation on the MFMA units.
//
// What the reference computes (reference: src/minfer/kernels/torch_ext/csrc/cuda/gemm/op.cuh:218-316,
// oracle src/minfer/kernels/refs.py:49-51, tests test/kernels.py:119-216): A is [M, K] activations (leading
// dims flattened), B is the weight either as [K, N] ("A x B", what its tuned kernel handles) or as [N, K]
// ("A x B^T", the layout of its QKV projection, whose launcher is empty in the reference), C and D are [M, N].
//
// Design.  From 65 rows on a workgroup of four waves owns a tile of D of 128 to 256 rows and columns (gemm_tile.h) and walks K in
// steps of 64; the A and B panels of a step are copied global->LDS without passing through registers into a ring of two or three
// stages, one barrier per step.  Which tile, and whether K is cut into slices that meet in a workspace, is what plan_tiles (gemm_plan.h,
// which has the rules of the dispatch) estimates to be quickest.  Up to 64 rows the work is reading the weight once: the kernels of this file.
#include <algorithm>
#include <atomic>
#include <type_traits>
#include <utility>

#include "gemm_common.h"
#include "quant_q8.h"

namespace minfer_attn {

// ---- K slices that meet inside the launch -------------------------------------------------------------------
// A slice's sums go to the workspace; the workgroup of a tile that comes last (a counter per tile) adds the tile's slices up
// and stores D: no second launch, which costs the host 2.7 us and the chip 4, as much as many of these products take
// themselves.  The sums pass from one XCD's L2 to another's, so they are written and read with device-scope accesses, which
// go past the L2s on both sides, and a workgroup counts itself only when its own have arrived (each thread waits for its stores,
// the barrier for the threads).  The reader's loads come after the count: its value decides whether they run at all, thread 0
// has it before the second barrier, and no load moves up over a barrier in the compiler or in the wave.  In the memory model
// that is not an order, since nothing here is a release or an acquire; with both on the count it would be, and then every arrival
// writes back its XCD's L2 and invalidates it (a single user's attention block, whose decode and output projection merge this way,
// 37.7 -> 40.1 us).  Slices are added in their order whoever comes last, as gemm_reduce_kernel adds them, which takes over where
// there are no counters (stream_counters: any stream but the null stream).
MA_DEV void store_slice4(const GemmParams& p, int slice, int m, int n, f32x4 v) {
    float* at = p.part + ((int64_t)slice * p.M + m) * p.N + n;
    if (!p.done) { *reinterpret_cast<f32x4*>(at) = v; return; }
    uint64_t* dst = reinterpret_cast<uint64_t*>(at);
    const u32x4 b = __builtin_bit_cast(u32x4, v);
    __hip_atomic_store(dst, ((uint64_t)b[1] << 32) | b[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(dst + 1, ((uint64_t)b[3] << 32) | b[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
MA_DEV f32x4 load_slice4(const GemmParams& p, int slice, int m, int n) {
    uint64_t* src = reinterpret_cast<uint64_t*>(p.part + ((int64_t)slice * p.M + m) * p.N + n);
    const uint64_t lo = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint64_t hi = __hip_atomic_load(src + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __builtin_bit_cast(f32x4, u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)});
}
// Called by all THREADS threads of a slice's workgroup after their store_slice4: columns n0 .. n1 - 1 (multiples of 4, four
// at least and COLS at most) of all the rows, one at least and kMeetRows at most (slices_meet); `flag`: a shared word.
template <class T, int THREADS, int COLS>
MA_DEV void finish_slices(const GemmParams& p, int tile, int n0, int n1, int* flag) {
    static_assert(kMeetRows * COLS / 4 <= 2 * THREADS, "two pieces of four columns a thread");
    if (!p.done) return;
    // C is requested before it is known who adds up, while the sums are on their way (pieces past the last one read that one's place), and a
    // thread without a piece reads no sums (us, before / after: 16 x 2560 x 2560 `[K, N]` 9.0 /
    // 8.3, 4096 x 4096 at one row 9.7 / 9.4, 16 x 2048 x 8192 `[N, K]` 10.8 / 10.3, Q8_0 10.5 / 10.1; requested with the slices 8 x 1000 x 4096 was slower, 7.6 / 7.8, now 7.5)
    const int n4 = (n1 - n0) >> 2, total = p.M * n4;
    int m[2], n[2];
    s16x4 c[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int i = min((int)threadIdx.x + e * THREADS, total - 1), r = i / n4;
        m[e] = r; n[e] = n0 + 4 * (i - r * n4);
        c[e] = load_c4(p, m[e], n[e]);
    }
    wait_vmcnt<0>();   // the thread's sums have arrived
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t before = __hip_atomic_fetch_add(p.done + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = before == (uint32_t)(p.splits - 1);
        if (*flag) __hip_atomic_store(p.done + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!*flag || (int)threadIdx.x >= total) return;
    // two pieces and eight slices at a time, so that sixteen loads of a thread are in flight
    f32x4 sum[2], x[2][8];
#pragma unroll
    for (int e = 0; e < 2; ++e) sum[e] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < p.splits; s0 += 8) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int u = 0; u < 8; ++u) x[e][u] = load_slice4(p, min(s0 + u, p.splits - 1), m[e], n[e]);
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (s0 + u < p.splits) sum[e] = s0 + u == 0 ? x[e][u] : sum[e] + x[e][u];
    }
    store_result<T>(p, m[0], n[0], sum[0], c[0]);
    if ((int)threadIdx.x + THREADS < total) store_result<T>(p, m[1], n[1], sum[1], c[1]);
}

// Up to 64 rows against a weight stored [K, N] (what a square weight is taken for): the work is reading the weight once.  A
// workgroup of four waves owns 128 columns over a slice of K; 64 k rows of its columns (16 KiB, 256 consecutive bytes of each
// row) and the activations' 64 values are a stage, copied global -> LDS, and a ring of six or seven stages fills the LDS: the
// whole slice of a 4096 x 4096 weight is in flight at once.  A wave multiplies all rows with its 32 columns, the weight
// fragments through transpose reads as in gemm_kernel.  The 128-row tiles that took these calls before copied 16 KiB of
// activation rows per stage whatever M is, with two stages in flight (one row of 4096 x 4096 13.1 -> 9.5 us, with the slices
// added up inside the launch).
template <int MB> struct KnRowsGeom {
    static constexpr int CA = (2 * MB + 3) / 4, CB = 4, NC = CA + CB;   // wave-wide copies per wave and stage (8 activation rows, 4 k rows each)
    static constexpr int A_BYTES = 4096 * CA, B_BYTES = 16384;         // (the activation copies past 16 MB rows land behind them)
    static constexpr int NS = MB <= 2 ? 7 : 6;                          // 140 / 144 KiB
};
template <class T, int MB>
__global__ __launch_bounds__(4 * 64) void gemm_kn_rows_kernel(const GemmParams p) {
    using G = KnRowsGeom<MB>;
    constexpr int NS = G::NS;
    __shared__ __attribute__((aligned(1024))) char b_lds[NS][G::B_BYTES];
    __shared__ __attribute__((aligned(1024))) char a_lds[NS][G::A_BYTES];
    const int lane = threadIdx.x & 63, w = wave_id(), l16 = lane & 15, quad = lane >> 4;
    const int tile = (int)blockIdx.x / p.splits, slice = (int)blockIdx.x - tile * p.splits;
    const int n0 = tile * 128;
    const int kt_all = p.K / kBK, kt_first = slice * kt_all / p.splits, KT = (slice + 1) * kt_all / p.splits - kt_first;

    uint32_t a_off[G::CA], b_off[G::CB];
#pragma unroll
    for (int j = 0; j < G::CA; ++j) {
        const int row = 8 * (4 * j + w) + (lane >> 3);
        a_off[j] = (uint32_t)((int64_t)min(row, p.M - 1) * p.lda + 8 * ((lane & 7) ^ swz_row_tile(row & 63))) * 2u;
    }
#pragma unroll
    for (int j = 0; j < G::CB; ++j) {
        const int row = 4 * (4 * j + w) + (lane >> 4);
        b_off[j] = (uint32_t)((int64_t)row * p.ldb + min(n0 + 8 * ((lane & 15) ^ swz_col_tile(row)), p.N - 8)) * 2u;
    }
    auto issue = [&](int t, int st) {
        const int64_t k0 = (int64_t)(kt_first + t) * kBK;
        const short* ab = (const short*)p.A + k0;
        const short* bb = (const short*)p.B + k0 * p.ldb;
#pragma unroll
        for (int j = 0; j < G::CB; ++j) copy16_global_to_lds<true>(bb, b_off[j], &b_lds[st][1024 * (4 * j + w)]);
#pragma unroll
        for (int j = 0; j < G::CA; ++j) copy16_global_to_lds<true>(ab, a_off[j], &a_lds[st][1024 * (4 * j + w)]);
    };
    // fragment addresses in stage 0 (see gemm_kernel)
    uint32_t m_rd[2], n_rd[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) m_rd[ks] = lds_addr(&a_lds[0][0]) + l16 * 128 + 16 * ((4 * ks + quad) ^ swz_row_tile(l16));
    {
        const int krow = 8 * quad + (l16 >> 2);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const int col = 32 * w + 16 * nb + 4 * (l16 & 3);
            n_rd[nb] = lds_addr(&b_lds[0][0]) + krow * 256 + 16 * ((col >> 3) ^ swz_col_tile(krow)) + 2 * (col & 7);
        }
    }
    f32x4 acc[2][MB];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
    // this wave's copies of all but the `later` most recently issued stages have landed (copies retire in order)
    auto wait_later = [&](int later) {
        if (later >= 5) wait_vmcnt<5 * G::NC>();
        else if (later == 4) wait_vmcnt<4 * G::NC>();
        else if (later == 3) wait_vmcnt<3 * G::NC>();
        else if (later == 2) wait_vmcnt<2 * G::NC>();
        else if (later == 1) wait_vmcnt<G::NC>();
        else wait_vmcnt<0>();
    };
#pragma unroll
    for (int t = 0; t < NS - 1; ++t)
        if (t < KT) issue(t, t);
    int st = 0;
    for (int t = 0; t < KT; ++t) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // step t - 1 has been read
        wait_later(min(NS - 2, KT - 1 - t));
        __syncthreads();                                     // ... by every wave, and step t has landed for every wave
        if (t + NS - 1 < KT) issue(t + NS - 1, st == 0 ? NS - 1 : st - 1);
        const uint32_t ao = st * G::A_BYTES, bo = st * G::B_BYTES;
        st = st == NS - 1 ? 0 : st + 1;
        s16x8 nf[2][2], mf[2][MB];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                const s16x4 t0 = lds_read_tr16(n_rd[nb] + bo, 32 * ks * 256), t1 = lds_read_tr16(n_rd[nb] + bo, (32 * ks + 4) * 256);
                nf[ks][nb] = s16x8{t0[0], t0[1], t0[2], t0[3], t1[0], t1[1], t1[2], t1[3]};
            }
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) mf[ks][mb] = lds_read_b128(m_rd[ks] + ao, mb * (kRowTile / 4));
        }
        __builtin_amdgcn_sched_barrier(0);   // all reads first
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int nb = 0; nb < 2; ++nb)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = T::mfma16(nf[ks][nb], mf[ks][mb], acc[nb][mb]);
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int m = 16 * mb + l16;
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
            const int n = n0 + 32 * w + 16 * nb + 4 * quad;
            if (m >= p.M || n >= p.N) continue;
            if (p.splits > 1) store_slice4(p, slice, m, n, acc[nb][mb]);
            else store_result<T>(p, m, n, acc[nb][mb]);
        }
    }
    if (p.splits > 1) {
        __shared__ int last_s;
        finish_slices<T, 4 * 64, 128>(p, tile, n0, min(n0 + 128, p.N), &last_s);
    }
}

// Few rows of A (the tokens of a decode step) against a weight stored [N, K]: the work is reading the weight once.
// A workgroup owns 16 columns n of D and all K; its 8 waves split K, each streaming its slice of the 16 weight rows
// (non-temporal 32-byte pieces per lane, four lanes covering one 128-byte line of a row) into the A operand of
// v_mfma_f32_16x16x32, the rows of A (from L2) being the B operand, 16 at a time; the waves' partial sums meet in LDS.
// Within a 64-wide K step lane (row, quad) takes k = 16*quad + 0..15 for both operands, which is just another order
// of the contraction.  MB = ceil(M / 16) <= 4.
constexpr int kSkinnyWaves = 8;
// NR groups of 16 columns per workgroup (2 for wide weights: half as many workgroups, each A fragment used twice)
template <class T, int MB, int NR, bool GROUPED = false>
__global__ __launch_bounds__(kSkinnyWaves * 64) void gemm_skinny_kernel(const GemmParams p) {
    __shared__ f32x4 part[kSkinnyWaves][NR][MB][64];
    const int lane = threadIdx.x & 63, w = wave_id();
    const int l16 = lane & 15, quad = lane >> 4;
    int n0 = (int)blockIdx.x * 16 * NR;
    const short* Bg = (const short*)p.B;
    short* Dg = (short*)p.D;
    int N = p.N;
    int64_t ldb = p.ldb, ldd = p.ldd;
    if (GROUPED) {   // the workgroup's weight, output and place inside them (uniform)
        int local;
        const int sg = group_of_unit(p.grp, (int)blockIdx.x, local);
        n0 = local * 16 * NR;
        Bg = (const short*)(sg == 0 ? p.grp.B[0] : sg == 1 ? p.grp.B[1] : p.grp.B[2]);
        Dg = (short*)(sg == 0 ? p.grp.D[0] : sg == 1 ? p.grp.D[1] : p.grp.D[2]);
        N = sg == 0 ? p.grp.N[0] : sg == 1 ? p.grp.N[1] : p.grp.N[2];
        ldb = sg == 0 ? p.grp.ldb[0] : sg == 1 ? p.grp.ldb[1] : p.grp.ldb[2];
        ldd = sg == 0 ? p.grp.ldd[0] : sg == 1 ? p.grp.ldd[1] : p.grp.ldd[2];
    }
    const int steps = p.K / 64, per = (steps + kSkinnyWaves - 1) / kSkinnyWaves;
    const int s0 = w * per, s1 = min(steps, s0 + per);
    const short* wrow[NR];
#pragma unroll
    for (int nr = 0; nr < NR; ++nr) wrow[nr] = Bg + (int64_t)min(n0 + 16 * nr + l16, N - 1) * ldb + 16 * quad;
    const short* xrow[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) xrow[mb] = (const short*)p.A + (int64_t)min(16 * mb + l16, p.M - 1) * p.lda + 16 * quad;
    f32x4 acc[NR][MB];
#pragma unroll
    for (int nr = 0; nr < NR; ++nr)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nr][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int s = s0; s < s1; ++s) {
        const int k0 = 64 * s;
        s16x8 w0[NR], w1[NR];
#pragma unroll
        for (int nr = 0; nr < NR; ++nr) {
            w0[nr] = stream_load(reinterpret_cast<const s16x8*>(wrow[nr] + k0));
            w1[nr] = stream_load(reinterpret_cast<const s16x8*>(wrow[nr] + k0 + 8));
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const s16x8 x0 = *reinterpret_cast<const s16x8*>(xrow[mb] + k0);
            const s16x8 x1 = *reinterpret_cast<const s16x8*>(xrow[mb] + k0 + 8);
#pragma unroll
            for (int nr = 0; nr < NR; ++nr) {
                acc[nr][mb] = T::mfma16(w0[nr], x0, acc[nr][mb]);
                acc[nr][mb] = T::mfma16(w1[nr], x1, acc[nr][mb]);
            }
        }
    }
#pragma unroll
    for (int nr = 0; nr < NR; ++nr)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) part[w][nr][mb][lane] = acc[nr][mb];
    __syncthreads();
    // wave j adds up block (nr, mb) = (j / MB, j % MB): register r of a lane is n = n0 + 16*nr + 4*quad + r, m = 16*mb + l16
    if (w >= NR * MB) return;
    const int nr = w / MB, mb = w - nr * MB;
    f32x4 sum = part[0][nr][mb][lane];
#pragma unroll
    for (int ww = 1; ww < kSkinnyWaves; ++ww) sum += part[ww][nr][mb][lane];
    const int m = 16 * mb + l16, n = n0 + 16 * nr + 4 * quad;
    if (m >= p.M || n >= N) return;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = p.alpha * sum[e];
    if (p.beta != 0.f) {
        const s16x4 c = *reinterpret_cast<const s16x4*>((const short*)p.C + (int64_t)m * p.ldc + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += p.beta * T::to_float(c[e]);
    }
    uint2 pk;
    pk.x = T::pack2(v[0], v[1]);
    pk.y = T::pack2(v[2], v[3]);
    *reinterpret_cast<uint2*>(Dg + (int64_t)m * ldd + n) = pk;
}

template <class T, int NR>
static void launch_skinny_nr(const GemmParams& p, hipStream_t stream) {
    const dim3 grid((p.N + 16 * NR - 1) / (16 * NR)), block(kSkinnyWaves * 64);
    const int mb = (p.M + 15) / 16;
    if (mb == 1) hipLaunchKernelGGL((gemm_skinny_kernel<T, 1, NR>), grid, block, 0, stream, p);
    else if (mb == 2) hipLaunchKernelGGL((gemm_skinny_kernel<T, 2, NR>), grid, block, 0, stream, p);
    else if (mb == 3) hipLaunchKernelGGL((gemm_skinny_kernel<T, 3, NR>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((gemm_skinny_kernel<T, 4, NR>), grid, block, 0, stream, p);
}
// The few-row kernel for large weights.  gemm_skinny_kernel's weight loads put 16 different weight rows into every
// quarter of a wave, 16 cache lines touched for 256 bytes, and that, not HBM, is what it runs at (4.5 TB/s of the weight
// at any row count).  Here the weight rows and the activation rows take the long way round: global -> LDS copies whose
// lanes walk along the rows (a copy instruction moves 256 consecutive bytes of each of four rows, 4 lines per quarter
// wave), and the MFMA fragments are read back from LDS.  A workgroup of four waves owns 16 columns; wave w takes every
// fourth 128-wide K segment, each wave with its own two-stage LDS area (no barrier until the final sum): per segment
// 4 copies for the 16 weight rows, 4 for up to 16 activation rows, 4 MFMAs.  Four rows of a copy share a 1 KiB block
// of LDS, blocks 64 bytes apart in the banks, so that the 16 rows of a fragment read hit 16 different bank groups.
constexpr int kRowsBlock = 1024 + 64;                          // LDS bytes of four rows' segment, padded
constexpr int kRowsStage = 4 * kRowsBlock;                     // 16 rows
// XI: copy instructions that hold activation rows (four rows each, M <= 4 * XI); fragment columns past them multiply
// whatever their LDS block holds into output columns that are never stored.
// GROUPED: the 16-column groups of up to three weights numbered through (p.grp.end in groups), alpha = 1 and no C.
template <class T, int XI, bool GROUPED>
__global__ __launch_bounds__(4 * 64) void gemm_rows_lds_kernel(const GemmParams p) {
    __shared__ __attribute__((aligned(16))) char wx[4][2][2][kRowsStage];   // [wave][stage][weights, activations]
    __shared__ f32x4 part[4][64];
    const int lane = threadIdx.x & 63, w = wave_id();
    const int l16 = lane & 15, quad = lane >> 4;
    int n0 = (int)blockIdx.x * 16;
    const short* Bg = (const short*)p.B;
    short* Dg = (short*)p.D;
    int N = p.N;
    int64_t ldb = p.ldb, ldd = p.ldd;
    if (GROUPED) {   // the workgroup's weight, output and place inside them (uniform)
        int local;
        const int sg = group_of_unit(p.grp, (int)blockIdx.x, local);
        n0 = local * 16;
        Bg = (const short*)(sg == 0 ? p.grp.B[0] : sg == 1 ? p.grp.B[1] : p.grp.B[2]);
        Dg = (short*)(sg == 0 ? p.grp.D[0] : sg == 1 ? p.grp.D[1] : p.grp.D[2]);
        N = sg == 0 ? p.grp.N[0] : sg == 1 ? p.grp.N[1] : p.grp.N[2];
        ldb = sg == 0 ? p.grp.ldb[0] : sg == 1 ? p.grp.ldb[1] : p.grp.ldb[2];
        ldd = sg == 0 ? p.grp.ldd[0] : sg == 1 ? p.grp.ldd[1] : p.grp.ldd[2];
    }
    const int nseg = p.K / kRowsSeg;                           // a multiple of 4: every wave the same number
    const int per = nseg / 4;
    // copy instruction i of a segment: lane L takes piece L >> 2 of row 4i + (L & 3)
    const short* wsrc[4];
    const short* xsrc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        wsrc[i] = Bg + (int64_t)min(n0 + 4 * i + (lane & 3), N - 1) * ldb + 8 * (lane >> 2);
        xsrc[i] = (const short*)p.A + (int64_t)min(4 * i + (lane & 3), p.M - 1) * p.lda + 8 * (lane >> 2);
    }
    auto issue = [&](int t, int stage) {                       // the wave's t-th segment
        const int k0 = (4 * t + w) * kRowsSeg;
#pragma unroll
        for (int i = 0; i < 4; ++i) copy16_global_to_lds(wsrc[i] + k0, &wx[w][stage][0][i * kRowsBlock]);
#pragma unroll
        for (int i = 0; i < XI; ++i) copy16_global_to_lds(xsrc[i] + k0, &wx[w][stage][1][i * kRowsBlock]);
    };
    // fragment of k step s (32 values) for row r = l16: piece 4s + quad of the row, inside the row's block of four
    const int frag = (l16 >> 2) * kRowsBlock + 16 * (l16 & 3) + 64 * quad;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    issue(0, 0);
    for (int t = 0; t < per; ++t) {
        if (t + 1 < per) { issue(t + 1, (t + 1) & 1); wait_vmcnt<4 + XI>(); } else wait_vmcnt<0>();
        const char* wb = &wx[w][t & 1][0][frag];
        const char* xb = &wx[w][t & 1][1][frag];
#pragma unroll
        for (int s = 0; s < kRowsSeg / 32; ++s) {
            const s16x8 a = *reinterpret_cast<const s16x8*>(wb + 256 * s);
            const s16x8 b = *reinterpret_cast<const s16x8*>(xb + 256 * s);
            acc = T::mfma16(a, b, acc);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // the fragments are in registers before the stage is refilled
    }
    part[w][lane] = acc;
    __syncthreads();
    if (w != 0) return;
    f32x4 sum = part[0][lane];
#pragma unroll
    for (int ww = 1; ww < 4; ++ww) sum += part[ww][lane];
    const int m = l16, n = n0 + 4 * quad;      // register r of a lane: weight row n + r, activation row m
    if (m >= p.M || n >= N) return;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = GROUPED ? sum[e] : p.alpha * sum[e];
    if (!GROUPED && p.beta != 0.f) {
        const s16x4 c = *reinterpret_cast<const s16x4*>((const short*)p.C + (int64_t)m * p.ldc + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += p.beta * T::to_float(c[e]);
    }
    uint2 pk;
    pk.x = T::pack2(v[0], v[1]);
    pk.y = T::pack2(v[2], v[3]);
    *reinterpret_cast<uint2*>(Dg + (int64_t)m * ldd + n) = pk;
}
// (16 rows at most, K a multiple of 512)
template <class T, bool GROUPED = false>
static int launch_rows_lds(const GemmParams& p, int groups, hipStream_t stream) {
    const dim3 grid(groups), block(4 * 64);
    if (p.M <= 4) hipLaunchKernelGGL((gemm_rows_lds_kernel<T, 1, GROUPED>), grid, block, 0, stream, p);
    else if (p.M <= 8) hipLaunchKernelGGL((gemm_rows_lds_kernel<T, 2, GROUPED>), grid, block, 0, stream, p);
    else if (p.M <= 12) hipLaunchKernelGGL((gemm_rows_lds_kernel<T, 3, GROUPED>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((gemm_rows_lds_kernel<T, 4, GROUPED>), grid, block, 0, stream, p);
    return check_launch("gemm_rows_lds_kernel");
}

// Up to 64 rows against an [N, K] weight (a batch of decode steps against a projection, FFN or output-head weight): a workgroup
// of four waves takes NB blocks of 16 columns at a time over the whole of K; K goes by in segments of 256 values, the 16 NB weight
// rows and the activation rows copied global -> LDS with instructions whose lanes walk along the rows (512 consecutive bytes
// of each of two rows, 2 lines per quarter wave); two or three weight stages and two or three
// activation stages, one workgroup per compute unit (segments of 128 values and two workgroups per unit are 15-25 %
// slower from 24 rows on).  No K slices across workgroups, so no partial sums in memory: the activations are read once
// per workgroup and the weight once.  Two rows of a copy share a 1 KiB block of LDS; inside block i
// the 16-byte pieces of a row sit at piece ^ (i & 7), so the 16 rows of a fragment read hit 16 different bank groups
// without padding.
// What bounds it, once the weight does not (5 TB/s), is the copies a unit makes, 50-60 bytes per ns: NB is what the workgroups have,
// one to four, and the four waves share the copies of the rows there are.  (With chunks of four whatever the workgroup had, the missing rows copied again, us, before / now: 6144 x 4096 at
// 16 / 32 / 40 / 64 rows 10.9 / 10.0, 13.7 / 11.0, 14.1 / 12.4, 15.9 / 15.1; 4096 + 1024 + 1024 columns at 24 / 40 rows 13.5 / 11.1, 15.1 /
// 12.5; 11008 x 4096 at 40 rows 20.4 / 19.5, 22016 x 4096 40.2 / 35.2; where chunks of four are still the choice, 28672 x 4096 at 64
// rows 48.2 / 46.0, for the even share of the copies.)
constexpr int kStripeBlock = 1024;                             // LDS bytes of two rows' segment
template <int MB, int NB = 4> struct StripeGeom {   // 16-row blocks of activations, 16-column blocks of the weight
    static constexpr int W_BYTES = NB * 8 * kStripeBlock;      // 16 * NB weight rows
    static constexpr int X_BYTES = MB * 8 * kStripeBlock;      // 16 * MB activation rows
    // 120 / 144 / 144 / 128 KiB with four blocks, 48 / 72 / 96 / 120 with one; a fourth and fifth stage of the smaller chunks cost 2-7 % (3072 x
    // 8192 at 16 rows 10.3 -> 11.1 us, 6144 x 4096 at 32 10.6 -> 11.0, Q8_0 14336 x 4096 at 16 16.7 -> 18.2)
    static constexpr int WST = NB == 4 && MB >= 4 ? 2 : 3, XST = MB + NB >= 7 ? 2 : 3;
    static constexpr int CW = 2 * NB, CX = 2 * MB;             // copies per wave and segment
};
// Copies issued after those of segment t, with `after` segments behind it: those of x(t) go out in front of w(t + WST - XST).
template <class G> constexpr int copies_behind(int after) {
    const int w = std::min(after, G::WST - 1) - (G::WST > G::XST ? G::WST - G::XST - 1 : 0);
    return std::max(w, 0) * G::CW + std::min(after, G::XST - 1) * G::CX;
}
// ... which is how many may be outstanding once segment t has landed
template <class G> MA_DEV void wait_behind(int after) {
    static_assert(G::WST <= 3 && G::XST <= G::WST, "three cases");
    if (after >= 2) wait_vmcnt<copies_behind<G>(2)>();
    else if (after >= 1) wait_vmcnt<copies_behind<G>(1)>();
    else wait_vmcnt<0>();
}
// SLICED: p.splits workgroups per stripe, each over its share of the segments; they leave raw fp32 sums in p.part
// ([slice][M][N]) for finish_slices.
// GROUPED: the stripes of up to three weights numbered through (p.grp.end in stripes), alpha = 1 and no C.
template <class T, int MB, bool SLICED = false, bool GROUPED = false, int NB = 4>
__global__ __launch_bounds__(4 * 64) void gemm_stripe_kernel(const GemmParams p) {
    static_assert(!(SLICED && GROUPED), "the grouped launch has no workspace");
    using G = StripeGeom<MB, NB>;
    constexpr int WST = G::WST, XST = G::XST;
    __shared__ __attribute__((aligned(16))) char w_lds[WST][G::W_BYTES];
    __shared__ __attribute__((aligned(16))) char x_lds[XST][G::X_BYTES];
    const int lane = threadIdx.x & 63, w = wave_id();
    const int l16 = lane & 15, quad = lane >> 4;
    int slice = 0, seg0 = 0, nseg = p.K / kStripeSeg;
    if (SLICED) {
        slice = (int)blockIdx.x % p.splits;
        seg0 = slice * nseg / p.splits;
        nseg = (slice + 1) * nseg / p.splits - seg0;
    }
    // Which columns.  SLICED: workgroup b / splits owns stripe b / splits.  Plain launches: the 16-column blocks of the weight
    // are shared out evenly: workgroup g of G owns blocks g * blocks / G ..
    // (g + 1) * blocks / G - 1 and goes through them NB at a time, a chunk ending early at the end of the workgroup's
    // range; its missing rows are the last one again (from L2) and
    // what they multiply is never stored.  Every compute unit so streams the same share of the weight to within one block,
    // whatever the number of columns (448 stripes of 64 columns are one and three quarter rounds of 256 workgroups:
    // 28672 x 4096 from memory 46.5 -> 41.5-42.3 us), and a narrow weight is spread over the whole chip.
    // GROUPED: every weight has a run of workgroups of its own (p.grp.end counts them, cumulatively; the host hands them
    // out in proportion to the weights' blocks), and a workgroup's share is worked out inside its weight, once, before the
    // chunk loop: with the lookup of a chunk's weight inside the loop the grouped launch ran 20 us where the plain one ran
    // 11, for the same instructions and the same L2 traffic.
    int blk_first = SLICED ? 4 * ((int)blockIdx.x / p.splits) : (int)((int64_t)blockIdx.x * p.tiles_n / (int)gridDim.x);
    int blk_last = SLICED ? min(blk_first + 4, p.tiles_n) : (int)((int64_t)(blockIdx.x + 1) * p.tiles_n / (int)gridDim.x);
    const short* Bg = (const short*)p.B;
    short* Dg = (short*)p.D;
    int Nw = p.N;
    int64_t ldb = p.ldb, ldd = p.ldd;
    if (GROUPED) {   // the workgroup's weight, output and place among that weight's workgroups (uniform)
        int idx;
        const int sg = group_of_unit(p.grp, (int)blockIdx.x, idx);
        Bg = (const short*)(sg == 0 ? p.grp.B[0] : sg == 1 ? p.grp.B[1] : p.grp.B[2]);
        Dg = (short*)(sg == 0 ? p.grp.D[0] : sg == 1 ? p.grp.D[1] : p.grp.D[2]);
        Nw = sg == 0 ? p.grp.N[0] : sg == 1 ? p.grp.N[1] : p.grp.N[2];
        ldb = sg == 0 ? p.grp.ldb[0] : sg == 1 ? p.grp.ldb[1] : p.grp.ldb[2];
        ldd = sg == 0 ? p.grp.ldd[0] : sg == 1 ? p.grp.ldd[1] : p.grp.ldd[2];
        const int wgs = (sg == 0 ? p.grp.end[0] : sg == 1 ? p.grp.end[1] - p.grp.end[0] : p.grp.end[2] - p.grp.end[1]);
        const int blocks = (Nw + 15) / 16;
        blk_first = (int)((int64_t)idx * blocks / wgs);
        blk_last = (int)((int64_t)(idx + 1) * blocks / wgs);
    }
    for (int cb = blk_first; cb < blk_last;) {
    const int local = cb;
    const int nb = min(NB, blk_last - cb);
    int N = Nw;
    N = min(N, 16 * (local + nb));                             // rows past the chunk are not this chunk's
    // copy instruction for row pair i: lane L lands at byte 16 L of the block and fetches piece (L >> 1) ^ (i & 7) of row
    // 2i + (L & 1); the wave's pairs are w, w + 4, .., eight in a row in K slices, whose chunks are full (40 rows of 6144 x 4096
    // 14.1 against 14.3 us)
    auto pair = [&](int j) { return SLICED ? 8 * w + j : w + 4 * j; };
    const short* wsrc[2 * NB];
#pragma unroll
    for (int j = 0; j < 2 * NB; ++j)
        wsrc[j] = Bg + (int64_t)min(16 * local + 2 * pair(j) + (lane & 1), N - 1) * ldb + 8 * ((lane >> 1) ^ (pair(j) & 7));
    const short* xsrc[2 * MB];                                 // this wave's share of the activation rows: row pairs w, w + 4, ...
#pragma unroll
    for (int j = 0; j < 2 * MB; ++j)
        xsrc[j] = (const short*)p.A + (int64_t)min(2 * (w + 4 * j) + (lane & 1), p.M - 1) * p.lda + 8 * ((lane >> 1) ^ ((w + 4 * j) & 7));
    // A chunk starts at segment (its place in the weight) mod nseg and wraps: the chunks running at one time then read
    // different segments of the activation rows instead of the same few lines of the same few L2 channels
    const int rot = (int)((SLICED ? blockIdx.x : (unsigned)(local >> 2)) % (unsigned)nseg);
    auto seg_k0 = [&](int t) { const int sg = t + rot; return (seg0 + (sg >= nseg ? sg - nseg : sg)) * kStripeSeg; };
    auto issue_w = [&](int t) {
        char* st = w_lds[t % WST];
        const int k0 = seg_k0(t);
#pragma unroll
        for (int j = 0; j < 2 * NB; ++j) copy16_global_to_lds(wsrc[j] + k0, st + pair(j) * kStripeBlock);
    };
    auto issue_x = [&](int t) {
        char* st = x_lds[t % XST];
        const int k0 = seg_k0(t);
#pragma unroll
        for (int j = 0; j < 2 * MB; ++j) copy16_global_to_lds(xsrc[j] + k0, st + (w + 4 * j) * kStripeBlock);
    };
    // Wave w multiplies k steps 2w and 2w + 1 of every segment for all 64 columns and all rows: every fragment is read
    // from LDS once per workgroup (a wave that owned 16 columns over the whole segment would read all activation
    // fragments, four times the traffic), and the four partial sums meet in LDS after the last segment.  Fragment of k
    // step s for row r = l16 of a 16-row set: piece 4s + quad of the row, in pair block r >> 1.
    const int row_off = (l16 >> 1) * kStripeBlock + 16 * (l16 & 1);
    int frag[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) frag[s] = row_off + 32 * ((4 * (2 * w + s) + quad) ^ (l16 >> 1));
    f32x4 acc[NB][MB];
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[c][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < WST - 1; ++t) {
        if (t < XST - 1 && t < nseg) issue_x(t);
        if (t < nseg) issue_w(t);
    }
    for (int t = 0; t < nseg; ++t) {
        __syncthreads();                                       // every wave has read segment t - 1: its stages may be refilled
        if (t + XST - 1 < nseg) issue_x(t + XST - 1);
        if (t + WST - 1 < nseg) issue_w(t + WST - 1);
        // segment t has landed once at most the copies issued after it are outstanding
        const int after = nseg - 1 - t;
        wait_behind<G>(after);
        __syncthreads();                                       // ... for every wave's copies
        const char* wb = w_lds[t % WST];
        const char* xb = x_lds[t % XST];
        // all fragments of the wave's two k steps first, then the MFMAs: left to itself the compiler pipelines these reads
        // in one instantiation and waits for each before its MFMA in another (the grouped one ran twice as long for it)
        s16x8 a[2][NB], b[2][MB];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) b[s][mb] = *reinterpret_cast<const s16x8*>(xb + mb * 8 * kStripeBlock + frag[s]);
#pragma unroll
            for (int c = 0; c < NB; ++c) a[s][c] = *reinterpret_cast<const s16x8*>(wb + c * 8 * kStripeBlock + frag[s]);
        }
        __builtin_amdgcn_sched_barrier(0);                     // (the scheduler moves nothing across this)
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int c = 0; c < NB; ++c)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) acc[c][mb] = T::mfma16(a[s][c], b[s][mb], acc[c][mb]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // fragments in registers before the barrier that frees the stage
    }
    // partial sums of the four waves: wave u leaves column block c at red[u][c][mb][lane]; wave w adds up column block w
    // in the order of the waves
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(&w_lds[0][0]);   // 16 MB KiB of the 96
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) red[((w * NB + c) * MB + mb) * 64 + lane] = acc[c][mb];
    __syncthreads();
    const int n = 16 * local + 16 * w + 4 * quad;                              // register r of a lane: weight row n + r, activation row 16mb + l16
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int m = 16 * mb + l16;
        if (m >= p.M || n >= N) continue;
        f32x4 sum = red[(w * MB + mb) * 64 + lane];
#pragma unroll
        for (int u = 1; u < 4; ++u) sum += red[((u * NB + w) * MB + mb) * 64 + lane];
        if (SLICED) {
            store_slice4(p, slice, m, n, sum);
            continue;
        }
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = p.alpha * sum[e];
        if (!GROUPED && p.beta != 0.f) {
            const s16x4 c = *reinterpret_cast<const s16x4*>((const short*)p.C + (int64_t)m * p.ldc + n);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += p.beta * T::to_float(c[e]);
        }
        uint2 pk;
        pk.x = T::pack2(v[0], v[1]);
        pk.y = T::pack2(v[2], v[3]);
        *reinterpret_cast<uint2*>(Dg + (int64_t)m * ldd + n) = pk;
    }
    cb += nb;
    if (cb < blk_last) __syncthreads();                        // the sums have been read: the next chunk's copies may land there
    }
    if constexpr (SLICED) {
        __shared__ int last_s;
        finish_slices<T, 4 * 64, 64>(p, (int)blockIdx.x / p.splits, 16 * blk_first, min(16 * blk_last, p.N), &last_s);
    }
}
// The smallest NB that goes through the `most` blocks of a workgroup in as few chunks as four would (five blocks as three and two: 18944 x 3584
// at 32 rows 33.4 -> 30.5 us).
template <class T, int MB, bool SLICED, bool GROUPED>
static void launch_stripe_rows(const GemmParams& p, int most, dim3 grid, hipStream_t stream) {
    const dim3 block(4 * 64);
    if constexpr (!SLICED) {
        if (most == 1) { hipLaunchKernelGGL((gemm_stripe_kernel<T, MB, false, GROUPED, 1>), grid, block, 0, stream, p); return; }
        if (most == 2) { hipLaunchKernelGGL((gemm_stripe_kernel<T, MB, false, GROUPED, 2>), grid, block, 0, stream, p); return; }
        if ((most + 2) / 3 == (most + 3) / 4) { hipLaunchKernelGGL((gemm_stripe_kernel<T, MB, false, GROUPED, 3>), grid, block, 0, stream, p); return; }
    }
    hipLaunchKernelGGL((gemm_stripe_kernel<T, MB, SLICED, GROUPED>), grid, block, 0, stream, p);
}
// `blocks`: 16-column blocks in all (GROUPED: workgroups in all, p.grp.end counting them per weight).
template <class T, bool SLICED = false, bool GROUPED = false>
static int launch_stripe(const GemmParams& p0, int blocks, hipStream_t stream) {
    GemmParams p = p0;
    p.tiles_n = blocks;
    const dim3 grid(SLICED ? (blocks + 3) / 4 * p.splits : GROUPED ? blocks : std::min(blocks, 256));   // (GROUPED: `blocks` is the number of workgroups)
    int most = 0;   // the 16-column blocks of a workgroup
    if (GROUPED) {
        for (int s = 0, at = 0; s < kMaxGroup; at = p.grp.end[s++])
            if (p.grp.end[s] > at) most = std::max(most, ((p.grp.N[s] + 15) / 16 + p.grp.end[s] - at - 1) / (p.grp.end[s] - at));
    } else {
        most = (blocks + (int)grid.x - 1) / (int)grid.x;
    }
    if (p.M <= 16) launch_stripe_rows<T, 1, SLICED, GROUPED>(p, most, grid, stream);
    else if (p.M <= 32) launch_stripe_rows<T, 2, SLICED, GROUPED>(p, most, grid, stream);
    else if (p.M <= 48) launch_stripe_rows<T, 3, SLICED, GROUPED>(p, most, grid, stream);
    else launch_stripe_rows<T, 4, SLICED, GROUPED>(p, most, grid, stream);
    return check_launch("gemm_stripe_kernel");
}

// One row against an [N, K] weight (a decode step's projection): a wave streams whole weight rows as consecutive 16-byte
// pieces (1 KiB per instruction, where the MFMA kernel above takes 128 bytes of each of 16 rows) and multiplies in the
// vector ALU, which one activation row leaves mostly idle; one fp32 sum per lane, added up over the lanes at the end of
// a row.  A row is cut into segments of 4096 values (8 pieces per lane); when it is a single segment the lane keeps the
// activations it needs in registers (XREG), otherwise the workgroup keeps the activation row in LDS.  A wave owns a run
// of consecutive rows and has the next two segments in flight.
constexpr int kGemvSegPieces = kGemvSegHalfs / 8 / 64;     // 16-byte pieces per lane and segment
template <class T> MA_DEV float dot8(uint4 a, uint4 b, float acc);
template <> MA_DEV float dot8<F16>(uint4 a, uint4 b, float acc) {
    acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h16x2, a.x), __builtin_bit_cast(h16x2, b.x), acc, false);
    acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h16x2, a.y), __builtin_bit_cast(h16x2, b.y), acc, false);
    acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h16x2, a.z), __builtin_bit_cast(h16x2, b.z), acc, false);
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(h16x2, a.w), __builtin_bit_cast(h16x2, b.w), acc, false);
}
template <> MA_DEV float dot8<BF16>(uint4 a, uint4 b, float acc) {   // a bf16 is the upper half of the fp32 of the same value
    const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        acc = __builtin_fmaf(__builtin_bit_cast(float, aw[i] << 16), __builtin_bit_cast(float, bw[i] << 16), acc);
        acc = __builtin_fmaf(__builtin_bit_cast(float, aw[i] & 0xffff0000u), __builtin_bit_cast(float, bw[i] & 0xffff0000u), acc);
    }
    return acc;
}
// GROUPED: the rows of up to three weights numbered through (p.grp.end[s] = rows of weights 0 .. s), every weight with
// its own output; alpha = 1, no C.
// MR: activation rows (1-4; more than one only ungrouped): every weight piece is multiplied with the same piece of each.
template <class T, bool XREG, bool GROUPED, int MR = 1>
__global__ __launch_bounds__(4 * 64) void gemv_kernel(const GemmParams p, int rows_per_wave) {
    static_assert(MR == 1 || !GROUPED, "several activation rows: one weight only");
    __shared__ __attribute__((aligned(16))) short x_lds[XREG ? 8 : (MR == 1 ? kGemvMaxKHalfs : 2 * kGemvMaxKHalfs)];   // MR rows of K values: MR * K <= 32768
    const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
    const int npiece = p.K / 8, nseg = XREG ? 1 : (p.K + kGemvSegHalfs - 1) / kGemvSegHalfs;
    const int wave = (int)blockIdx.x * 4 + w;
    const int n_rows = GROUPED ? p.grp.end[kMaxGroup - 1] : p.N;
    const int r0 = min(wave * rows_per_wave, n_rows - 1), r1 = min(n_rows, wave * rows_per_wave + rows_per_wave);
    const int units = max(r1 - r0, 0) * nseg;              // (row, segment) pairs of this wave (none for a wave past the rows)
    // where row number `row` lives: its weight row and its output element (wave-uniform)
    auto locate = [&](int row, const short*& wrow, short*& out) {
        if (GROUPED) {
            const int sg = (row >= p.grp.end[0]) + (row >= p.grp.end[1]);
            const int local = row - (sg == 0 ? 0 : sg == 1 ? p.grp.end[0] : p.grp.end[1]);
            wrow = (const short*)(sg == 0 ? p.grp.B[0] : sg == 1 ? p.grp.B[1] : p.grp.B[2]) +
                   (int64_t)local * (sg == 0 ? p.grp.ldb[0] : sg == 1 ? p.grp.ldb[1] : p.grp.ldb[2]);
            out = (short*)(sg == 0 ? p.grp.D[0] : sg == 1 ? p.grp.D[1] : p.grp.D[2]) + local;
        } else {
            wrow = (const short*)p.B + (int64_t)row * p.ldb;
            out = (short*)p.D + row;
        }
    };
    struct Unit { uint4 piece[kGemvSegPieces]; };
    auto request = [&](int u, Unit& un) {
        u = max(min(u, units - 1), 0);                     // past the end: the last unit again, never used
        const int row = r0 + u / nseg, seg = u % nseg;
        const short* base; short* unused;
        locate(row, base, unused);
#pragma unroll
        for (int j = 0; j < kGemvSegPieces; ++j)
            un.piece[j] = __builtin_bit_cast(uint4, stream_load(reinterpret_cast<const u32x4*>(base + 8 * min(seg * (kGemvSegHalfs / 8) + 64 * j + lane, npiece - 1))));
    };
    Unit ring[2];
    request(0, ring[0]);
    request(1, ring[1]);
    uint4 xr[MR][kGemvSegPieces];
    if (XREG) {
#pragma unroll
        for (int m = 0; m < MR; ++m)
#pragma unroll
            for (int j = 0; j < kGemvSegPieces; ++j)
                xr[m][j] = *reinterpret_cast<const uint4*>((const short*)p.A + (int64_t)min(m, p.M - 1) * p.lda + 8 * min(64 * j + lane, npiece - 1));
    } else {
        for (int i = tid; i < MR * npiece; i += 4 * 64) {
            const int m = i / npiece, pc = i - m * npiece;
            *reinterpret_cast<uint4*>(x_lds + 8 * i) = *reinterpret_cast<const uint4*>((const short*)p.A + (int64_t)min(m, p.M - 1) * p.lda + 8 * pc);
        }
        __syncthreads();
    }
    float acc[MR];
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[m] = 0.f;
    auto consume = [&](int u, Unit& un) {
        const int row = r0 + u / nseg, seg = u % nseg;
        uint4 wv[kGemvSegPieces];
#pragma unroll
        for (int j = 0; j < kGemvSegPieces; ++j) wv[j] = un.piece[j];
        request(u + 2, un);
#pragma unroll
        for (int j = 0; j < kGemvSegPieces; ++j) {
            const int piece = seg * (kGemvSegHalfs / 8) + 64 * j + lane;
            if (piece < npiece) {
#pragma unroll
                for (int m = 0; m < MR; ++m)
                    acc[m] = dot8<T>(wv[j], XREG ? xr[m][j] : *reinterpret_cast<const uint4*>(x_lds + 8 * (m * npiece + piece)), acc[m]);
            }
        }
        if (seg == nseg - 1) {
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                float v = lane_sum<64>(acc[m]);
                acc[m] = 0.f;
                if (lane == 0 && m < p.M) {
                    const short* unused; short* out;
                    locate(row, unused, out);
                    if (!GROUPED) {
                        v *= p.alpha;
                        if (p.beta != 0.f) v += p.beta * T::to_float(((const short*)p.C)[(int64_t)m * p.ldc + row]);
                        out += (int64_t)m * p.ldd;
                    }
                    *out = (short)(T::pack2(v, 0.f) & 0xffffu);
                }
            }
        }
    };
    for (int u = 0; u < units; u += 2) {
        consume(u, ring[0]);
        if (u + 1 < units) consume(u + 1, ring[1]);
    }
}
template <class T, bool GROUPED = false>
static int launch_gemv(const GemmParams& p, int n_rows, hipStream_t stream) {
    const int max_waves = 256 * 2 * 4;   // two workgroups of four waves per compute unit
    const int rows_per_wave = (n_rows + max_waves - 1) / max_waves;
    const int waves = (n_rows + rows_per_wave - 1) / rows_per_wave;
    const dim3 grid((waves + 3) / 4), block(4 * 64);
    const bool xreg = p.K <= kGemvSegHalfs;
#define MINFER_GEMV(XR, MR) hipLaunchKernelGGL((gemv_kernel<T, XR, GROUPED, MR>), grid, block, 0, stream, p, rows_per_wave)
    if (GROUPED || p.M == 1) { if (xreg) MINFER_GEMV(true, 1); else MINFER_GEMV(false, 1); }
    else if (p.M == 2) MINFER_GEMV(false, GROUPED ? 1 : 2);   // (several rows: rows longer than a segment only, see gemv_takes)
    else if (p.M == 3) MINFER_GEMV(false, GROUPED ? 1 : 3);
    else MINFER_GEMV(false, GROUPED ? 1 : 4);
#undef MINFER_GEMV
    return check_launch("gemv_kernel");
}
// which calls it takes: one row, or up to four rows longer than a segment whose activations fit its LDS area

template <class T>
static int launch_skinny(const GemmParams& p, hipStream_t stream) {
    // two column groups per workgroup once that still leaves 160 workgroups and there is more than one block of rows
    // to share between them (32 rows x 14336 columns: 52 -> 40 us; 64 x 6144: 38 -> 27; a single block of rows loses 5-10 %)
    if (p.M > 16 && p.N >= 160 * 32) launch_skinny_nr<T, 2>(p, stream);
    else launch_skinny_nr<T, 1>(p, stream);
    return check_launch("gemm_skinny_kernel");
}

// The few-row kernel over a weight stored as rows of Q8_0 blocks, [N][K/32] blocks of 34 bytes (an fp16 scale and 32
// int8; reference block format: csrc/common/types.hpp:141-146): every weight is dequantised to fp16 exactly as
// minfer_dequant_q8_0 does (reference: cuda/quants/impls.cuh:121-143) on its way into the MFMA, so the result is that of
// the fp16 kernel on the dequantised weight while the launch streams 34 bytes per 32 weights instead of 64.
// A K step is 128 wide: lane (row n, quad q) owns block 4s + q of its weight row, which is one MFMA A fragment per
// 8 values, and the activations of the same k for the B operand (64 contiguous bytes of row m).  Blocks start on
// 2-byte boundaries; a lane reads its block as the nine aligned words that cover it, and whether the block starts on a
// word or in the middle of one depends only on q (rows are multiples of 4 bytes), so one byte permute per quant word with
// a per-lane constant selector undoes the shift (dequant8_shifted).  fp16 activations only.
// The weight loads carry no non-temporal hint, unlike the fp16 kernel's: a 128-byte line of a weight row holds 3.8
// blocks, so the line a step ends in is the line the next step starts in, and a line loaded with the hint is not kept
// for that second touch (14336 x 4096 at one row: 31 us with the hint, 17.5 us without).
template <int MB, int NR>
__global__ __launch_bounds__(kSkinnyWaves * 64) void gemm_skinny_q8_kernel(const GemmParams p) {
    using T = F16;
    __shared__ f32x4 part[kSkinnyWaves][NR][MB][64];
    const int lane = threadIdx.x & 63, w = wave_id();
    const int l16 = lane & 15, quad = lane >> 4;
    const int n0 = (int)blockIdx.x * 16 * NR;
    const int nblk = p.K / 32;                                  // blocks per weight row
    const int steps = (nblk + 3) / 4, per = (steps + kSkinnyWaves - 1) / kSkinnyWaves;
    const int s0 = w * per, s1 = min(steps, s0 + per);
    const bool odd = (quad & 1) != 0;                           // block 4s + q starts 2 bytes past a word boundary
    const uint32_t sel = odd ? kQ8SelOdd : kQ8SelEven;
    const char* wrow[NR];
#pragma unroll
    for (int nr = 0; nr < NR; ++nr) wrow[nr] = (const char*)p.B + (int64_t)min(n0 + 16 * nr + l16, p.N - 1) * p.ldb;   // ldb in bytes here
    const short* xrow[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) xrow[mb] = (const short*)p.A + (int64_t)min(16 * mb + l16, p.M - 1) * p.lda;
    f32x4 acc[NR][MB];
#pragma unroll
    for (int nr = 0; nr < NR; ++nr)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nr][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int s = s0; s < s1; ++s) {
        const int blk = 4 * s + quad;
        const bool real = blk < nblk;                           // K need not be a multiple of 128: the last step may be short
        const int bc = real ? blk : (quad & 1);               // a block of the same alignment class that exists (nblk is even)
        uint32_t wq[NR][9];
#pragma unroll
        for (int nr = 0; nr < NR; ++nr) {
            // four words per load, at addresses that are only word-aligned: the vector type says so
            typedef uint32_t u32x4_w __attribute__((ext_vector_type(4), aligned(4)));
            const uint32_t* src = reinterpret_cast<const uint32_t*>(wrow[nr] + (int64_t)bc * 34 - (odd ? 2 : 0));
            const u32x4_w a = *reinterpret_cast<const u32x4_w*>(src);
            const u32x4_w b = *reinterpret_cast<const u32x4_w*>(src + 4);
            wq[nr][0] = a[0]; wq[nr][1] = a[1]; wq[nr][2] = a[2]; wq[nr][3] = a[3];
            wq[nr][4] = b[0]; wq[nr][5] = b[1]; wq[nr][6] = b[2]; wq[nr][7] = b[3];
            wq[nr][8] = src[8];
        }
        s16x8 x[MB][4];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int j = 0; j < 4; ++j)   // a lane past the last block contributes exact zeros, whatever block 0 or 1 holds
                x[mb][j] = real ? *reinterpret_cast<const s16x8*>(xrow[mb] + 32 * bc + 8 * j) : s16x8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int nr = 0; nr < NR; ++nr) {
            const uint16_t bits = (uint16_t)(odd ? wq[nr][0] >> 16 : wq[nr][0]);
            const _Float16 dh = real ? __builtin_bit_cast(_Float16, bits) : (_Float16)0.f;
            const h16x2 d2 = {dh, dh};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const s16x8 wf = dequant8_shifted(wq[nr][2 * j], wq[nr][2 * j + 1], wq[nr][2 * j + 2], sel, d2);
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) acc[nr][mb] = T::mfma16(wf, x[mb][j], acc[nr][mb]);
            }
        }
    }
#pragma unroll
    for (int nr = 0; nr < NR; ++nr)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) part[w][nr][mb][lane] = acc[nr][mb];
    __syncthreads();
    // wave j adds up block (nr, mb) = (j / MB, j % MB): register r of a lane is n = n0 + 16*nr + 4*quad + r, m = 16*mb + l16
    if (w >= NR * MB) return;
    const int nr = w / MB, mb = w - nr * MB;
    f32x4 sum = part[0][nr][mb][lane];
#pragma unroll
    for (int ww = 1; ww < kSkinnyWaves; ++ww) sum += part[ww][nr][mb][lane];
    const int m = 16 * mb + l16, n = n0 + 16 * nr + 4 * quad;
    if (m >= p.M || n >= p.N) return;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = p.alpha * sum[e];
    if (p.beta != 0.f) {
        const s16x4 c = *reinterpret_cast<const s16x4*>((const short*)p.C + (int64_t)m * p.ldc + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += p.beta * T::to_float(c[e]);
    }
    uint2 pk;
    pk.x = T::pack2(v[0], v[1]);
    pk.y = T::pack2(v[2], v[3]);
    *reinterpret_cast<uint2*>((short*)p.D + (int64_t)m * p.ldd + n) = pk;
}

// One row against Q8_0 weights (a decode step's projections): the MFMA kernel above reads 136 bytes of each of 16 weight
// rows per instruction, which this chip's memory system serves at about half its rate.  Here a wave streams whole weight
// rows instead, as consecutive aligned 16-byte pieces (1 KiB per instruction), and does the arithmetic in the vector
// ALU, of which one activation row needs little: a weight row is cut into segments of 128 blocks (4352 bytes, a multiple
// of 16, which is why K must be a multiple of 256 and the rows 16-byte aligned); a segment's pieces go through the wave's
// LDS area, from which lane l takes blocks l and l + 64 as the nine aligned words that cover each (as
// gemm_skinny_q8_kernel does), dequantises them exactly as minfer_dequant_q8_0 does and multiplies them with the
// activations of the same positions into one fp32 sum per lane; after a row's last segment the 64 sums are added up.
// The activations a lane needs are the same for every weight row when a row is one segment (K <= 4096, XREG): it keeps
// them in registers; otherwise the workgroup keeps the activation row in LDS.  A wave owns a run of consecutive weight
// rows and always has the next two segments' pieces in flight.  (Two rows this way cost as much as the MFMA kernel, four
// half as much again: the dot products fill the vector ALU.)
constexpr int kGemvWaves = 4;
constexpr int kGemvSegBlocks = 128;                       // blocks per segment: two per lane
constexpr int kGemvSegBytes = kGemvSegBlocks * 34;        // 4352
constexpr int kGemvPieces = (kGemvSegBytes + 1023) / 1024;   // 16-byte pieces per lane and segment (5, the last one partly)
template <bool XREG>
__global__ __launch_bounds__(kGemvWaves * 64) void gemv_q8_kernel(const GemmParams p, int rows_per_wave) {
    using T = F16;
    __shared__ __attribute__((aligned(16))) char raw[kGemvWaves][kGemvSegBytes + 48];   // + the words a last block's read runs over
    __shared__ __attribute__((aligned(16))) short x_lds[XREG ? 8 : kGemvMaxK];
    const int tid = threadIdx.x, lane = tid & 63, w = wave_id();
    const int nblk = p.K / 32, nseg = XREG ? 1 : (nblk + kGemvSegBlocks - 1) / kGemvSegBlocks;
    const int wave = (int)blockIdx.x * kGemvWaves + w;
    const int r0 = min(wave * rows_per_wave, p.N - 1), r1 = min(p.N, wave * rows_per_wave + rows_per_wave);
    const int units = max(r1 - r0, 0) * nseg;              // (row, segment) pairs of this wave, row-major (none for a wave past the rows)
    const bool odd = (lane & 1) != 0;                      // blocks l and l + 64 start 2 bytes past a word boundary
    const uint32_t sel = odd ? kQ8SelOdd : kQ8SelEven;
    char* my_raw = raw[w];

    struct Unit { u32x4 piece[kGemvPieces]; };
    auto request = [&](int u, Unit& un) {
        u = max(min(u, units - 1), 0);                     // past the end: the last unit again (one cache line, never used)
        const int row = r0 + u / nseg, seg = u % nseg;
        const int pieces = min(kGemvSegBlocks, nblk - seg * kGemvSegBlocks) * 34 / 16;   // a multiple of 8 blocks: whole pieces
        const char* base = (const char*)p.B + (int64_t)row * p.ldb + (int64_t)seg * kGemvSegBytes;
#pragma unroll
        for (int j = 0; j < kGemvPieces; ++j)
            un.piece[j] = *reinterpret_cast<const u32x4*>(base + 16 * min(64 * j + lane, pieces - 1));
    };
    Unit ring[2];
    request(0, ring[0]);
    request(1, ring[1]);
    // ---- the activations, while the first weight pieces are on their way ---------------------------------
    uint4 xr[2][4];
    if (XREG) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                xr[i][j] = *reinterpret_cast<const uint4*>((const short*)p.A + 32 * min(lane + 64 * i, nblk - 1) + 8 * j);
    } else {
        for (int i = tid; i < p.K / 8; i += kGemvWaves * 64)
            *reinterpret_cast<s16x8*>(x_lds + 8 * i) = *reinterpret_cast<const s16x8*>((const short*)p.A + 8 * i);
        __syncthreads();
    }
    float acc = 0.f;
    auto consume = [&](int u, Unit& un) {
        const int row = r0 + u / nseg, seg = u % nseg;
        const int seg_blocks = min(kGemvSegBlocks, nblk - seg * kGemvSegBlocks);
        const int pieces = seg_blocks * 34 / 16;
#pragma unroll
        for (int j = 0; j < kGemvPieces; ++j)
            *reinterpret_cast<u32x4*>(my_raw + 16 * min(64 * j + lane, pieces - 1)) = un.piece[j];
        wave_lds_order();
        request(u + 2, un);                                // the registers are free again: two units ahead
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int b = lane + 64 * i;
            if (b < seg_blocks) {
                const uint32_t* wp = reinterpret_cast<const uint32_t*>(my_raw + ((34 * b) & ~3));
                uint32_t wq[9];
#pragma unroll
                for (int j = 0; j < 9; ++j) wq[j] = wp[j];
                const uint16_t bits = (uint16_t)(odd ? wq[0] >> 16 : wq[0]);
                const _Float16 dh = __builtin_bit_cast(_Float16, bits);
                const h16x2 d2 = {dh, dh};
                const short* xb = x_lds + (XREG ? 0 : 32 * (seg * kGemvSegBlocks + b));
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint4 wf = __builtin_bit_cast(uint4, dequant8_shifted(wq[2 * j], wq[2 * j + 1], wq[2 * j + 2], sel, d2));
                    const uint4 xv = XREG ? xr[i][j] : *reinterpret_cast<const uint4*>(xb + 8 * j);
                    acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h16x2, wf.x), __builtin_bit_cast(h16x2, xv.x), acc, false);
                    acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h16x2, wf.y), __builtin_bit_cast(h16x2, xv.y), acc, false);
                    acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h16x2, wf.z), __builtin_bit_cast(h16x2, xv.z), acc, false);
                    acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(h16x2, wf.w), __builtin_bit_cast(h16x2, xv.w), acc, false);
                }
            }
        }
        if (seg == nseg - 1) {                             // the row is complete: add the lanes' sums up and store
            float v = lane_sum<64>(acc);
            acc = 0.f;
            if (lane == 0) {
                v *= p.alpha;
                if (p.beta != 0.f) v += p.beta * T::to_float(((const short*)p.C)[row]);
                ((short*)p.D)[row] = (short)(T::pack2(v, 0.f) & 0xffffu);
            }
        }
    };
    for (int u = 0; u < units; u += 2) {
        consume(u, ring[0]);
        if (u + 1 < units) consume(u + 1, ring[1]);
    }
}

static int launch_gemv_q8(const GemmParams& p, hipStream_t stream) {
    // as many waves as the chip holds at a time when there are rows enough for them: two workgroups per compute unit
    const int max_waves = 256 * 2 * kGemvWaves;
    const int rows_per_wave = (p.N + max_waves - 1) / max_waves;
    const int waves = (p.N + rows_per_wave - 1) / rows_per_wave;
    const dim3 grid((waves + kGemvWaves - 1) / kGemvWaves), block(kGemvWaves * 64);
    if (p.K <= 32 * kGemvSegBlocks) hipLaunchKernelGGL((gemv_q8_kernel<true>), grid, block, 0, stream, p, rows_per_wave);
    else hipLaunchKernelGGL((gemv_q8_kernel<false>), grid, block, 0, stream, p, rows_per_wave);
    return check_launch("gemv_q8_kernel");
}

static int launch_skinny_q8(const GemmParams& p, hipStream_t stream) {
    const int mb = (p.M + 15) / 16;
    // two column groups per workgroup as soon as there is more than one row and the weight is wide enough to leave 160
    // workgroups: the activations are re-read from L2 for every group of columns, and from 8 rows on they are more bytes than
    // a group's blocks (14336 columns, 8 / 16 rows: 22.2 -> 18.4 us, 27.1 -> 20.7 us)
    const bool two = p.M > 1 && p.N >= 160 * 32;
    const dim3 grid((p.N + (two ? 32 : 16) - 1) / (two ? 32 : 16)), block(kSkinnyWaves * 64);
#define MINFER_SKINNY_Q8(MB, NR) hipLaunchKernelGGL((gemm_skinny_q8_kernel<MB, NR>), grid, block, 0, stream, p)
    if (!two) { if (mb == 1) MINFER_SKINNY_Q8(1, 1); else if (mb == 2) MINFER_SKINNY_Q8(2, 1); else if (mb == 3) MINFER_SKINNY_Q8(3, 1); else MINFER_SKINNY_Q8(4, 1); }
    else { if (mb == 1) MINFER_SKINNY_Q8(1, 2); else if (mb == 2) MINFER_SKINNY_Q8(2, 2); else if (mb == 3) MINFER_SKINNY_Q8(3, 2); else MINFER_SKINNY_Q8(4, 2); }
#undef MINFER_SKINNY_Q8
    return check_launch("gemm_skinny_q8_kernel");
}

// The stripe kernel over a weight of Q8_0 blocks ([N][K/32] blocks of 34 bytes, K a multiple of 256, rows 16-byte
// aligned): the same sharing out of 16-column blocks, chunks of four, segments of 256 values, split of a segment's k
// steps over the four waves and sum through LDS as gemm_stripe_kernel, with the weight staged as the raw blocks.  A
// segment of a row is 8 blocks = 272 bytes = 17 pieces of 16 bytes; the 64 rows of a chunk are 1088 pieces = 17 copy
// instructions of 64 lanes, lane L of instruction j taking piece 64 j + L of the chunk (row (64 j + L) / 17), so that
// a stage is the 64 row segments one after the other, 272 bytes each (a fragment's 16 rows are 68 words apart: 16
// different groups of four banks).  Every wave issues five of them per segment (j = w, w + 4, ..; the three past the
// seventeenth fetch the chunk's last piece again and land behind the stage).  A k step is one block: the lane of row
// r, k quarter q reads the three aligned words that cover values 8 q .. 8 q + 7 of block 2 w + s of its row's segment
// and dequantises them exactly as minfer_dequant_q8_0 does (dequant8_shifted; block 2 w starts on a word boundary,
// block 2 w + 1 two bytes past one), so the result is that of the fp16 kernels on the dequantised weight.
constexpr int kQ8SegBytes = 272;
template <int MB, int NB> struct Q8StripeGeom {
    static constexpr int X_BYTES = MB * 8 * kStripeBlock, CW = (17 * NB + 15) / 16, CX = 2 * MB;   // copies per wave and segment
    static constexpr int WST = 3, XST = MB + NB >= 7 ? 2 : 3;
    static constexpr int SUM_BYTES = 4 * NB * MB * 1024;   // the partial sums reuse the weight stages
    // the row segments and what the extra copies land in (with four blocks 22 KiB: in stages of 20 14336 x 4096 at 16 rows 16.5 -> 16.6 us)
    static constexpr int W_BYTES = (NB == 4 ? 22 : std::max(4 * CW, (SUM_BYTES / 1024 + WST - 1) / WST)) * 1024;
    static_assert(WST * W_BYTES >= SUM_BYTES && W_BYTES >= 4 * CW * 1024, "the partial sums, a segment");
    static_assert(WST * W_BYTES + XST * X_BYTES < 160 * 1024, "with a word to spare for finish_slices");
};
// SLICED: p.splits workgroups per chunk of four blocks, each over its share of the segments; raw fp32 sums into p.part
// ([slice][M][N]) for finish_slices (a narrow weight with a workspace, as gemm_stripe_kernel has it).
template <int MB, bool SLICED = false, int NB = 4>
__global__ __launch_bounds__(4 * 64) void gemm_stripe_q8_kernel(const GemmParams p) {
    using T = F16;
    using G = Q8StripeGeom<MB, NB>;
    constexpr int WST = G::WST, XST = G::XST, CW = G::CW, CX = G::CX;
    __shared__ __attribute__((aligned(16))) char w_lds[WST][G::W_BYTES];
    __shared__ __attribute__((aligned(16))) char x_lds[XST][G::X_BYTES];
    const int lane = threadIdx.x & 63, w = wave_id();
    const int l16 = lane & 15, quad = lane >> 4;
    int slice = 0, seg0 = 0, nseg = p.K / kStripeSeg;
    if (SLICED) {
        slice = (int)blockIdx.x % p.splits;
        seg0 = slice * nseg / p.splits;
        nseg = (slice + 1) * nseg / p.splits - seg0;
    }
    const int blk_first = SLICED ? 4 * ((int)blockIdx.x / p.splits) : (int)((int64_t)blockIdx.x * p.tiles_n / (int)gridDim.x);
    const int blk_last = SLICED ? min(blk_first + 4, p.tiles_n) : (int)((int64_t)(blockIdx.x + 1) * p.tiles_n / (int)gridDim.x);
    // x fragments as in gemm_stripe_kernel; weight fragment of (column block c, k step s): three words at
    // 272 (16 c + l16) + 68 w + 32 s + 8 quad, the block's scale two bytes further for s = 1
    const int row_off = (l16 >> 1) * kStripeBlock + 16 * (l16 & 1);
    int frag[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) frag[s] = row_off + 32 * ((4 * (2 * w + s) + quad) ^ (l16 >> 1));
    const int wfrag = kQ8SegBytes * l16 + 68 * w + 8 * quad;
    for (int cb = blk_first; cb < blk_last;) {
    const int nb = min(NB, blk_last - cb);
    const int N = min(p.N, 16 * (cb + nb));                    // rows past the chunk are not this chunk's
    const char* wsrc[CW];
#pragma unroll
    for (int i = 0; i < CW; ++i) {
        const int pc = min(64 * (w + 4 * i) + lane, 16 * NB * 17 - 1), row = pc / 17;
        wsrc[i] = (const char*)p.B + (int64_t)min(16 * cb + row, N - 1) * p.ldb + 16 * (pc - 17 * row);
    }
    const short* xsrc[CX];
#pragma unroll
    for (int j = 0; j < CX; ++j)
        xsrc[j] = (const short*)p.A + (int64_t)min(2 * (w + 4 * j) + (lane & 1), p.M - 1) * p.lda + 8 * ((lane >> 1) ^ ((w + 4 * j) & 7));
    const int rot = (int)((SLICED ? blockIdx.x : (unsigned)(cb >> 2)) % (unsigned)nseg);
    auto seg_of = [&](int t) { const int sg = t + rot; return seg0 + (sg >= nseg ? sg - nseg : sg); };
    auto issue_w = [&](int t) {
        char* st = w_lds[t % WST];
        const int off = seg_of(t) * kQ8SegBytes;
#pragma unroll
        for (int i = 0; i < CW; ++i) copy16_global_to_lds(wsrc[i] + off, st + 1024 * (w + 4 * i));
    };
    auto issue_x = [&](int t) {
        char* st = x_lds[t % XST];
        const int k0 = seg_of(t) * kStripeSeg;
#pragma unroll
        for (int j = 0; j < CX; ++j) copy16_global_to_lds(xsrc[j] + k0, st + (w + 4 * j) * kStripeBlock);
    };
    f32x4 acc[NB][MB];
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[c][mb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < WST - 1; ++t) {
        if (t < XST - 1 && t < nseg) issue_x(t);
        if (t < nseg) issue_w(t);
    }
    for (int t = 0; t < nseg; ++t) {
        __syncthreads();                                       // every wave has read segment t - 1: its stages may be refilled
        if (t + XST - 1 < nseg) issue_x(t + XST - 1);
        if (t + WST - 1 < nseg) issue_w(t + WST - 1);
        const int after = nseg - 1 - t;
        wait_behind<G>(after);
        __syncthreads();                                       // ... for every wave's copies
        const char* wb = w_lds[t % WST] + wfrag;
        const char* xb = x_lds[t % XST];
        uint32_t wq[2][NB][3], dbits[2][NB];
        s16x8 b[2][MB];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) b[s][mb] = *reinterpret_cast<const s16x8*>(xb + mb * 8 * kStripeBlock + frag[s]);
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                const uint32_t* wp = reinterpret_cast<const uint32_t*>(wb + 16 * kQ8SegBytes * c + 32 * s);
                wq[s][c][0] = wp[0]; wq[s][c][1] = wp[1]; wq[s][c][2] = wp[2];
                dbits[s][c] = *reinterpret_cast<const uint16_t*>(wb + 16 * kQ8SegBytes * c + 34 * s - 8 * quad);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                const _Float16 dh = __builtin_bit_cast(_Float16, (uint16_t)dbits[s][c]);
                const s16x8 a = dequant8_shifted(wq[s][c][0], wq[s][c][1], wq[s][c][2], s == 0 ? kQ8SelEven : kQ8SelOdd, h16x2{dh, dh});
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) acc[c][mb] = T::mfma16(a, b[s][mb], acc[c][mb]);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");     // fragments in registers before the barrier that frees the stage
    }
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(&w_lds[0][0]);
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) red[((w * NB + c) * MB + mb) * 64 + lane] = acc[c][mb];
    __syncthreads();
    const int n = 16 * cb + 16 * w + 4 * quad;               // register r of a lane: weight row n + r, activation row 16mb + l16
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int m = 16 * mb + l16;
        if (m >= p.M || n >= N) continue;
        f32x4 sum = red[(w * MB + mb) * 64 + lane];
#pragma unroll
        for (int u = 1; u < 4; ++u) sum += red[((u * NB + w) * MB + mb) * 64 + lane];
        if (SLICED) {
            store_slice4(p, slice, m, n, sum);
            continue;
        }
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = p.alpha * sum[e];
        if (p.beta != 0.f) {
            const s16x4 c = *reinterpret_cast<const s16x4*>((const short*)p.C + (int64_t)m * p.ldc + n);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += p.beta * T::to_float(c[e]);
        }
        uint2 pk;
        pk.x = T::pack2(v[0], v[1]);
        pk.y = T::pack2(v[2], v[3]);
        *reinterpret_cast<uint2*>((short*)p.D + (int64_t)m * p.ldd + n) = pk;
    }
    cb += nb;
    if (cb < blk_last) __syncthreads();
    }
    if constexpr (SLICED) {
        __shared__ int last_s;
        finish_slices<T, 4 * 64, 64>(p, (int)blockIdx.x / p.splits, 16 * blk_first, min(16 * blk_last, p.N), &last_s);
    }
}
template <int MB, bool SLICED>
static void launch_stripe_q8_rows(const GemmParams& p, int most, dim3 grid, hipStream_t stream) {   // (NB as in launch_stripe_rows)
    const dim3 block(4 * 64);
    if constexpr (!SLICED) {
        if (most == 1) { hipLaunchKernelGGL((gemm_stripe_q8_kernel<MB, false, 1>), grid, block, 0, stream, p); return; }
        if (most == 2) { hipLaunchKernelGGL((gemm_stripe_q8_kernel<MB, false, 2>), grid, block, 0, stream, p); return; }
        if ((most + 2) / 3 == (most + 3) / 4) { hipLaunchKernelGGL((gemm_stripe_q8_kernel<MB, false, 3>), grid, block, 0, stream, p); return; }
    }
    hipLaunchKernelGGL((gemm_stripe_q8_kernel<MB, SLICED>), grid, block, 0, stream, p);
}
template <bool SLICED = false>
static int launch_stripe_q8(const GemmParams& p0, hipStream_t stream) {
    GemmParams p = p0;
    p.tiles_n = (p.N + 15) / 16;
    const dim3 grid(SLICED ? (p.tiles_n + 3) / 4 * p.splits : std::min(p.tiles_n, 256));
    const int most = (p.tiles_n + (int)grid.x - 1) / (int)grid.x;
    if (p.M <= 16) launch_stripe_q8_rows<1, SLICED>(p, most, grid, stream);
    else if (p.M <= 32) launch_stripe_q8_rows<2, SLICED>(p, most, grid, stream);
    else if (p.M <= 48) launch_stripe_q8_rows<3, SLICED>(p, most, grid, stream);
    else launch_stripe_q8_rows<4, SLICED>(p, most, grid, stream);
    return check_launch("gemm_stripe_q8_kernel");
}

// Any shape and alignment: one thread per element of D, fp32 accumulation.  Small or odd problems only.
template <class T, bool NT>
__global__ __launch_bounds__(256) void gemm_plain_kernel(const GemmParams p) {
    const int64_t total = (int64_t)p.M * p.N;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int m = (int)(i / p.N), n = (int)(i % p.N);
        const short* a = (const short*)p.A + (int64_t)m * p.lda;
        const short* b = (const short*)p.B + (NT ? (int64_t)n * p.ldb : (int64_t)n);
        float s = 0.f;
        for (int k = 0; k < p.K; ++k) s += T::to_float(a[k]) * T::to_float(b[NT ? k : (int64_t)k * p.ldb]);
        float v = p.alpha * s;
        if (p.beta != 0.f) v += p.beta * T::to_float(((const short*)p.C)[(int64_t)m * p.ldc + n]);
        ((short*)p.D)[(int64_t)m * p.ldd + n] = (short)(T::pack2(v, 0.f) & 0xffffu);
    }
}

// D = alpha * (sum of the K slices' partial products) + beta * C, four columns per thread, the slices added in their order.
// Bound by latency: the sums of AT slices (eight at most) and C are requested together (one after the other, each with the memory's
// latency, 4 us beside a product of 7: 40 x 4096 x 4096 `[K, N]` with C 12.8 -> 11.7 us, 64 x 2048 x 8192 15.7 -> 13.8, 24 x 2048 x 8192
// `[N, K]` 11.9 -> 10.4, 24 x 4096 x 14336 Q8_0 20.0 -> 19.2), and a thread's place is a 32-bit division.  Many rows of few slices are bound by
// their bytes: AT divides the slices as evenly as it can, since the loads past the last one repeat it (500 x 4096 x 4096, two slices, 26.3 before; two
// loads 26.3, up to eight behind a branch each 27.2; 400 x 2048 x 8192, five slices, 25.8; five read as eight 26.1).
template <class T, int AT>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const GemmParams p) {
    const uint32_t n4 = (uint32_t)p.N >> 2, total = (uint32_t)p.M * n4;   // (64 rows of under 16 K columns, or 8 M sums of a slice, at most)
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const int m = (int)(i / n4), n = 4 * (int)(i % n4);
        const s16x4 c = load_c4(p, m, n);
        const float* src = p.part + (int64_t)m * p.N + n;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f}, x[AT];
        for (int s0 = 0; s0 < p.splits; s0 += AT) {
#pragma unroll
            for (int u = 0; u < AT; ++u) x[u] = *reinterpret_cast<const f32x4*>(src + (int64_t)min(s0 + u, p.splits - 1) * p.M * p.N);
#pragma unroll
            for (int u = 0; u < AT; ++u)
                if (s0 + u < p.splits) sum = s0 + u == 0 ? x[u] : sum + x[u];
        }
        store_result<T>(p, m, n, sum, c);
    }
}

// The counters of a sliced launch, when its workgroups are to add the slices up themselves.
static uint32_t* slice_counters(const GemmParams& p, hipStream_t stream) {
    static_assert(kMeetTiles <= kStreamCounters, "a counter per tile");
    return slices_meet(p.M) ? stream_counters(stream) : nullptr;
}

// After a sliced launch: nothing where its workgroups have added the slices up themselves.
template <class T>
static int launch_reduce(const GemmParams& p, hipStream_t stream) {
    if (p.done) return MINFER_ATTN_OK;
    const int grid = (int)std::min<int64_t>(((int64_t)p.M * (p.N / 4) + 255) / 256, 256 * 8);
    const int rounds = (p.splits + 7) / 8;
    switch ((p.splits + rounds - 1) / rounds) {
        case 2: hipLaunchKernelGGL((gemm_reduce_kernel<T, 2>), dim3(grid), dim3(256), 0, stream, p); break;
        case 3: hipLaunchKernelGGL((gemm_reduce_kernel<T, 3>), dim3(grid), dim3(256), 0, stream, p); break;
        case 4: hipLaunchKernelGGL((gemm_reduce_kernel<T, 4>), dim3(grid), dim3(256), 0, stream, p); break;
        case 5: hipLaunchKernelGGL((gemm_reduce_kernel<T, 5>), dim3(grid), dim3(256), 0, stream, p); break;
        case 6: hipLaunchKernelGGL((gemm_reduce_kernel<T, 6>), dim3(grid), dim3(256), 0, stream, p); break;
        case 7: hipLaunchKernelGGL((gemm_reduce_kernel<T, 7>), dim3(grid), dim3(256), 0, stream, p); break;
        default: hipLaunchKernelGGL((gemm_reduce_kernel<T, 8>), dim3(grid), dim3(256), 0, stream, p);
    }
    return check_launch("gemm_reduce_kernel");
}

static int launch_stripe_q8_slices(GemmParams& p, hipStream_t stream) {
    p.done = slice_counters(p, stream);
    if (int rc = launch_stripe_q8<true>(p, stream)) return rc;
    return launch_reduce<F16>(p, stream);
}

template <class T>
static int launch_stripe_slices(GemmParams& p, hipStream_t stream) {
    p.done = slice_counters(p, stream);
    if (int rc = launch_stripe<T, true>(p, (p.N + 15) / 16, stream)) return rc;
    return launch_reduce<T>(p, stream);
}

template <class T>
static int launch_kn_rows(GemmParams& p, hipStream_t stream) {
    const dim3 grid((unsigned)((p.N + 127) / 128 * p.splits)), block(4 * 64);
    p.done = p.splits > 1 ? slice_counters(p, stream) : nullptr;
    if (p.M <= 16) hipLaunchKernelGGL((gemm_kn_rows_kernel<T, 1>), grid, block, 0, stream, p);
    else if (p.M <= 32) hipLaunchKernelGGL((gemm_kn_rows_kernel<T, 2>), grid, block, 0, stream, p);
    else if (p.M <= 48) hipLaunchKernelGGL((gemm_kn_rows_kernel<T, 3>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((gemm_kn_rows_kernel<T, 4>), grid, block, 0, stream, p);
    if (int rc = check_launch("gemm_kn_rows_kernel")) return rc;
    return p.splits > 1 ? launch_reduce<T>(p, stream) : MINFER_ATTN_OK;
}


static int compute_units() {
    static std::atomic<int> cached[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
    int cus = cached[dev].load(std::memory_order_relaxed);
    if (cus == 0) {
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
        cached[dev].store(cus, std::memory_order_relaxed);
    }
    return cus;
}
template <class T> static int launch_tile(const GemmParams& p, bool nt, int tile, hipStream_t stream) {
    return std::is_same<T, F16>::value ? launch_gemm_tile_f16(p, nt, tile, stream) : launch_gemm_tile_bf16(p, nt, tile, stream);
}
template <class T>
static int launch_gemm(GemmParams& p, bool nt, int tile, hipStream_t stream) {   // (p.splits K slices)
    if (int rc = launch_tile<T>(p, nt, tile, stream)) return rc;
    return p.splits > 1 ? launch_reduce<T>(p, stream) : MINFER_ATTN_OK;
}

template <class T, bool NT>
static int launch_plain(const GemmParams& p, hipStream_t stream) {
    const int grid = (int)std::min<int64_t>(((int64_t)p.M * p.N + 255) / 256, 256 * 16);
    hipLaunchKernelGGL((gemm_plain_kernel<T, NT>), dim3(grid), dim3(256), 0, stream, p);
    return check_launch("gemm_plain_kernel");
}

template <class T>
static int launch_route(GemmParams& p, bool nt, const GemmRoute& route, hipStream_t stream) {
    p.splits = route.slices;
    switch (route.kernel) {
        case GemmKernel::gemv: return launch_gemv<T>(p, p.N, stream);
        case GemmKernel::rows_lds: return launch_rows_lds<T>(p, (p.N + 15) / 16, stream);
        case GemmKernel::skinny: return launch_skinny<T>(p, stream);
        case GemmKernel::stripe: return launch_stripe<T>(p, (p.N + 15) / 16, stream);
        case GemmKernel::stripe_slices: return launch_stripe_slices<T>(p, stream);
        case GemmKernel::kn_rows: return launch_kn_rows<T>(p, stream);
        case GemmKernel::tiles: return launch_gemm<T>(p, nt, route.tile, stream);
        case GemmKernel::plain: break;
    }
    return nt ? launch_plain<T, true>(p, stream) : launch_plain<T, false>(p, stream);
}

// Up to three weights [N_s, K] against one A in one launch (alpha = 1, no C): the tiled kernel over the concatenated
// column tiles of the weights, or, for a decode step's few rows, the few-row kernel over their column groups.
template <class T>
static int launch_grouped(GemmParams& p, int n_w, hipStream_t stream) {
    int64_t n_sum = 0;
    for (int s = 0; s < n_w; ++s) n_sum += p.grp.N[s];
    auto fill_ends = [&](int unit) {
        int acc = 0;
        for (int s = 0; s < kMaxGroup; ++s) {
            if (s < n_w) acc += (p.grp.N[s] + unit - 1) / unit;
            p.grp.end[s] = acc;
        }
        return acc;
    };
    if (p.M == 1 && p.K <= kGemvMaxKHalfs && (n_sum * p.K >= (INT64_C(1) << 25) || !rows_lds_takes(p.M, p.K))) {   // one row: whole weight rows per wave, numbered through (the rule of gemm_route)
        int acc = 0;
        for (int s = 0; s < kMaxGroup; ++s) { if (s < n_w) acc += p.grp.N[s]; p.grp.end[s] = acc; }
        return launch_gemv<T, true>(p, (int)n_sum, stream);
    }
    // a batch of decode steps: the stripe kernel over the three weights from 5 rows on (us, the 16-column and few-row kernels / it: 4096 +
    // 1024 + 1024 columns of 4096 values at 5 / 16 rows 12.6 / 10.3, 17.4 / 10.5, up to 4 rows level; 2560 + 640 + 640 of 2560 at 16 / 24 / 64
    // rows 6.7 / 6.4, 11.1 / 6.8, 15.4 / 9.3)
    {
        int64_t stripes = 0;
        for (int s = 0; s < n_w; ++s) stripes += (p.grp.N[s] + 63) / 64;
        if (p.M >= 5 && stripes <= 640 && stripe_takes(p.M, stripes, p.K)) {
            // every weight a run of workgroups in proportion to its 16-column blocks, 256 or nearly in all
            int64_t blocks = 0;
            for (int s = 0; s < n_w; ++s) blocks += (p.grp.N[s] + 15) / 16;
            const int64_t total = std::min<int64_t>(blocks, 256);
            int acc = 0;
            for (int s = 0; s < kMaxGroup; ++s) {
                if (s < n_w) {
                    const int64_t bs = (p.grp.N[s] + 15) / 16;
                    acc += (int)std::max<int64_t>(1, std::min<int64_t>(bs, total * bs / blocks));
                }
                p.grp.end[s] = acc;
            }
            return launch_stripe<T, false, true>(p, acc, stream);
        }
    }
    if (rows_lds_takes(p.M, p.K)) return launch_rows_lds<T, true>(p, fill_ends(16), stream);
    if (p.M <= 32 || (p.M <= 64 && n_sum * p.K <= (INT64_C(1) << 25))) {
        const int nr = (p.M > 16 && n_sum >= 160 * 32) ? 2 : 1;
        const int groups = fill_ends(16 * nr);
        const dim3 grid(groups), block(kSkinnyWaves * 64);
        const int mb = (p.M + 15) / 16;
#define MINFER_SKINNY(MB, NR) hipLaunchKernelGGL((gemm_skinny_kernel<T, MB, NR, true>), grid, block, 0, stream, p)
        if (nr == 1) { if (mb == 1) MINFER_SKINNY(1, 1); else if (mb == 2) MINFER_SKINNY(2, 1); else if (mb == 3) MINFER_SKINNY(3, 1); else MINFER_SKINNY(4, 1); }
        else { if (mb == 2) MINFER_SKINNY(2, 2); else if (mb == 3) MINFER_SKINNY(3, 2); else MINFER_SKINNY(4, 2); }
#undef MINFER_SKINNY
        return check_launch("gemm_skinny_kernel (grouped)");
    }
    fill_ends(1);   // the tiled kernel takes the weights' columns numbered through
    p.N = (int)n_sum;
    p.splits = 1;
    return launch_gemm<T>(p, true, tile_plan(p.M, n_sum, p.K, true, 1, compute_units()).tile, stream);
}

}  // namespace minfer_attn

using namespace minfer_attn;

MINFER_ATTN_EXPORT int minfer_qkv(int dtype, const void* x, const void* wq, const void* wk, const void* wv,
                                  void* q_out, void* k_out, void* v_out, int64_t M, int64_t K,
                                  int64_t Nq, int64_t Nk, int64_t Nv, int64_t ldx, int64_t ldwq, int64_t ldwk, int64_t ldwv,
                                  int64_t ldq, int64_t ldk, int64_t ldv, void* stream_v) {
    clear_error();
    if (dtype != MINFER_ATTN_F16 && dtype != MINFER_ATTN_BF16)
        return fail(MINFER_ATTN_EINVAL, "qkv: dtype must be MINFER_ATTN_F16 or MINFER_ATTN_BF16");
    const int64_t Ns[3] = {Nq, Nk, Nv}, ldw[3] = {ldwq, ldwk, ldwv}, ldo[3] = {ldq, ldk, ldv};
    const void* W[3] = {wq, wk, wv};
    void* O[3] = {q_out, k_out, v_out};
    if (M < 0 || K < 0 || M > 0x7fffffffLL || K > 0x7fffffffLL) return fail(MINFER_ATTN_EINVAL, "qkv: bad M or K");
    if (!x || ldx < K) return fail(MINFER_ATTN_EINVAL, "qkv: x is null or its leading dimension is smaller than K");
    bool fast = K > 0 && K % kBK == 0 && ldx % 8 == 0 && aligned16(x) && (int64_t)256 * ldx < (1LL << 30);
    for (int s = 0; s < 3; ++s) {
        if (Ns[s] < 0 || Ns[s] > 0x7fffffffLL) return fail(MINFER_ATTN_EINVAL, "qkv: bad output width");
        if (!W[s] || !O[s]) return fail(MINFER_ATTN_EINVAL, "qkv: null pointer");
        if (ldw[s] < K || ldo[s] < Ns[s]) return fail(MINFER_ATTN_EINVAL, "qkv: a leading dimension is smaller than its row");
        fast = fast && Ns[s] % 8 == 0 && ldw[s] % 8 == 0 && ldo[s] % 4 == 0 && aligned16(W[s]) && ((uintptr_t)O[s] & 7u) == 0 &&
               (int64_t)256 * ldw[s] < (1LL << 30);
    }
    if (M == 0) return MINFER_ATTN_OK;
    if (!fast || Nq == 0 || Nk == 0 || Nv == 0 || Nq + Nk + Nv > 0x7fffffffLL) {   // shapes the tiled kernels cannot take: three separate launches
        for (int s = 0; s < 3; ++s)
            if (int rc = minfer_gemm(dtype, MINFER_GEMM_B_NK, x, W[s], nullptr, O[s], M, Ns[s], K, ldx, ldw[s], Ns[s], ldo[s], 1.0, 0.0, stream_v))
                return rc;
        return MINFER_ATTN_OK;
    }
    GemmParams p{};
    p.A = x; p.M = (int)M; p.K = (int)K; p.lda = ldx; p.alpha = 1.f; p.beta = 0.f; p.C = nullptr;
    p.B = wq; p.D = q_out; p.N = (int)Nq; p.ldb = ldwq; p.ldd = ldq; p.ldc = ldq;
    for (int s = 0; s < 3; ++s) { p.grp.B[s] = W[s]; p.grp.D[s] = O[s]; p.grp.N[s] = (int)Ns[s]; p.grp.ldb[s] = ldw[s]; p.grp.ldd[s] = ldo[s]; }
    hipStream_t stream = (hipStream_t)stream_v;
    return dtype == MINFER_ATTN_F16 ? launch_grouped<F16>(p, 3, stream) : launch_grouped<BF16>(p, 3, stream);
}

static int gemm_impl(int dtype, int b_layout, const void* A, const void* B, const void* C, void* D,
                     int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int64_t ldd,
                     double alpha, double beta, void* workspace, size_t workspace_bytes, void* stream_v) {
    clear_error();
    if (dtype != MINFER_ATTN_F16 && dtype != MINFER_ATTN_BF16)
        return fail(MINFER_ATTN_EINVAL, "gemm: dtype must be MINFER_ATTN_F16 or MINFER_ATTN_BF16");
    if (b_layout != MINFER_GEMM_B_KN && b_layout != MINFER_GEMM_B_NK)
        return fail(MINFER_ATTN_EINVAL, "gemm: b_layout must be MINFER_GEMM_B_KN or MINFER_GEMM_B_NK");
    if (M < 0 || N < 0 || K < 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL)
        return fail(MINFER_ATTN_EINVAL, "gemm: bad M, N or K");
    if (!A || !B || !D || (beta != 0.0 && !C)) return fail(MINFER_ATTN_EINVAL, "gemm: null pointer");
    const bool nt = b_layout == MINFER_GEMM_B_NK;
    if (lda < K || ldd < N || (beta != 0.0 && ldc < N) || ldb < (nt ? K : N))
        return fail(MINFER_ATTN_EINVAL, "gemm: a leading dimension is smaller than its row");
    if (M == 0 || N == 0) return MINFER_ATTN_OK;
    GemmParams p{};
    p.A = A; p.B = B; p.C = C; p.D = D; p.M = (int)M; p.N = (int)N; p.K = (int)K;
    p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.ldd = ldd; p.alpha = (float)alpha; p.beta = (float)beta;
    // the tiled kernel moves 16-byte pieces and whole 64-wide K steps, and addresses a panel with 32-bit offsets
    const bool fast = K > 0 && K % kBK == 0 && N % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && ldc % 4 == 0 && ldd % 4 == 0 &&
                      aligned16(A) && aligned16(B) && ((uintptr_t)D & 7u) == 0 && ((uintptr_t)C & 7u) == 0 &&
                      (int64_t)256 * lda < (1LL << 30) && (int64_t)256 * ldb < (1LL << 30);
    hipStream_t stream = (hipStream_t)stream_v;
    const size_t fit = workspace && aligned16(workspace) ? workspace_bytes / ((size_t)M * (size_t)N * sizeof(float)) : 0;   // slices the workspace holds
    p.part = (float*)workspace;
    const GemmRoute route = gemm_route(M, N, K, nt, fast, (int64_t)std::min<size_t>(fit, 2 * kMostSlices), compute_units);
    return dtype == MINFER_ATTN_F16 ? launch_route<F16>(p, nt, route, stream) : launch_route<BF16>(p, nt, route, stream);
}

MINFER_ATTN_EXPORT int minfer_gemm(int dtype, int b_layout, const void* A, const void* B, const void* C, void* D,
                                   int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int64_t ldd,
                                   double alpha, double beta, void* stream_v) {
    return gemm_impl(dtype, b_layout, A, B, C, D, M, N, K, lda, ldb, ldc, ldd, alpha, beta, nullptr, 0, stream_v);
}

MINFER_ATTN_EXPORT size_t minfer_gemm_layout_workspace_bytes(int b_layout, int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL) return 0;
    // what gemm_route cuts K into for this layout when it has all the room it wants (sizes the tiled kernels take; others use none)
    const bool fast = K % kBK == 0 && N % 8 == 0;
    const int splits = gemm_route(M, N, K, b_layout != MINFER_GEMM_B_KN, fast, 2 * kMostSlices, compute_units).slices;
    return splits > 1 ? (size_t)splits * (size_t)M * (size_t)N * sizeof(float) : 0;
}

MINFER_ATTN_EXPORT size_t minfer_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL) return 0;
    const int cus = compute_units();
    const int splits = std::max(std::max(gemm_slices(M, N, K, true, cus), gemm_slices(M, N, K, false, cus)), std::max(stripe_slices(M, N, K), kn_slices(M, N, K)));
    return splits > 1 ? (size_t)splits * (size_t)M * (size_t)N * sizeof(float) : 0;
}

MINFER_ATTN_EXPORT int minfer_gemm_ws(int dtype, int b_layout, const void* A, const void* B, const void* C, void* D,
                                      int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int64_t ldd,
                                      double alpha, double beta, void* workspace, size_t workspace_bytes, void* stream_v) {
    return gemm_impl(dtype, b_layout, A, B, C, D, M, N, K, lda, ldb, ldc, ldd, alpha, beta, workspace, workspace_bytes, stream_v);
}

// ---- weights stored as Q8_0 blocks ------------------------------------------------------------------------------
static size_t q8_dequant_bytes(int64_t N, int64_t K) { return ((size_t)N * (size_t)K * 2 + 255) & ~(size_t)255; }

// What the kernels that stream the blocks (q8_streams) need besides: 16-byte pieces of A, aligned 8-byte pieces of C (only when beta != 0)
// and D.
static bool q8_stream_operands(const void* A, const void* C, const void* D, int64_t lda, int64_t ldc, int64_t ldd, double beta) {
    return aligned16(A) && lda % 8 == 0 && ldd % 4 == 0 && ((uintptr_t)D & 7u) == 0 &&
           (beta == 0.0 || (ldc % 4 == 0 && ((uintptr_t)C & 7u) == 0));
}

MINFER_ATTN_EXPORT size_t minfer_gemm_q8_0_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 32 != 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL) return 0;
    if (q8_streams(M, N, K)) {   // optional: K slices of the stripe kernel for a narrow weight
        const int slices = q8_slices(M, N, K);
        return slices > 1 ? (size_t)slices * (size_t)M * (size_t)N * sizeof(float) : 0;
    }
    const int slices = std::max(stripe_slices(M, N, K), M > 16 ? gemm_slices(M, N, K, true, compute_units()) : 1);   // (the size has been that)
    return q8_dequant_bytes(N, K) + (slices > 1 ? (size_t)slices * (size_t)M * (size_t)N * sizeof(float) : 0);
}

MINFER_ATTN_EXPORT int minfer_gemm_q8_0(const void* A, const void* Bq, const void* C, void* D, int64_t M, int64_t N, int64_t K,
                                        int64_t lda, int64_t ldc, int64_t ldd, double alpha, double beta,
                                        void* workspace, size_t workspace_bytes, void* stream_v) {
    clear_error();
    if (M < 0 || N < 0 || K < 0 || M > 0x7fffffffLL || N > 0x7fffffffLL || K > 0x7fffffffLL)
        return fail(MINFER_ATTN_EINVAL, "gemm_q8_0: bad M, N or K");
    if (K % 32 != 0) return fail(MINFER_ATTN_EINVAL, "gemm_q8_0: K must be a multiple of the block size 32");
    if (!A || !Bq || !D || (beta != 0.0 && !C)) return fail(MINFER_ATTN_EINVAL, "gemm_q8_0: null pointer");
    if (lda < K || ldd < N || (beta != 0.0 && ldc < N)) return fail(MINFER_ATTN_EINVAL, "gemm_q8_0: a leading dimension is smaller than its row");
    if (M == 0 || N == 0) return MINFER_ATTN_OK;
    if (K == 0) return fail(MINFER_ATTN_EINVAL, "gemm_q8_0: K must be positive");
    hipStream_t stream = (hipStream_t)stream_v;
    const int64_t row_bytes = K / 32 * 34;
    if (((uintptr_t)Bq & 3u) != 0) return fail(MINFER_ATTN_EINVAL, "gemm_q8_0: the weight must be 4-byte aligned");
    if (q8_streams(M, N, K) && q8_stream_operands(A, C, D, lda, ldc, ldd, beta)) {
        GemmParams p{};
        p.A = A; p.B = Bq; p.C = beta != 0.0 ? C : nullptr; p.D = D; p.M = (int)M; p.N = (int)N; p.K = (int)K;
        p.lda = lda; p.ldb = row_bytes; p.ldc = ldc; p.ldd = ldd; p.alpha = (float)alpha; p.beta = (float)beta;
        const size_t fit = workspace && aligned16(workspace) ? workspace_bytes / ((size_t)M * (size_t)N * sizeof(float)) : 0;
        const Q8Route route = q8_route(M, N, K, aligned16(Bq), (int64_t)std::min<size_t>(fit, kMostSlices));
        p.splits = route.slices; p.part = (float*)workspace;
        switch (route.kernel) {
            case Q8Kernel::gemv: return launch_gemv_q8(p, stream);
            case Q8Kernel::stripe_slices: return launch_stripe_q8_slices(p, stream);
            case Q8Kernel::stripe: return launch_stripe_q8(p, stream);
            case Q8Kernel::skinny: return launch_skinny_q8(p, stream);
        }
    }
    // otherwise: the weight as fp16 in the workspace, then the fp16 kernels on it, or the call in parts (q8_part_rows)
    const size_t deq = q8_dequant_bytes(N, K);
    if (!workspace || !aligned16(workspace) || workspace_bytes < deq)
        return fail(MINFER_ATTN_EWORKSPACE, "gemm_q8_0: this call needs a workspace of N*K*2 bytes (rounded up to 256) for the dequantised weight "
                                            "(more than 64 rows, an odd number of blocks per row, N not a multiple of 4, or A/C/D not aligned for the streaming kernel: "
                                            "A 16 bytes with lda a multiple of 8, C and D 8 bytes with strides multiples of 4)");
    if (const int64_t rows = q8_part_rows(M, N, K, aligned16(Bq)); rows < M && q8_stream_operands(A, C, D, lda, ldc, ldd, beta)) {
        for (int64_t m = 0; m < M; m += rows)
            if (int rc = minfer_gemm_q8_0((const short*)A + m * lda, Bq, C ? (const short*)C + m * ldc : nullptr, (short*)D + m * ldd, std::min(rows, M - m), N, K,
                                          lda, ldc, ldd, alpha, beta, workspace, workspace_bytes, stream_v)) return rc;
        return MINFER_ATTN_OK;
    }
    if (int rc = minfer_dequant_q8_0(MINFER_ATTN_F16, Bq, workspace, N, K, stream_v)) return rc;
    return gemm_impl(MINFER_ATTN_F16, MINFER_GEMM_B_NK, A, workspace, C, D, M, N, K, lda, K, ldc, ldd, alpha, beta,
                     (char*)workspace + deq, workspace_bytes - deq, stream_v);
}
