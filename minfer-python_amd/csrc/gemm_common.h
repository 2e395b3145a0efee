// What the kernels of the GEMM family share: the parameters of a launch, the swizzles of the staged panels, the last step of a
// result.
#pragma once

#include <type_traits>
#include <utility>

#include "attn_common.h"
#include "attn_host.h"
#include "gemm_plan.h"

namespace minfer_attn {

constexpr int kRowTile = 8192;              // sub-tile [64 rows][64 k], 128-byte rows (A, and B as [N, K])
constexpr int kColTile = 16384;             // sub-tile [64 k][128 n], 256-byte rows (B as [K, N])

// [N, K] weights that share A in one launch (the QKV projection): the column units of weight s follow those of weight s - 1, and `end`
// holds the cumulative counts: columns for the tiled kernel, whose tiles may hold columns of two weights, and gemv_kernel, column groups or
// workgroups for the other few-row kernels.  More than one weight: no C operand.
constexpr int kMaxGroup = 3;
struct GemmGroup {
    const void* B[kMaxGroup]; void* D[kMaxGroup];
    int N[kMaxGroup], end[kMaxGroup];
    int64_t ldb[kMaxGroup], ldd[kMaxGroup];
};
struct GemmParams {
    const void* A; const void* B; const void* C; void* D;
    int M, N, K;
    int64_t lda, ldb, ldc, ldd;   // row strides in elements
    float alpha, beta;
    int tiles_m, tiles_n, per_xcd;
    int splits;                   // SPLIT instantiations: K is cut into this many slices, one workgroup per (tile, slice)
    float* part;                  // their fp32 partial products, [splits][M][N]
    uint32_t* done;               // zeroed arrival counters, one per tile (stripe), left zero; null: gemm_reduce_kernel adds the slices up
    GemmGroup grp;                // used by the GROUPED instantiations, and by every [N, K] launch of the tiled kernel (one weight: a group of one)
};
// Which weight column unit `c` (a tile column or a column group) belongs to, and its index inside that weight.
MA_DEV int group_of_unit(const GemmGroup& g, int c, int& local) {
    const int s = c < g.end[0] ? 0 : (c < g.end[1] ? 1 : 2);
    local = c - (s == 0 ? 0 : (s == 1 ? g.end[0] : g.end[1]));
    return s;
}

// Four consecutive columns of C, which are requested together with the sums that they are added to; not read where beta is 0.
MA_DEV s16x4 load_c4(const GemmParams& p, int m, int n) {
    s16x4 c = {0, 0, 0, 0};
    if (p.beta != 0.f) c = *reinterpret_cast<const s16x4*>((const short*)p.C + (int64_t)m * p.ldc + n);
    return c;
}
// Four consecutive columns of D from the sums in fp32 and those of C: alpha, beta and C, one rounding.
template <class T> MA_DEV void store_result(const GemmParams& p, int m, int n, f32x4 sum, s16x4 c) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = p.alpha * sum[e];
    if (p.beta != 0.f) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += p.beta * T::to_float(c[e]);
    }
    uint2 pk;
    pk.x = T::pack2(v[0], v[1]);
    pk.y = T::pack2(v[2], v[3]);
    *reinterpret_cast<uint2*>((short*)p.D + (int64_t)m * p.ldd + n) = pk;
}
template <class T> MA_DEV void store_result(const GemmParams& p, int m, int n, f32x4 sum) { store_result<T>(p, m, n, sum, load_c4(p, m, n)); }

// swizzles: granule index of a row XORed with a function of the row (see the attention kernel's TileGeom)
MA_DEV int swz_row_tile(int row) { return (row >> 1) & 7; }        // 128-byte rows, read 32 rows x 16 bytes
MA_DEV int swz_col_tile(int row) { return ((row & 3) << 2) | ((row >> 2) & 2); }   // 256-byte rows, transposing reads of 4 rows x 32 bytes by each of two 16-lane groups 8 rows apart

int launch_gemm_tile_f16(const GemmParams& p, bool nt, int tile, hipStream_t stream);
int launch_gemm_tile_bf16(const GemmParams& p, bool nt, int tile, hipStream_t stream);

}  // namespace minfer_attn
