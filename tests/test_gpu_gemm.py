"""GPU parity tests (-m gpu) of the GEMM kernels and of the gemm / qkv operators, through the C ABI and the
registered torch ops, against the fp64 CPU oracle on identical seeded inputs.

Tolerance: the reference's tests allow atol 6e-1 (gemm) and 2e-1 (qkv) (reference: test/kernels.py:145,
212-214).  Here every element must lie within 0.51 units in the last place of the output format of the
oracle's exact value, plus 2^-17 of the largest magnitude of the result for the fp32 accumulation (which
shows only where a sum of a few hundred terms cancels to something far smaller than its terms)."""
import os

import numpy as np
import pytest
import torch

import capi
import gemm_plan_probe as rules
import oracle
import workloads

pytestmark = pytest.mark.gpu
DEV = "cuda"
MANT = {torch.float16: 10, torch.bfloat16: 7}
MIN_EXP = {torch.float16: -14, torch.bfloat16: -126}
KN, NK = capi.GEMM_B_KN, capi.GEMM_B_NK


def assert_close(got, exact, dtype, what=""):
    got = got.float().cpu().numpy().astype(np.float64)
    exact = exact.astype(np.float64)
    e = np.floor(np.log2(np.maximum(np.abs(exact), 2.0 ** MIN_EXP[dtype])))
    bound = 0.51 * 2.0 ** (e - MANT[dtype]) + 2.0 ** -17 * float(np.abs(exact).max())
    err = np.abs(got - exact)
    worst = np.unravel_index(np.argmax(err - bound), err.shape)
    assert not (err > bound).any(), (f"{what}: {(err > bound).sum()} elements out of bound; at {worst} got {got[worst]!r}, "
                                     f"exact {float(exact[worst])!r}")


def make(M, N, K, layout, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, K, generator=g).to(dtype)
    b = ((1 / K ** 0.5) * torch.randn((K, N) if layout == KN else (N, K), generator=g)).to(dtype)
    c = torch.randn(M, N, generator=g).to(dtype)
    return a, b, c


@pytest.mark.parametrize("layout", [KN, NK])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,alpha,beta", [
    (256, 256, 64, 1.0, 0.0),        # four tiles of the 128 x 128 kernel, one K step
    (512, 384, 256, 2.0, 3.0),
    (300, 264, 192, 0.5, 2.0),       # ragged rows and columns (N a multiple of 8 only)
    (100, 72, 64, 1.0, 1.0),
    (1, 128, 128, 1.0, 0.0),         # a single row (decode-time projection)
    (4096, 4096, 128, 1.0, 1.0),     # enough tiles for the 256 x 256 kernel
    (3000, 4104, 64, 2.0, 0.0),      # the same with ragged edges
    (33, 17, 50, 1.0, 1.0),          # nothing tileable: plain kernel
    (64, 64, 72, 1.0, 0.0),          # K not a multiple of 64: plain kernel
    (8, 4096, 4096, 1.0, 0.0),       # a decode step's tokens: kernels that stream the weight once
    (64, 1024, 1792, 2.0, 3.0),      # their largest row count; K steps not a multiple of the eight waves
    (48, 8192, 8192, 1.0, 0.0),      # more than 32 rows against a large weight
    (2048, 6144, 128, 1.0, 1.0),     # 256 x 256, three quarters of a round
    (1800, 6144, 64, 2.0, 3.0),      # the same with a ragged last tile row, one K step
    (30, 5200, 128, 2.0, 1.0),       # wide enough for two column groups per workgroup, the last one ragged
    (37, 24, 192, 0.5, 1.0),         # ragged rows, a last group of 16 columns that is half empty
    (17, 4104, 64, 1.0, 1.0),        # one K step: seven of the eight waves have nothing to add
    (64, 6144, 4096, 2.0, 3.0),      # 64 rows, 96 stripes
    (40, 5128, 1024, 1.0, 1.0),      # 40 rows (three row blocks), 81 stripes, the last one of 8 columns
    (64, 5152, 192, 2.0, 3.0),       # K no multiple of 256, two column groups per workgroup: the few-row kernel's largest instantiation
    (40, 5128, 448, 1.0, 1.0),       # ... with three row blocks, the last group ragged
    # up to 16 rows against an [N, K] weight with K a multiple of 512: weight and activation rows copied to LDS along the rows
    (2, 4096, 4096, 1.0, 0.0),
    (5, 264, 512, 1.0, 1.0),         # one segment per wave; rows 5..7 of the second activation copy do not exist
    (12, 1000, 1536, 2.0, 3.0),      # three activation copies, a last group of 8 columns
    (16, 4104, 1024, 1.0, 1.0),
    (3, 8, 512, 1.0, 0.0),           # a single half-empty group
    (9, 2048, 14336, 0.5, 0.0),      # 28 segments per wave
    # 1-64 rows, K a multiple of 256: 16-column blocks over the whole of K
    (2, 12288, 256, 1.0, 0.0),       # one segment
    (1, 12296, 1024, 2.0, 3.0),      # one row
    (1, 6144, 4096, 1.0, 0.0),       # 96 stripes: the narrowest weight it takes at any row count
    (8, 5120, 768, 2.0, 3.0),        # 80 stripes
    (40, 4104, 1024, 1.0, 1.0),      # 65 stripes, the last one of 8 columns
    (9, 12296, 512, 2.0, 3.0),       # a last stripe of 8 columns; two segments (fewer than the three stages)
    (16, 14336, 1024, 1.0, 1.0),
    (17, 12288, 768, 1.0, 0.0),      # two blocks of activation rows, the second with one row
    (32, 12352, 1280, 0.5, 1.0),
    (33, 12288, 512, 1.0, 1.0),      # four blocks of activation rows, two stages
    (64, 14336, 1792, 2.0, 0.0),
    # one row against an [N, K] weight: whole weight rows per wave (segments of 4096 values)
    (1, 4096, 4096, 1.0, 0.0),       # a small weight and K a multiple of 512: the LDS-staged few-row kernel
    (1, 8200, 4096, 2.0, 3.0),       # one segment, the activations in registers; three rows per wave, a last wave with fewer
    (1, 1000, 4160, 2.0, 3.0),       # a second segment of 64 values, the activations in LDS
    (1, 1000, 8192, 2.0, 3.0),       # longer than a segment and a multiple of 512: the LDS-staged few-row kernel as well
    (1, 20000, 64, 2.0, 3.0),        # ten short rows per wave
    (1, 264, 16384, 1.0, 1.0),       # the longest activation row its LDS area holds
    (1, 264, 16448, 1.0, 0.0),       # longer: the 16-rows-per-instruction kernel
    (1, 8, 192, 1.0, 1.0),           # two waves with rows, the others none
    # two to four rows against long rows of a wide weight: whole weight rows per wave, every piece times the same piece of each activation row
    (2, 10240, 8192, 1.0, 0.0),
    (3, 10248, 8192, 2.0, 3.0),      # a last wave with fewer rows
    (4, 16384, 8192, 1.0, 1.0),
])
def test_gemm_matches_oracle(layout, dtype, M, N, K, alpha, beta):
    a, b, c = make(M, N, K, layout, dtype, M + N + K)
    if M * N * K <= 1 << 26 or M <= 64:
        exact = oracle.gemm(a, b, c, alpha, beta, layout)
        rows = slice(None)
    else:       # the oracle is a scalar CPU program: a sample of rows at this size
        rows = torch.tensor(sorted({0, 1, 255, 256, 257, M // 2, M - 257, M - 2, M - 1} | set(range(1000, 1064))))
        exact = oracle.gemm(a[rows], b, c[rows], alpha, beta, layout)
    d = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
    assert capi.gemm(a.to(DEV), b.to(DEV), c.to(DEV), d, alpha, beta, layout) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert_close(d[rows], exact, dtype, "gemm")
    if not isinstance(rows, slice):   # the whole result against an fp32 torch evaluation of the same expression
        ref = alpha * (a.to(DEV).float() @ (b.to(DEV).float() if layout == KN else b.to(DEV).float().T)) + beta * c.to(DEV).float()
        assert float((d.float() - ref).abs().max()) <= 2.0 ** -MANT[dtype] * float(ref.abs().max())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout,M,N,K,alpha,beta", [
    (NK, 593, 14344, 64, 1.0, 0.0),      # 160 x 256: one K step of the three stages, a ragged last tile row and column
    (NK, 470, 16392, 256, 2.0, 3.0),     # 160 x 224: four steps
    (NK, 900, 8200, 320, 1.0, 1.0),      # five steps
    (NK, 1003, 8200, 192, 2.0, 3.0),     # 160 x 256: a last tile of 8 columns
    (NK, 385, 8200, 128, 1.0, 1.0),      # 224 x 128: two steps
    (NK, 130, 16392, 448, 2.0, 3.0),     # 160 x 128
    (KN, 385, 8200, 192, 1.0, 0.0),
    (KN, 257, 12296, 64, 2.0, 3.0),
    (KN, 520, 14344, 64, 1.0, 1.0),      # 160 x 256
    (KN, 385, 16392, 320, 2.0, 3.0),     # an odd number of steps
    (NK, 1545, 4904, 192, 2.0, 3.0),     # 160 x 224
    (KN, 1545, 4904, 192, 2.0, 3.0),     # 128 x 128, two workgroups to a unit
])
def test_gemm_tiles_between_the_small_and_the_large_one(layout, dtype, M, N, K, alpha, beta):
    """Every element against torch's product in 64 bits, within the bound of assert_close."""
    a, b, c = make(M, N, K, layout, dtype, M + N + K)
    d = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
    assert capi.gemm(a.to(DEV), b.to(DEV), c.to(DEV), d, alpha, beta, layout) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert_close(d, (alpha * (a.double() @ (b if layout == KN else b.T).double()) + beta * c.double()).numpy(), dtype)


@pytest.mark.parametrize("layout,M,N,K,tile", [   # tile: rows, columns, workgroups to a unit
    (KN, 977, 4152, 64, (128, 128, 2)),
    (NK, 1173, 3384, 64, (128, 128, 2)),
    (KN, 71, 424, 192, (128, 128, 1)),
    (NK, 67, 360, 256, (128, 128, 1)),
    (NK, 1147, 3640, 320, (128, 192, 1)),
    (KN, 899, 6536, 448, (128, 256, 1)),
    (NK, 905, 6568, 640, (128, 256, 1)),
    (KN, 137, 1944, 64, (160, 128, 1)),
    (NK, 137, 3816, 128, (160, 128, 1)),
    (NK, 897, 6632, 192, (160, 224, 1)),
    (KN, 1059, 7192, 256, (160, 256, 1)),
    (NK, 1349, 6296, 320, (160, 256, 1)),
    (KN, 651, 6584, 448, (192, 128, 1)),
    (NK, 647, 6568, 640, (192, 128, 1)),
    (NK, 903, 3592, 64, (192, 192, 1)),
    (KN, 1287, 7176, 128, (192, 256, 1)),
    (NK, 1811, 5416, 192, (192, 256, 1)),
    (KN, 645, 6200, 256, (224, 128, 1)),
    (NK, 657, 6632, 320, (224, 128, 1)),
    (NK, 1773, 4904, 448, (224, 192, 1)),
    (KN, 1561, 6440, 640, (224, 256, 1)),
    (NK, 2119, 4824, 64, (224, 256, 1)),
    (NK, 1949, 5656, 320, (256, 192, 1)),
    (NK, 2025, 4888, 128, (256, 224, 1)),
    (KN, 2027, 5976, 192, (256, 256, 1)),
    (NK, 1807, 7192, 256, (256, 256, 1)),
])
def test_gemm_every_tile_shape(gemm_plan, layout, M, N, K, tile):
    """A shape for which plan_tiles takes each tile (without a workspace, on 256 compute units), the last tile row and column
    ragged, from one K step (fewer than the ring has stages) to ten: every element against torch's product in 64 bits, within the
    bound of assert_close."""
    assert gemm_plan(M, N, K, layout == NK, 0) == (rules.TILES, 1, *tile)
    dtype = torch.float16 if (M + K // 64) % 2 else torch.bfloat16
    alpha, beta = (2.0, 3.0) if K % 128 else (1.0, 0.0)
    a, b, c = make(M, N, K, layout, dtype, M + N + K)
    d = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
    assert capi.gemm(a.to(DEV), b.to(DEV), c.to(DEV), d, alpha, beta, layout) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert_close(d, (alpha * (a.double() @ (b if layout == KN else b.T).double()) + beta * c.double()).numpy(), dtype)


@pytest.mark.parametrize("layout,M,N,K", [   # tiles of 4 to 8 block rows a wave, 4 to 8 blocks across, the last ones not full
    (NK, 65, 136, 64), (KN, 129, 264, 128), (NK, 300, 1000, 192), (NK, 258, 5424, 384), (KN, 487, 8584, 128),
    (NK, 1949, 5656, 320), (NK, 2025, 4888, 128), (KN, 2027, 5976, 192),
])
def test_gemm_adds_c_in_place(layout, M, N, K):
    """The residual added in place, in rows of a wider buffer: C's pieces are requested block rows before the same places are
    stored, bit-equal to the call with C apart, nothing else written."""
    a, b, c = (x.to(DEV) for x in make(M, N, K, layout, torch.float16, M + N + K))
    d = torch.full_like(c, float("nan"))
    assert capi.gemm(a, b, c, d, 2.0, 3.0, layout) == capi.OK, capi.last_error()
    wide = torch.full((M + 3, N + 24), float("nan"), dtype=c.dtype, device=DEV)
    view = wide[1:M + 1, 8:N + 8]
    view.copy_(c)
    assert capi.gemm(a, b, view, view, 2.0, 3.0, layout) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert_close(d, (2.0 * torch.mm(a.double(), (b if layout == KN else b.T.contiguous()).double()) + 3.0 * c.double()).cpu().numpy(), torch.float16)
    assert torch.equal(view, d)
    view.fill_(float("nan"))
    assert torch.isnan(wide).all()


@pytest.mark.parametrize("M", [9, 24, 40, 64])
@pytest.mark.parametrize("N,K", [
    (2056, 256),      # one 16-column block a workgroup, the last of 8 columns; one segment
    (4096, 512),
    (2048, 2560),     # more segments than the ring has stages
    (4104, 1280),     # two blocks
    (8184, 768),
    (8200, 1024),     # three
    (18440, 512),     # five: three and two
    (28680, 1024),    # eight at most: four by four
])
def test_gemm_stripe_blocks(M, N, K):
    """Every number of 16-column blocks that the stripe kernel takes at a time, from fewer segments of K than stages to more, every number
    of activation row blocks: all elements against torch's product in 64 bits, within the bound of assert_close."""
    dtype = torch.float16 if (M + K // 256) % 2 else torch.bfloat16
    a, b, c = make(M, N, K, NK, dtype, M + N + K)
    alpha, beta = (2.0, 3.0) if M % 16 else (1.0, 0.0)
    d = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
    assert capi.gemm(a.to(DEV), b.to(DEV), c.to(DEV), d, alpha, beta, NK) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert_close(d, (alpha * (a.double() @ b.T.double()) + beta * c.double()).numpy(), dtype)


@pytest.mark.parametrize("M,N,K", [
    (16, 2056, 256),      # one block a workgroup, the last of 8 columns; one segment
    (33, 4096, 2048),
    (64, 2048, 2560),
    (17, 4104, 1280),     # two
    (9, 8184, 768),
    (32, 6144, 4096),
    (2, 10248, 512),      # three
    (40, 18440, 768),     # five: three and two
    (64, 12280, 1024),
])
def test_gemm_q8_0_stripe_blocks(M, N, K):
    """The same over Q8_0 blocks, with and without a workspace, of each number of column blocks at a time: every element against torch's product
    with the dequantised weight in 64 bits, within the bound of assert_close."""
    a, wq, c, w = make_q8(M, N, K, seed=M + N + K)
    want = (2.0 * (a.double() @ w.double().T) + c.double()).numpy()
    ws = torch.empty(capi.lib().minfer_gemm_q8_0_workspace_bytes(M, N, K), dtype=torch.uint8, device=DEV)
    for space in (None, ws if ws.numel() else None):
        d = torch.full((M, N), float("nan"), dtype=torch.float16, device=DEV)
        assert capi.gemm_q8_0(a.to(DEV), wq.to(DEV), c.to(DEV), d, 2.0, 1.0, space) == capi.OK, capi.last_error()
        torch.cuda.synchronize()
        assert_close(d, want, torch.float16)


def test_gemm_golden_strided_and_in_place():
    z = np.load(os.path.join(os.path.dirname(__file__), "golden", "gemm_small.npz"))
    a, b, c = (torch.from_numpy(z[k]).to(DEV) for k in "abc")
    alpha, beta = float(z["alpha"]), float(z["beta"])
    d = torch.empty_like(c)
    assert capi.gemm(a, b, c, d, alpha, beta) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert_close(d, z["d"], torch.float16, "golden")
    # C aliasing D
    d2 = c.clone()
    assert capi.gemm(a, b, d2, d2, alpha, beta) == capi.OK
    torch.cuda.synchronize()
    assert torch.equal(d2, d)
    # row strides larger than the rows (views of wider buffers), beta = 0 with no C
    big_a = torch.randn(70, 200, device=DEV).half()
    big_d = torch.full((70, 96), float("nan"), dtype=torch.float16, device=DEV)
    av, dv = big_a[:, 8:136], big_d[:, 16:88]
    assert capi.gemm(av, b, None, dv, 1.0, 0.0) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert_close(dv, oracle.gemm(av.cpu().contiguous(), b.cpu(), None, 1.0, 0.0), torch.float16, "strided")
    assert torch.isnan(big_d[:, :16]).all() and torch.isnan(big_d[:, 88:]).all()


@pytest.mark.parametrize("S", [1024, 2048])
@pytest.mark.parametrize("alpha,beta", [(1.0, 0.0), (2.0, 3.0)])
def test_gemm_op_reference_test_recipe(kerns, S, alpha, beta):
    """The reference's test recipe (test/kernels.py:119-147): A [1,S,S] ~ N(0,1), weight [S,S] ~ N(0,1)/sqrt(S), bias
    ~ N(0,1), through the op with the reference's signature; sampled rows against the oracle, everything against
    the reference's own expression at its own tolerance."""
    a, w, bias = workloads.gemm_input(S, S, S, seed=S, device=DEV)
    out = torch.zeros_like(bias)
    assert kerns.gemm(1, 1, 2, alpha, beta, a, w, bias, out) is None
    torch.cuda.synchronize()
    rows = torch.arange(0, S, S // 16)
    assert_close(out[0, rows], oracle.gemm(a[0, rows].cpu(), w.cpu(), bias[0, rows].cpu(), alpha, beta), torch.float16, "op")
    assert torch.allclose((alpha * (a @ w) + beta * bias).float(), out.float(), atol=6e-1)
    d = torch.empty(S, S, dtype=torch.float16, device=DEV)
    ws = torch.empty(max(capi.lib().minfer_gemm_workspace_bytes(S, S, S), 16), dtype=torch.uint8, device=DEV)   # the op brings one too
    assert capi.gemm_ws(a[0], w, bias[0], d, alpha, beta, ws) == capi.OK
    torch.cuda.synchronize()
    assert torch.equal(d, out[0])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,Nq,Nk,Nv", [
    (4096, 4096, 4096, 1024, 1024),    # Llama-3-8B prefill: 256 x 192 tiles over the weights' columns numbered through (two full rounds)
    (2000, 128, 4096, 1024, 1024),     # 224 x 256: a ragged last tile row and column
    (4096, 128, 4096, 2048, 2048),     # 256 x 256
    (512, 6144, 6144, 1024, 1024),     # the reference test's head shape at a smaller batch: 128 x 128 tiles
    (300, 256, 200, 72, 136),          # ragged rows, widths that end inside a tile
    (593, 128, 12288, 1024, 1088),     # 160 x 256 tiles over the columns numbered through, the last one past the third weight's end
    (300, 320, 12288, 1024, 1088),     # 160 x 128 ones
    (1003, 64, 8192, 1024, 1088),      # 256 x 256 ones
    (1, 4096, 4096, 1024, 1024),       # a decode step, 25 M weight values: the LDS-staged few-row kernel over the three weights' column groups
    (1, 8192, 1032, 8, 520),           # the same with ragged last groups
    (1, 4096, 7176, 1032, 8),          # 33 M: whole weight rows per wave, the three weights' rows numbered through, runs that cross from one to the next
    (1, 8256, 1032, 8, 520),           # the same with the activations in LDS
    (2, 4096, 4096, 1024, 1024),       # up to 16 rows, K a multiple of 512: the LDS-staged few-row kernel over the three weights' column groups
    (13, 1024, 520, 264, 8),           # the same with ragged last groups
    (16, 576, 4096, 1024, 1024),       # K not a multiple of 512: the few-row kernel that loads fragments directly
    (24, 1024, 5120, 1280, 1288),      # stripes of 64 columns, see below
    (24, 192, 4104, 1024, 1032),       # the few-row kernel, two column groups per workgroup, ragged last groups; two blocks of rows
    (40, 448, 5120, 520, 8),           # ... three
    (64, 192, 4096, 1024, 1032),       # ... four
    (64, 512, 768, 256, 256),          # the few-row kernel at its largest row count, one column group per workgroup
    (33, 50, 17, 17, 9),               # nothing tileable: three plain launches
    (300, 320, 1000, 72, 136),         # tiles and 16-column blocks that hold columns of two or three weights
    (1100, 192, 1032, 1000, 8),
    # 5-64 rows, K a multiple of 256, 96 stripes of 64 columns or more over the three weights: the stripe kernel, every weight
    # with workgroups of its own in proportion to its width
    (5, 4096, 4096, 1024, 1024),
    (16, 512, 4096, 1024, 1032),       # a last stripe of 8 columns in the third weight
    (40, 1024, 4104, 1024, 1024),      # ... in the first; three blocks of activation rows
    (64, 256, 5120, 520, 8),           # one segment; a weight of a single partial stripe
])
def test_qkv_one_launch_equals_three_gemms(dtype, M, K, Nq, Nk, Nv):
    """minfer_qkv (one grid over the column tiles of the three weights) against minfer_gemm per weight: from 65 rows on
    the same tiles run the same arithmetic and the results are equal bit for bit; up to 64 rows which few-row kernel runs
    depends on the width, which is the three weights' together in one case and one weight's in the other, and the
    results are equal up to the order of the fp32 sums (every output against the oracle there); k always against the
    oracle."""
    g = torch.Generator().manual_seed(M + K + Nq)
    x = torch.randn(M, K, generator=g).to(dtype).to(DEV)
    ws = [((1 / K ** 0.5) * torch.randn(n, K, generator=g)).to(dtype).to(DEV) for n in (Nq, Nk, Nv)]
    outs = [torch.full((M, n), float("nan"), dtype=dtype, device=DEV) for n in (Nq, Nk, Nv)]
    assert capi.qkv(x, *ws, *outs) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    for w, o, name in zip(ws, outs, "qkv"):
        ref = torch.full_like(o, float("nan"))
        assert capi.gemm(x, w, None, ref, 1.0, 0.0, NK) == capi.OK, capi.last_error()
        torch.cuda.synchronize()
        if M > 64:
            assert torch.equal(o, ref), name
        else:
            assert_close(o, oracle.gemm(x.cpu(), w.cpu(), None, 1.0, 0.0, NK), dtype, name + " against the oracle")
            assert float((o.float() - ref.float()).abs().max()) <= 2.0 ** -MANT[dtype] * float(ref.float().abs().max()), name
    rows = torch.arange(0, M, max(1, M // 24))
    assert_close(outs[1][rows], oracle.gemm(x[rows].cpu(), ws[1].cpu(), None, 1.0, 0.0, NK), dtype, "k against the oracle")


def test_qkv_op_and_reference_checks(kerns):
    """The QKV recipe of the reference's test at a smaller batch (test/kernels.py:173-214: hidden 6144, 48 query and
    8 KV heads of 128): x @ W^T for the three weights stored [out, hidden]."""
    B, L, hidden, q_dim, kv_dim = 2, 512, 6144, 48 * 128, 8 * 128
    g = torch.Generator().manual_seed(3)
    x = torch.randn(B, L, hidden, generator=g).half().to(DEV)
    wq, wk, wv = (((1 / hidden ** 0.5) * torch.randn(n, hidden, generator=g)).half().to(DEV) for n in (q_dim, kv_dim, kv_dim))
    q, k, v = (torch.zeros(B, L, n, dtype=torch.float16, device=DEV) for n in (q_dim, kv_dim, kv_dim))
    assert kerns.qkv(1, 1, 1, 1, 1, 1, 2, 2, 2, x, wq, wk, wv, q, k, v) is None
    torch.cuda.synchronize()
    rows = torch.arange(0, B * L, 64)
    xs = x.view(B * L, hidden)[rows].cpu()
    for out, w, name in ((q, wq, "q"), (k, wk, "k"), (v, wv, "v")):
        assert_close(out.view(B * L, -1)[rows], oracle.gemm(xs, w.cpu(), None, 1.0, 0.0, oracle.GEMM_B_NK), torch.float16, name)
        assert torch.allclose((x @ w.T).float(), out.float(), atol=2e-1)
    # weights stored [hidden, out] are recognised by their shape
    k2 = torch.zeros_like(k)
    kerns.qkv(1, 1, 1, 1, 1, 1, 2, 2, 2, x, wq, wk.T.contiguous(), wv, q, k2, v)
    torch.cuda.synchronize()
    assert float((k2.float() - k.float()).abs().max()) <= 4e-3
    with pytest.raises(RuntimeError):
        kerns.qkv(1, 1, 1, 1, 1, 1, 2, 2, 2, x, wq, wk[:, :100].contiguous(), wv, q, k, v)
    with pytest.raises(RuntimeError):
        kerns.qkv(2, 2, 2, 32, 32, 32, 18, 18, 18, x, wq, wk, wv, q, k, v)          # quantised weights: not implemented
    # gemm's reference checks (gemm/op.cuh:229-273)
    a, w, bias = workloads.gemm_input(64, 64, 64, seed=1, device=DEV)
    out = torch.zeros_like(bias)
    with pytest.raises(RuntimeError):
        kerns.gemm(1, 1, 2, 0.0, 1.0, a, w, bias, out)                              # alpha == 0
    with pytest.raises(RuntimeError):
        kerns.gemm(1, 1, 2, 1.0, 0.0, a[0], w, bias, out)                           # A must be 3-D
    with pytest.raises(RuntimeError):
        kerns.gemm(1, 1, 2, 1.0, 0.0, a, w[:, :32], bias, out)                      # not contiguous / wrong shape
    with pytest.raises(RuntimeError):
        kerns.gemm(1, 1, 2, 1.0, 0.0, a, w.float(), bias, out)
    with pytest.raises((RuntimeError, NotImplementedError)):
        kerns.gemm(1, 1, 2, 1.0, 0.0, a.cpu(), w.cpu(), bias.cpu(), out.cpu())


# ---- K slices through a workspace (minfer_gemm_ws) -------------------------------------------------------------
@pytest.mark.parametrize("layout", [KN, NK])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,alpha,beta", [
    (64, 4096, 4096, 1.0, 0.0),      # [K, N]: 32 tiles of 128 columns, 8 slices of 8 steps; [N, K]: four slices of 64 stripes
    (100, 1032, 2048, 2.0, 3.0),     # tiles of whole rows: the workspace is not needed
    (256, 2048, 1024, 0.5, 1.0),
    (40, 512, 1984, 1.0, 0.0),       # [K, N]: 31 K steps in 7 slices; [N, K]: whole rows
    (1, 4096, 4096, 1.0, 1.0),       # one row: with [K, N] slices of 128 columns, with [N, K] still the few-row kernel
    (24, 1024, 2048, 1.0, 1.0),      # [K, N]: 8 slices of four steps; [N, K]: whole rows
    (256, 8192, 1024, 1.0, 1.0),     # 128 tiles of whole rows
    # [N, K] weights of fewer than 192 stripes of 64 columns: K slices of the stripe kernel, or whole rows where those are ahead
    (8, 5120, 5120, 2.0, 3.0),       # 80 stripes, 320 blocks of 16 columns shared out: the workspace is not needed
    (16, 4104, 8192, 1.0, 1.0),      # three slices, a last stripe of 8 columns
    (33, 8192, 2048, 0.5, 0.0),      # whole rows
    (1, 8192, 4096, 1.0, 0.0),       # one row: whole rows
    (64, 6144, 4096, 1.0, 1.0),      # whole rows
    (12, 1024, 14336, 1.0, 0.0),     # long rows of a small weight: 16 stripes, 14 slices of 4 segments
    (24, 2048, 4096, 2.0, 1.0),      # whole rows
    (3, 1536, 8960, 1.0, 1.0),       # long rows, 24 stripes: slices from 2 rows on (8 slices of 4 or 5 segments)
])
def test_gemm_k_slices_against_oracle(layout, dtype, M, N, K, alpha, beta):
    a, b, c = make(M, N, K, layout, dtype, seed=M + N + K)
    need = capi.lib().minfer_gemm_workspace_bytes(M, N, K)
    assert need > 0 and need % (4 * M * N) == 0, need
    exact = oracle.gemm(a.float().numpy(), b.float().numpy(), c.float().numpy(), alpha, beta, layout)
    da, db, dc = a.to(DEV), b.to(DEV), c.to(DEV)
    d = torch.zeros(M, N, dtype=dtype, device=DEV)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=DEV)      # NaN patterns: every slot read must have been written
    assert capi.gemm_ws(da, db, dc, d, alpha, beta, ws, layout) == capi.OK, capi.last_error()
    assert_close(d, exact, dtype, "k slices")
    # a workspace that is too small, or none, is the plain call
    d2 = torch.zeros_like(d)
    assert capi.gemm_ws(da, db, dc, d2, alpha, beta, ws[: 4 * M * N], layout) == capi.OK, capi.last_error()   # room for one slice: no path takes it
    d3 = torch.zeros_like(d)
    assert capi.gemm(da, db, dc, d3, alpha, beta, layout) == capi.OK, capi.last_error()
    assert torch.equal(d2, d3)
    assert_close(d2, exact, dtype, "fallback")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [
    (1, 8, 64),          # one K step, one column block half a wave wide
    (16, 128, 128),      # one tile
    (17, 136, 512),      # a second tile of 8 columns; four slices of two steps
    (32, 264, 576),      # nine steps
    (33, 4096, 4096),    # eight slices of as many steps as the ring has stages
    (48, 1000, 3072),
    (49, 520, 5120),     # slices longer than the ring
    (64, 4104, 2048),
    (64, 33000, 128),    # more tiles than compute units
])
def test_few_rows_against_a_kn_weight(dtype, M, N, K):
    """The [K, N] kernel of up to 64 rows: edges of its row blocks, column tiles, K slices and ring, with slices that meet inside
    the launch (twice on one stream: the arrival counters end as they began), in a second launch (under graph capture, same
    bits) and without a workspace; the bound is this file's."""
    a, b, c = make(M, N, K, KN, dtype, seed=M + N + K)
    exact = oracle.gemm(a.float().numpy(), b.float().numpy(), c.float().numpy(), 2.0, 3.0, KN)
    da, db, dc = a.to(DEV), b.to(DEV), c.to(DEV)
    need = capi.lib().minfer_gemm_workspace_bytes(M, N, K)
    ws = torch.full((max(need, 16),), 0xFF, dtype=torch.uint8, device=DEV)
    outs = [torch.full((M, N), float("nan"), dtype=dtype, device=DEV) for _ in range(4)]
    for d in outs[:2]:
        assert capi.gemm_ws(da, db, dc, d, 2.0, 3.0, ws, KN) == capi.OK, capi.last_error()
    assert capi.gemm(da, db, dc, outs[2], 2.0, 3.0, KN) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert capi.gemm_ws(da, db, dc, outs[3], 2.0, 3.0, ws, KN) == capi.OK, capi.last_error()
    for _ in range(2):
        outs[3].fill_(float("nan"))
        ws.fill_(0xFF)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(outs[3], outs[0])
    assert torch.equal(outs[1], outs[0])
    assert_close(outs[0], exact, dtype, "slices")
    assert_close(outs[2], exact, dtype, "no workspace")


@pytest.mark.parametrize("M,N,K", [(9, 1000, 4096), (40, 4096, 4096), (64, 2056, 2048)])
def test_few_rows_against_a_kn_weight_in_a_smaller_workspace(M, N, K):
    """A workspace one byte short of minfer_gemm_workspace_bytes, one of two slices and one of less than two: as many slices as it
    holds, eight at most, none past its end; the bound is this file's."""
    a, b, c = make(M, N, K, KN, torch.float16, seed=M + N)
    exact = oracle.gemm(a.float().numpy(), b.float().numpy(), c.float().numpy(), 2.0, 3.0, KN)
    da, db, dc = a.to(DEV), b.to(DEV), c.to(DEV)
    need = capi.lib().minfer_gemm_workspace_bytes(M, N, K)
    for size in (need - 1, 2 * 4 * M * N, 2 * 4 * M * N - 1):
        ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=DEV)
        d = torch.full((M, N), float("nan"), dtype=torch.float16, device=DEV)
        assert capi.gemm_ws(da, db, dc, d, 2.0, 3.0, ws[:size], KN) == capi.OK, capi.last_error()
        torch.cuda.synchronize()
        assert_close(d, exact, torch.float16, f"{size} bytes")
        slices = ws[:need // (4 * M * N) * 4 * M * N].view(-1, 4 * M * N)
        written = [bool((s != 0xFF).any()) for s in slices]
        fit = min(size // (4 * M * N), 8)
        assert written == [i < fit and fit > 1 for i in range(len(written))], (size, written)


def sliced_call(a, b, c, layout, M, N, K):
    """2 A B + 3 C with a workspace of minfer_gemm_workspace_bytes that holds a NaN pattern: every slot read must have been written."""
    ws = torch.full((capi.lib().minfer_gemm_workspace_bytes(M, N, K),), 0xFF, dtype=torch.uint8, device=DEV)
    d = torch.full((M, N), float("nan"), dtype=a.dtype, device=DEV)
    assert capi.gemm_ws(a, b, c, d, 2.0, 3.0, ws, layout) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    return ws, d


def written_slices(ws, M, N):
    """How many slices of M x N sums the call wrote, from the workspace's start on and without a gap."""
    written = [bool((x != 0xFF).any()) for x in ws[:ws.numel() // (4 * M * N) * 4 * M * N].view(-1, 4 * M * N)]
    assert written == sorted(written, reverse=True)
    return sum(written)


@pytest.mark.parametrize("layout,M,N,K,slices,tile", [   # tile: rows, columns, workgroups to a unit
    (NK, 70, 8136, 8256, 4, (128, 128, 1)),
    (KN, 70, 8136, 8256, 4, (128, 128, 1)),
    (NK, 250, 8072, 4160, 2, (128, 128, 1)),
    (KN, 129, 8072, 4160, 3, (160, 128, 1)),
    (KN, 130, 272, 5952, 31, (128, 128, 1)),
    (KN, 987, 2616, 8000, 3, (128, 128, 2)),
    (KN, 65, 8312, 7936, 7, (128, 256, 1)),
    (KN, 964, 136, 2496, 13, (160, 128, 1)),
    (KN, 261, 5560, 6848, 5, (160, 256, 1)),
    (KN, 162, 5488, 2112, 3, (192, 128, 1)),
    (KN, 517, 6864, 8384, 3, (192, 256, 1)),
    (KN, 199, 5384, 4160, 5, (224, 128, 1)),
    (KN, 391, 5384, 8896, 5, (224, 256, 1)),
    (KN, 487, 8584, 8064, 3, (256, 256, 1)),
    (NK, 129, 264, 6080, 31, (128, 128, 1)),
    (NK, 487, 3112, 11200, 5, (128, 128, 2)),
    (NK, 67, 8208, 5056, 5, (128, 192, 1)),
    (NK, 322, 5488, 4032, 3, (128, 256, 1)),
    (NK, 980, 136, 2496, 13, (160, 128, 1)),
    (NK, 258, 5424, 5376, 5, (160, 224, 1)),
    (NK, 261, 5744, 6720, 5, (160, 256, 1)),
    (NK, 163, 2064, 6336, 11, (192, 128, 1)),
    (NK, 327, 5400, 4544, 4, (192, 192, 1)),
    (NK, 527, 4104, 16960, 5, (192, 256, 1)),
    (NK, 193, 5464, 4160, 5, (224, 128, 1)),
    (NK, 387, 5448, 5312, 4, (224, 192, 1)),
    (NK, 386, 6296, 9920, 5, (224, 256, 1)),
    (NK, 485, 3096, 19264, 9, (256, 224, 1)),
    (NK, 227, 8240, 14784, 7, (256, 256, 1)),
])
def test_gemm_k_slices_of_tiles(gemm_plan, layout, M, N, K, slices, tile):
    """Every tile that the plan cuts K for, in each layout, a last tile row and column that are not full, slices of different lengths: so
    many slices written and no more, every element against torch's product in 64 bits within the bound of assert_close."""
    assert gemm_plan(M, N, K, layout == NK, rules.MOST_SLICES) == (rules.TILES, slices, *tile)
    dtype = torch.float16 if (M + K // 64) % 2 else torch.bfloat16
    a, b, c = (x.to(DEV) for x in make(M, N, K, layout, dtype, M + N + K))
    ws, d = sliced_call(a, b, c, layout, M, N, K)
    assert written_slices(ws, M, N) == slices
    exact = 2.0 * torch.mm(a.double(), (b if layout == KN else b.T.contiguous()).double()) + 3.0 * c.double()
    assert_close(d, exact.cpu().numpy(), dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,slices", [
    (9, 520, 6144, 6),       # one block of activation rows; a last stripe of 8 columns
    (17, 520, 8448, 8),      # two, the second of one row; 33 segments
    (32, 3080, 8448, 5),
    (33, 2056, 4352, 4),     # three; 17 segments
    (48, 1544, 9216, 9),
    (49, 1032, 8448, 8),     # four
    (64, 3080, 6144, 5),
])
def test_gemm_k_slices_of_stripes(gemm_plan, dtype, M, N, K, slices):
    """K slices of the stripe kernel with every number of activation row blocks, their edges: as above."""
    assert gemm_plan(M, N, K, rules.NK, rules.MOST_SLICES)[:2] == (rules.STRIPE_SLICES, slices)
    a, b, c = (x.to(DEV) for x in make(M, N, K, NK, dtype, M + N + K))
    ws, d = sliced_call(a, b, c, NK, M, N, K)
    assert written_slices(ws, M, N) == slices
    assert_close(d, (2.0 * torch.mm(a.double(), b.T.contiguous().double()) + 3.0 * c.double()).cpu().numpy(), dtype)


@pytest.mark.parametrize("layout,M,N,K,kernel,slices", [   # just past and just below where K slices are taken from 17 rows on
    (NK, 28, 2560, 5120, rules.STRIPE_SLICES, 5), (NK, 24, 2560, 5120, rules.STRIPE, 1),
    (NK, 63, 3080, 4096, rules.STRIPE_SLICES, 4), (NK, 41, 3072, 4096, rules.STRIPE_SLICES, 4), (NK, 40, 3072, 4096, rules.STRIPE, 1),
    (NK, 40, 4096, 6144, rules.STRIPE_SLICES, 4), (NK, 35, 4096, 6144, rules.STRIPE_SLICES, 4), (NK, 34, 4096, 6144, rules.STRIPE, 1),
    (NK, 64, 4096, 4096, rules.STRIPE_SLICES, 4), (NK, 59, 4096, 4096, rules.STRIPE, 1),
    (NK, 30, 4096, 8192, rules.STRIPE_SLICES, 4), (NK, 29, 4096, 8192, rules.STRIPE, 1),
    (KN, 17, 264, 4160, rules.KN_ROWS, 16), (KN, 64, 1024, 4096, rules.KN_ROWS, 16), (KN, 64, 1032, 4096, rules.KN_ROWS, 8),
])
def test_gemm_k_slices_beside_their_lines(gemm_plan, layout, M, N, K, kernel, slices):
    assert gemm_plan(M, N, K, layout == NK, rules.MOST_SLICES)[:2] == (kernel, slices)
    a, b, c = (x.to(DEV) for x in make(M, N, K, layout, torch.float16, M + N + K))
    ws, d = sliced_call(a, b, c, layout, M, N, K)
    assert written_slices(ws, M, N) == (slices if slices > 1 else 0)
    exact = 2.0 * torch.mm(a.double(), (b if layout == KN else b.T.contiguous()).double()) + 3.0 * c.double()
    assert_close(d, exact.cpu().numpy(), torch.float16)


Q8 = "q8_0"


@pytest.mark.parametrize("dtype,weight,M,N,K,slices", [(dtype, *case) for case in [
    (KN, 1, 4096, 4096, 8), (KN, 9, 1000, 4096, 8), (KN, 16, 264, 8192, 16),   # up to 16 rows: a tile's last workgroup adds the slices up
    (NK, 9, 520, 6144, 6), (NK, 16, 2048, 8192, 8),
    (Q8, 9, 1544, 8448, 8), (Q8, 2, 520, 8192, 8),
    (KN, 17, 264, 4160, 16), (KN, 40, 4096, 4096, 8),                          # more: a second launch does
    (NK, 17, 520, 8448, 8), (NK, 64, 3080, 6144, 5),
    (Q8, 17, 2056, 6144, 6),
    (KN, 130, 272, 5952, 31), (NK, 322, 5488, 4032, 3),                        # K slices of tiles
] for dtype in (torch.float16, torch.bfloat16) if dtype == torch.float16 or case[0] != Q8])   # (a Q8_0 weight has float16 activations)
def test_gemm_adds_c_in_place_over_k_slices(gemm_plan, dtype, weight, M, N, K, slices):
    """The residual added in place over K slices, in rows of a wider buffer that start at multiples of 8 bytes only: bit-equal to the call
    with C apart on the null stream and on one without counters, nothing else written."""
    if weight == Q8:
        a, b, c, w = make_q8(M, N, K, M + N + K)
        assert gemm_plan.q8(M, N, K, True, rules.MOST_SLICES) == (rules.Q8_STRIPE_SLICES, slices)
        w = w.T.contiguous()
    else:
        a, b, c = make(M, N, K, weight, dtype, M + N + K)
        assert gemm_plan(M, N, K, weight == NK, rules.MOST_SLICES)[1] == slices
        w = b if weight == KN else b.T.contiguous()
    a, b, c = a.to(DEV), b.to(DEV), c.to(DEV)
    ws = torch.empty(4 * M * N * slices, dtype=torch.uint8, device=DEV)

    def call(c, d):
        ws.fill_(0xFF)
        rc = capi.gemm_q8_0(a, b, c, d, 2.0, 3.0, ws) if weight == Q8 else capi.gemm_ws(a, b, c, d, 2.0, 3.0, ws, weight)
        assert rc == capi.OK, capi.last_error()
        assert written_slices(ws, M, N) == slices

    d = torch.full_like(c, float("nan"))
    call(c, d)
    assert_close(d, (2.0 * torch.mm(a.double(), w.to(DEV).double()) + 3.0 * c.double()).cpu().numpy(), dtype)
    wide = torch.full((M + 2, N + 12), float("nan"), dtype=dtype, device=DEV)
    view = wide[1:M + 1, 4:N + 4]
    torch.cuda.synchronize()
    for stream in (torch.cuda.default_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            view.copy_(c)
            call(view, view)
            assert torch.equal(view, d)
            view.fill_(float("nan"))
            assert torch.isnan(wide).all()
        stream.synchronize()


def test_gemm_workspace_bytes_is_zero_where_tiles_fill_the_chip():
    L = capi.lib()
    assert L.minfer_gemm_workspace_bytes(4096, 4096, 4096) == 0
    assert L.minfer_gemm_workspace_bytes(64, 4096, 100) == 0       # K not a multiple of 64
    assert L.minfer_gemm_workspace_bytes(64, 4096, 256) == 0       # too few K steps to slice
    assert L.minfer_gemm_workspace_bytes(0, 4096, 4096) == 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gemm_op_uses_k_slices_and_matches_oracle(dtype):
    from minfer.kernels import KernelBackend
    from minfer.const import GGMLQuantizationType, GGML_QUANT_SIZES
    kerns = KernelBackend("torch_ext")
    qt = GGMLQuantizationType.F16 if dtype == torch.float16 else GGMLQuantizationType.BF16
    qb, qs = GGML_QUANT_SIZES[qt]
    M, N, K = 96, 2048, 4096
    a, b, c = make(M, N, K, KN, dtype, seed=5)
    exact = oracle.gemm(a.float().numpy(), b.float().numpy(), c.float().numpy(), 1.0, 1.0, KN)
    A, Cc = a.view(2, 48, K).to(DEV), c.view(2, 48, N).to(DEV)
    D = torch.empty_like(Cc)
    kerns.gemm(qt, qb, qs, 1.0, 1.0, A, b.to(DEV), Cc, D)
    assert_close(D.view(M, N), exact, dtype, "gemm op, k slices")


# ---- weights stored as Q8_0 blocks (minfer_gemm_q8_0; the gemm op with the type triple (8, 32, 34)) -----------------
def make_q8(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, K, generator=g).half()
    w = (1 / K ** 0.5) * torch.randn(N, K, generator=g)
    c = torch.randn(M, N, generator=g).half()
    wq = torch.from_numpy(oracle.quant_q8_0(w.numpy()))                        # uint8 [N, K/32*34]
    w_deq = torch.from_numpy(oracle.dequant_q8_0(wq.numpy(), np.float16))      # what every kernel must multiply with
    return a, wq, c, w_deq


@pytest.mark.parametrize("M,N,K,alpha,beta", [
    (1, 4096, 4096, 1.0, 0.0),       # a decode step against a Llama-3-8B projection: the kernel that streams the blocks
    (8, 1024, 4096, 1.0, 1.0),
    (16, 256, 14336, 2.0, 3.0),      # a long contraction split over the eight waves
    (17, 5152, 192, 1.0, 0.0),       # two column groups per workgroup, a ragged last one
    (4, 5200, 512, 1.0, 1.0),        # one block of rows
    (40, 5160, 448, 2.0, 1.0),       # three and four blocks of rows with two column groups
    (64, 5120, 192, 1.0, 0.0),
    (17, 5152, 256, 1.0, 0.0),       # K a multiple of 256: the stripe kernel, see below
    (40, 5152, 512, 2.0, 1.0),
    (64, 5120, 256, 1.0, 0.0),
    (64, 264, 192, 0.5, 1.0),        # its largest row count; K a multiple of 64 but not of 128: a short last step
    (37, 24, 64, 1.0, 1.0),          # one step, half-empty column group
    (65, 256, 256, 1.0, 2.0),        # above 64 rows: dequantise into the workspace, then the fp16 kernels
    (300, 1032, 512, 2.0, 0.0),
    (5, 64, 96, 1.0, 1.0),           # an odd number of blocks per row: workspace path at any row count
    (3, 18, 256, 1.0, 1.0),          # out_dim not a multiple of 4 with few rows: workspace path as well
    (64, 1030, 128, 2.0, 0.0),
    # one row with K a multiple of 256: the kernel that streams whole weight rows (segments of 128 blocks)
    (1, 264, 14336, 2.0, 1.0),       # three whole segments and one of 64 blocks, the activations in LDS
    (1, 520, 4352, 1.0, 0.0),        # a last segment of 8 blocks
    (1, 2052, 768, 0.5, 1.0),        # a single segment of 24 blocks, the activations in registers
    (1, 20000, 256, 1.0, 1.0),       # ten weight rows per wave
    (1, 4, 256, 1.0, 0.0),           # one wave with four rows, the others none
    (1, 4096, 16384, 1.0, 0.0),      # the longest activation row its LDS area holds
    (1, 512, 16640, 1.0, 0.0),       # longer: back to the 16-rows-per-instruction kernel
    (2, 2052, 768, 0.5, 1.0),        # two rows: that kernel as well
    # 2-64 rows with K a multiple of 256: the stripe kernel over the raw blocks (16-column blocks shared out, chunks of four)
    (9, 12296, 256, 1.0, 1.0),       # 769 blocks over 256 workgroups, the last one half empty; one segment
    (33, 6152, 1024, 2.0, 3.0),      # from 33 rows on narrower weights too; three blocks of rows, chunks of one and two blocks
    (48, 12288, 2560, 1.0, 0.0),     # ten segments
    (64, 12304, 512, 0.5, 1.0),      # chunks of four and of three blocks
    (16, 8192, 4096, 1.0, 0.0),      # two blocks per workgroup
    (2, 14336, 4096, 1.0, 0.0),
    # fewer than 192 stripes and a workspace: K slices of the stripe kernel, summed by a second launch
    (16, 4096, 14336, 1.0, 1.0),     # 4 slices of 14 segments
    (33, 5120, 5120, 2.0, 0.0),      # 3 slices of 7, 7 and 6 segments; three blocks of rows
    (8, 8192, 8192, 1.0, 0.0),       # 2 slices
    (64, 4104, 2048, 0.5, 1.0),      # 65 stripes, the last of 8 columns: whole rows, the workspace is not needed
    (2, 6144, 4096, 1.0, 0.0),       # ... as here
    (3, 1536, 8960, 1.0, 1.0),       # long rows, 24 stripes: 8 slices of 4 or 5 segments
])
def test_gemm_q8_0_weights_against_oracle(M, N, K, alpha, beta):
    a, wq, c, w_deq = make_q8(M, N, K, seed=M * 7 + N + K)
    exact = oracle.gemm(a.float().numpy(), w_deq.float().numpy(), c.float().numpy(), alpha, beta, NK)
    da, dwq, dc = a.to(DEV), wq.to(DEV), c.to(DEV)
    d = torch.zeros(M, N, dtype=torch.float16, device=DEV)
    need = capi.lib().minfer_gemm_q8_0_workspace_bytes(M, N, K)
    streams = M <= 64 and (K // 32) % 2 == 0 and N % 4 == 0      # the raw blocks are multiplied: a workspace only for K slices
    assert streams or need > 0
    if streams:
        stripes = (N + 63) // 64
        slices = min(256 // stripes, K // 1024, 16) if M >= 2 and K % 256 == 0 and N % 8 == 0 and stripes < 192 and (N * K > 1 << 24 or M >= 16 or (K >= 6144 and M >= 8) or (K >= 8192 and stripes <= 24)) else 1
        assert need == (slices * M * N * 4 if slices > 1 else 0)
    ws = torch.full((max(need, 16),), 0xFF, dtype=torch.uint8, device=DEV)
    assert capi.gemm_q8_0(da, dwq, dc, d, alpha, beta, ws if need else None) == capi.OK, capi.last_error()
    assert_close(d, exact, torch.float16, "q8_0 weight")
    if streams and need:            # the slices are optional: without the workspace, or with too small a one, one launch
        for small in (None, ws[:need // 2]):
            d.fill_(float("nan"))
            assert capi.gemm_q8_0(da, dwq, dc, d, alpha, beta, small) == capi.OK, capi.last_error()
            assert_close(d, exact, torch.float16, "q8_0 weight, no slices")
    # the same numbers as the fp16 kernel on the dequantised weight, up to the order of the fp32 sums
    d_ref = torch.zeros_like(d)
    assert capi.gemm(da, w_deq.to(DEV), dc, d_ref, alpha, beta, NK) == capi.OK, capi.last_error()
    assert_close(d_ref, exact, torch.float16, "fp16 kernel on the dequantised weight")
    if not streams:
        assert capi.gemm_q8_0(da, dwq, dc, d, alpha, beta, None) == capi.EWORKSPACE and "workspace" in capi.last_error()


@pytest.mark.parametrize("M,N,K,slices", [
    (9, 1544, 8448, 8),      # one block of activation rows; a last stripe of 8 columns; 33 segments
    (17, 2056, 6144, 6),     # two, the second of one row
    (32, 4104, 4352, 3),     # 17 segments
    (48, 3080, 6144, 5),     # three
    (64, 2056, 4608, 4),     # four
])
def test_gemm_q8_0_k_slices_of_stripes(gemm_plan, M, N, K, slices):
    """K slices of the stripe kernel over Q8_0 blocks with every number of activation row blocks: so many slices written, every element
    against torch's product with the dequantised weight in 64 bits, within the bound of assert_close."""
    assert gemm_plan.q8(M, N, K, True, slices) == (rules.Q8_STRIPE_SLICES, slices)
    a, wq, c, w = make_q8(M, N, K, seed=M + N + K)
    ws = torch.full((capi.lib().minfer_gemm_q8_0_workspace_bytes(M, N, K),), 0xFF, dtype=torch.uint8, device=DEV)
    d = torch.full((M, N), float("nan"), dtype=torch.float16, device=DEV)
    assert capi.gemm_q8_0(a.to(DEV), wq.to(DEV), c.to(DEV), d, 2.0, 3.0, ws) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert written_slices(ws, M, N) == slices
    assert_close(d, (2.0 * (a.double() @ w.double().T) + 3.0 * c.double()).numpy(), torch.float16)


@pytest.mark.parametrize("M,N,K,alpha,beta", [
    (65, 10248, 2048, 2.0, 3.0),     # 48 rows and 17
    (96, 4104, 4096, 1.0, 0.0),      # 48 and 48 in K slices, in the workspace that a dequantised weight would take
    (113, 10248, 2048, 1.0, 1.0),    # 64 and 49
    (128, 6152, 4096, 0.5, 0.0),
    (130, 12296, 4352, 1.0, 1.0),    # 48, 48 and 34
    (96, 4100, 4096, 2.0, 1.0),      # 48 and 48 where the dequantised weight is no width for the tiled kernel
    (65, 4100, 4160, 1.0, 0.0),      # ... and K is no whole segments
])
def test_gemm_q8_0_in_parts(M, N, K, alpha, beta):
    """65 to 160 rows against a large weight go through the block-streaming kernels in parts: every element against torch's product
    with the dequantised weight in 64 bits, within the bound of assert_close; no less workspace is accepted than before."""
    a, wq, c, w_deq = make_q8(M, N, K, seed=M + N)
    need = capi.lib().minfer_gemm_q8_0_workspace_bytes(M, N, K)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device=DEV)
    d = torch.full((M, N), float("nan"), dtype=torch.float16, device=DEV)
    da, dwq, dc = a.to(DEV), wq.to(DEV), c.to(DEV)
    assert capi.gemm_q8_0(da, dwq, dc, d, alpha, beta, ws) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert_close(d, (alpha * (a.double() @ w_deq.double().T) + beta * c.double()).numpy(), torch.float16)
    assert capi.gemm_q8_0(da, dwq, dc, d, alpha, beta, ws[:N * K * 2 - 256]) == capi.EWORKSPACE


def test_gemm_op_with_q8_0_weight(kerns):
    M, N, K = 8, 2048, 4096
    a, wq, c, w_deq = make_q8(M, N, K, seed=3)
    exact = oracle.gemm(a.float().numpy(), w_deq.float().numpy(), c.float().numpy(), 1.0, 1.0, NK)
    A, Cc = a.view(2, 4, K).to(DEV), c.view(2, 4, N).to(DEV)
    D = torch.empty_like(Cc)
    assert kerns.gemm(8, 32, 34, 1.0, 1.0, A, wq.to(DEV), Cc, D) is None
    assert_close(D.view(M, N), exact, torch.float16, "gemm op, q8_0 weight")
    A2 = torch.randn(1, 200, K, dtype=torch.float16, device=DEV)
    C2 = torch.zeros(1, 200, N, dtype=torch.float16, device=DEV)
    D2 = torch.empty_like(C2)
    kerns.gemm(8, 32, 34, 1.0, 0.0, A2, wq.to(DEV), C2, D2)                      # prefill-sized: workspace path
    exact2 = oracle.gemm(A2[0].float().cpu().numpy(), w_deq.float().numpy(), None, 1.0, 0.0, NK)
    assert_close(D2[0], exact2, torch.float16, "gemm op, q8_0 weight, 200 rows")
    with pytest.raises(RuntimeError, match="Unsupported dims"):
        kerns.gemm(8, 32, 34, 1.0, 0.0, A2, wq.to(DEV)[:, :-34].contiguous(), C2, D2)
    with pytest.raises(RuntimeError, match="float16"):
        kerns.gemm(8, 32, 34, 1.0, 0.0, A2.bfloat16(), wq.to(DEV), C2.bfloat16(), D2.bfloat16())


def test_qkv_op_with_q8_0_weights(kerns):
    """The reference's QKV recipe (test/kernels.py:173-214) with the k and v weights as Q8_0 blocks and q as float16."""
    B, L, K, Nq, Nkv = 2, 3, 2048, 1024, 256
    g = torch.Generator().manual_seed(11)
    x = torch.randn(B, L, K, generator=g).half()
    wq = ((1 / K ** 0.5) * torch.randn(Nq, K, generator=g)).half()
    wk = (1 / K ** 0.5) * torch.randn(Nkv, K, generator=g)
    wv = (1 / K ** 0.5) * torch.randn(Nkv, K, generator=g)
    wk8, wv8 = (torch.from_numpy(oracle.quant_q8_0(w.numpy())) for w in (wk, wv))
    q, k, v = (torch.empty(B, L, n, dtype=torch.float16, device=DEV) for n in (Nq, Nkv, Nkv))
    assert kerns.qkv(1, 8, 8, 1, 32, 32, 2, 34, 34, x.to(DEV), wq.to(DEV), wk8.to(DEV), wv8.to(DEV), q, k, v) is None
    x2 = x.view(B * L, K).float().numpy()
    assert_close(q.view(B * L, Nq), oracle.gemm(x2, wq.float().numpy(), None, 1.0, 0.0, NK), torch.float16, "q")
    for out, w8, name in ((k, wk8, "k"), (v, wv8, "v")):
        w_deq = torch.from_numpy(oracle.dequant_q8_0(w8.numpy(), np.float16)).float().numpy()
        assert_close(out.view(B * L, Nkv), oracle.gemm(x2, w_deq, None, 1.0, 0.0, NK), torch.float16, name)
    with pytest.raises(RuntimeError, match="Q8_0 weight is uint8"):
        kerns.qkv(1, 8, 8, 1, 32, 32, 2, 34, 34, x.to(DEV), wq.to(DEV), wk8.to(DEV)[:, :-34].contiguous(), wv8.to(DEV), q, k, v)
