"""The rules of the GEMM dispatch (csrc/gemm_plan.h), compiled for the host: which kernel takes a call, when a plan of tiles is
estimated and how often."""
import pytest

import capi
from gemm_plan_probe import KN, KN_ROWS, NK, PLAIN, Q8_STRIPE, Q8_STRIPE_SLICES, STRIPE, STRIPE_SLICES, TILES


@pytest.fixture
def plan(gemm_plan):
    return gemm_plan


# (out, in) of the projections of a layer: q, k and v fused, output, gate and up, down; and the sizes of a narrower model
LAYERS = [[(6144, 4096), (4096, 4096), (28672, 4096), (14336, 4096), (4096, 14336)], [(10240, 8192), (8192, 8192), (57344, 8192), (8192, 28672)],
          [(2048, 1536), (1536, 1536), (17920, 1536), (8960, 1536), (1536, 8960)]]


@pytest.mark.parametrize("M", [65, 100, 200, 600, 1777, 4096])
@pytest.mark.parametrize("layer", LAYERS)
def test_the_projections_of_a_layer_keep_their_plans(plan, layer, M):
    """The second walk through a layer estimates nothing, with weights of either layout, a workspace or none, and the grouped projection."""
    def walk():
        for N, K in layer:
            for nt in (KN, NK):
                plan(M, N, K, nt, 64)
        plan.grouped_tile(M, layer[0][0], layer[0][1])
    walk()
    before = plan.estimates()
    walk()
    assert plan.estimates() == before


def test_a_call_with_a_smaller_workspace_keeps_its_plan(plan):
    assert plan(100, 4096, 14336, NK, 64)[1] > 2
    plan(100, 4096, 14336, NK, 2)
    before = plan.estimates()
    assert plan(100, 4096, 14336, NK, 2)[1] <= 2 and plan(100, 4096, 14336, NK, 64)[1] > 2
    assert plan.estimates() == before


def test_few_rows_need_no_plan_of_tiles(plan):
    """Up to 16 rows of an [N, K] weight, up to 64 of a [K, N] weight, and up to 64 where K is whole segments of the stripe kernel."""
    before = plan.estimates()
    for fit in (0, 1, 2, 64):
        for N, K in [s for layer in LAYERS for s in layer] + [(1000, 4160), (264, 16448), (128256, 4096), (512, 64)]:
            for M in (1, 2, 5, 16):
                assert plan(M, N, K, NK, fit)[0] not in (TILES, PLAIN)
            for M in (1, 16, 17, 64):
                assert plan(M, N, K, KN, fit)[0] == KN_ROWS
            if K % 256 == 0 and N >= 6144:
                for M in (17, 40, 64):
                    assert plan(M, N, K, NK, fit)[0] in (STRIPE, STRIPE_SLICES)
    assert plan.estimates() == before


@pytest.mark.parametrize("M,N,K,most", [(9, 1000, 4096, 8), (1, 512, 8192, 16), (40, 4096, 4096, 8), (17, 264, 14336, 16), (64, 14336, 4096, 2), (64, 33000, 4096, 1)])
def test_a_kn_weight_gets_no_more_slices_from_a_smaller_workspace(plan, M, N, K, most):
    """As many as it holds, up to what a call with all the room takes."""
    for fit in range(65):
        assert plan(M, N, K, KN, fit)[:2] == (KN_ROWS, max(1, min(fit, most))), fit


def layout_slices(layout, M, N, K):
    need = capi.lib().minfer_gemm_layout_workspace_bytes(layout, M, N, K)
    assert need % (4 * M * N) == 0
    return need // (4 * M * N)


def test_workspace_of_a_layout_is_what_its_route_uses(plan):
    """minfer_gemm_layout_workspace_bytes: no less than a call can use, and no more."""
    # whole rows of an [N, K] weight: from 96 stripes of 64 columns on always, and where stripe_blocks_pay says so
    for M, N, K in ((40, 8192, 2048), (64, 6144, 4096), (9, 12280, 8192), (59, 4096, 4096), (29, 4096, 8192), (24, 2048, 4096)):
        assert layout_slices(capi.GEMM_B_NK, M, N, K) == 0
    # a [K, N] weight: eight slices, or sixteen of long rows, however many would fill the chip
    assert layout_slices(capi.GEMM_B_KN, 9, 1000, 4096) == 8 and layout_slices(capi.GEMM_B_KN, 9, 1000, 8192) == 16
    for M in (1, 3, 9, 16, 17, 40, 64, 65, 100, 300, 600, 1777):
        for N in (8, 520, 1000, 1536, 4096, 4104, 6144, 8192, 14336):
            for K in (64, 256, 512, 1984, 4096, 4160, 8192, 8960, 14336):
                for layout, nt in ((capi.GEMM_B_KN, KN), (capi.GEMM_B_NK, NK)):
                    slices = layout_slices(layout, M, N, K)
                    assert slices * 4 * M * N <= capi.lib().minfer_gemm_workspace_bytes(M, N, K)
                    best = plan(M, N, K, nt, 64)
                    assert plan(M, N, K, nt, slices) == best and best[1] == max(slices, 1), (M, N, K, layout)


def test_parts_of_a_q8_0_product_are_streamed(plan):
    """65 to 160 rows against a large Q8_0 weight: whatever goes in parts, every part as it runs is a product that a kernel streams, one of
    the stripe kernels wherever the tiled kernel could take the dequantised weight."""
    assert plan.q8_part_rows(65, 14336, 4096, 1) == 48 and plan.q8_part_rows(160, 14336, 4096, 1) == 64
    assert plan.q8_part_rows(64, 14336, 4096, 1) == 64 and plan.q8_part_rows(161, 14336, 4096, 1) == 161   # whole
    assert plan.q8_part_rows(65, 10246, 4096, 1) == 65      # a width that no kernel streams: dequantised once, not once a part
    assert plan.q8_part_rows(65, 14336, 4096, 0) == 65      # a weight off the 16-byte boundaries
    assert plan.q8_part_rows(96, 4100, 4096, 1) == 48       # streamed, and no width for the tiled kernel
    in_parts = 0
    for M in range(65, 161):
        for N in (1024, 1536, 2048, 3000, 4096, 4100, 4104, 5120, 6144, 6146, 8192, 8196, 10240, 10244, 14336, 28672, 128256):
            for K in (1024, 2048, 4096, 4160, 8192, 8960, 14336):
                rows = plan.q8_part_rows(M, N, K, 1)
                room = N * K * 2
                for m in range(0, M, rows) if rows < M else ():
                    r = min(rows, M - m)
                    assert N % 4 == 0 and (K // 32) % 2 == 0, (M, N, K, r)
                    assert N % 8 != 0 or plan.q8(r, N, K, 1, min(room // (r * N * 4), 32))[0] in (Q8_STRIPE, Q8_STRIPE_SLICES), (M, N, K, r)
                    in_parts += 1
    assert in_parts > 5000


def test_slices_that_meet_inside_the_launch_have_pieces_and_counters(plan):
    """Wherever a launch adds its slices up itself: two pieces of four columns for each of a workgroup's 256 threads hold the tile (128 columns
    of a [K, N] weight, 64 of the others), there is a counter for every tile, and the sums are 2 MiB at most."""
    assert plan.meet_rows * 128 // 4 <= 2 * 256
    met = 0
    for M in range(1, 20):
        for N in (8, 64, 72, 520, 1000, 2048, 4096, 4104, 6144, 8192, 12280, 12288, 16384, 16392, 33000):
            for K in (512, 1024, 2048, 4096, 8192, 14336, 28672):
                for kernel, slices, columns in (*((*plan(M, N, K, KN, fit)[:2], 128) for fit in (2, 7, 64)), (*plan(M, N, K, NK, 64)[:2], 64), (*plan.q8(M, N, K, 1, 64), 64)):
                    if slices > 1 and kernel != TILES and plan.slices_meet(M):
                        assert M <= plan.meet_rows and -(-N // columns) <= plan.meet_tiles and slices * M * N * 4 <= 2 << 20, (M, N, K, kernel, slices)
                        met += 1
    assert met > 1000
    assert plan.slices_meet(16) and not plan.slices_meet(17)
