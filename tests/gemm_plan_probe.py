"""csrc/gemm_plan.h, the rules of the GEMM dispatch, compiled for the host as they are: which kernel a call goes to, in which tiles
and in how many K slices, on 256 compute units."""
import ctypes
import os
import subprocess

import capi

PLAIN, GEMV, ROWS_LDS, SKINNY, STRIPE, STRIPE_SLICES, KN_ROWS, TILES = range(8)   # enum GemmKernel
Q8_GEMV, Q8_STRIPE, Q8_STRIPE_SLICES, Q8_SKINNY = range(4)                        # enum Q8Kernel
KN, NK = False, True
MOST_SLICES = 64          # as many as any rule asks for

PROBE = """
#include <math.h>
#include <algorithm>
static long estimates = 0;
static double counting_sqrt(double x) { ++estimates; return sqrt(x); }
#define sqrt counting_sqrt                      // plan_cost takes one square root
#include "gemm_plan.h"
using namespace minfer_attn;
static void tile_of(int tile, int* out) {
    const GemmTile& t = kGemmTiles[tile];
    out[0] = 32 * t.m16; out[1] = 32 * t.n16; out[2] = t.occ;
}
extern "C" void route(int64_t M, int64_t N, int64_t K, int nt, int fast, int64_t fit, int* out) {
    const GemmRoute r = gemm_route(M, N, K, nt, fast, fit, []() { return 256; });
    out[0] = (int)r.kernel; out[1] = r.slices;
    tile_of(r.tile, out + 2);
}
extern "C" void q8(int64_t M, int64_t N, int64_t K, int aligned, int64_t fit, int* out) {
    const Q8Route r = q8_route(M, N, K, aligned, fit);
    out[0] = (int)r.kernel; out[1] = r.slices;
}
extern "C" int64_t q8_rows_of_a_part(int64_t M, int64_t N, int64_t K, int aligned) { return q8_part_rows(M, N, K, aligned); }
extern "C" void grouped(int64_t M, int64_t N, int64_t K, int* out) { tile_of(tile_plan(M, N, K, true, 1, 256).tile, out); }
extern "C" int stripe_blocks_ahead(int64_t M, int64_t N, int64_t K) { return stripe_blocks_pay(M, (N + 63) / 64, K); }
extern "C" int q8_blocks_ahead(int64_t M, int64_t N, int64_t K) { return q8_blocks_pay(M, N, K); }
extern "C" int meet(int64_t M) { return slices_meet(M); }
extern "C" int meet_rows() { return kMeetRows; }
extern "C" int meet_tiles() { return kMeetTiles; }
extern "C" long estimates_made() { return estimates; }
"""


class GemmPlan:
    """plan(M, N, K, nt, fit): (kernel, K slices, tile rows, tile columns, workgroups of it to a unit) of an aligned call whose workspace
    holds `fit` slices; the last three are those of the tiled kernel's calls."""

    def __init__(self, folder):
        src, so = os.path.join(folder, "probe.cpp"), os.path.join(folder, "probe.so")
        with open(src, "w") as f:
            f.write(PROBE)
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(capi.ROOT, "minfer-python_amd", "csrc"), src, "-o", so], check=True)
        L = ctypes.CDLL(so)
        i64, ints = ctypes.c_int64, ctypes.POINTER(ctypes.c_int)
        L.route.argtypes = [i64, i64, i64, ctypes.c_int, ctypes.c_int, i64, ints]
        L.q8.argtypes = [i64, i64, i64, ctypes.c_int, i64, ints]
        L.q8_rows_of_a_part.argtypes, L.q8_rows_of_a_part.restype = [i64, i64, i64, ctypes.c_int], i64
        L.grouped.argtypes = [i64, i64, i64, ints]
        L.stripe_blocks_ahead.argtypes = L.q8_blocks_ahead.argtypes = [i64, i64, i64]
        L.meet.argtypes = [i64]
        L.estimates_made.restype = ctypes.c_long
        self.lib = L
        self.estimates = L.estimates_made
        self.q8_part_rows = L.q8_rows_of_a_part
        self.slices_meet, self.meet_rows, self.meet_tiles = L.meet, L.meet_rows(), L.meet_tiles()
        self.stripe_blocks_pay, self.q8_blocks_pay = L.stripe_blocks_ahead, L.q8_blocks_ahead

    def __call__(self, M, N, K, nt, fit, fast=True):
        out = (ctypes.c_int * 5)()
        self.lib.route(M, N, K, int(nt), int(fast), fit, out)
        return tuple(out)

    def q8(self, M, N, K, aligned, fit):
        out = (ctypes.c_int * 2)()
        self.lib.q8(M, N, K, int(aligned), fit, out)
        return tuple(out)

    def grouped_tile(self, M, N, K):
        out = (ctypes.c_int * 3)()
        self.lib.grouped(M, N, K, out)
        return tuple(out)
