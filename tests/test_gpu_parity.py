"""GPU parity tests (-m gpu): the HIP kernels, called through the C ABI of libminfer_attn.so (and
through the registered torch ops), against the CPU oracle on identical seeded inputs.

Tolerances are the ones the task fixes: max-abs error <= 2e-3 for fp16 and <= 1e-2 for bf16 against
an fp32-or-better reference.  Masking and the GQA head mapping are checked for exact equality.
At the full benchmark sizes the oracle is evaluated on a sample of query rows (it is a scalar CPU
program) and the whole output is additionally compared with a plain fp32 torch evaluation of the
same formula on the GPU.
"""
import ctypes
import math

import numpy as np
import pytest
import torch

import capi
import oracle
import workloads

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = {torch.float16: 2e-3, torch.bfloat16: 1e-2}


# ------------------------------------------------------------------------------------------------
def torch_ref(q, k, v, mask, row_chunk=1024):
    """softmax(q k^T / sqrt(D) | mask) v in fp32 on the GPU, a chunk of query rows at a time."""
    B, Hq, L, D = q.shape
    n_rep = Hq // k.shape[1]
    kf = k.float().repeat_interleave(n_rep, 1).transpose(-1, -2).contiguous()
    vf = v.float().repeat_interleave(n_rep, 1).contiguous()
    out = torch.empty(B, Hq, L, D, dtype=torch.float32, device=q.device)
    for lo in range(0, L, row_chunk):
        hi = min(lo + row_chunk, L)
        s = (q[:, :, lo:hi].float() @ kf) / math.sqrt(D)
        s.masked_fill_(~mask[:, :, lo:hi], float("-inf"))
        p = torch.nan_to_num(torch.softmax(s, -1), nan=0.0)
        out[:, :, lo:hi] = p @ vf
    return out


def run_prefill(q, k, v, mask, out=None):
    if out is None:
        out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=q.device)
    rc = capi.flash_attn(q, k, v, mask, out)
    assert rc == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    return out


def max_err(a, b):
    return float((torch.as_tensor(a).float().cpu() - torch.as_tensor(b).float().cpu()).abs().max())


def make_mask(kind, B, L, gen):
    i = torch.arange(L)
    if kind == "causal":
        m = (i[None, :] <= i[:, None])[None].expand(B, L, L)
    elif kind == "window":
        m = ((i[None, :] - i[:, None]).abs() < 37)[None].expand(B, L, L)
    elif kind == "full":
        m = torch.ones(B, L, L, dtype=torch.bool)
    elif kind == "random":       # different per batch element, with rows that attend nothing
        m = torch.rand(B, L, L, generator=gen) < 0.5
        m[:, L // 3, :] = False
    elif kind == "blocky":       # whole 64x64 tiles switched off, to exercise tile skipping with holes
        t = (L + 63) // 64
        tiles = torch.rand(B, t, t, generator=gen) < 0.5
        tiles[:, :, 0] = True
        m = tiles.repeat_interleave(64, 1).repeat_interleave(64, 2)[:, :L, :L]
    return m[:, None].contiguous()


# ------------------------------------------------------------------------------------------------
# golden vectors (pin: torch SDPA on the reference's call, see tests/golden/make_golden.py)
# ------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("name", ["dense_causal_b1_h4_kv2_l16_d64", "dense_window_b2_h6_kv2_l40_d128",
                                  "dense_random_b1_h8_kv1_l70_d64"])
def test_golden_dense(name):
    z = np.load(f"{capi.ROOT}/tests/golden/{name}.npz")
    q, k, v = (torch.from_numpy(z[n]).to(DEV) for n in ("q", "k", "v"))
    out = run_prefill(q, k, v, torch.from_numpy(z["mask"]).to(DEV))
    assert max_err(out, z["out"]) <= TOL[torch.float16]


def test_golden_decode_and_varlen():
    z = np.load(f"{capi.ROOT}/tests/golden/decode_b3_h8_kv2_l50_d128.npz")
    q, k, v = (torch.from_numpy(z[n]).to(DEV) for n in ("q", "k", "v"))
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV)
    assert capi.flash_attn_decode(q, k, v, torch.from_numpy(z["ctx"]).to(DEV), out) == capi.OK, capi.last_error()
    assert max_err(out, z["out"]) <= TOL[torch.float16]
    z = np.load(f"{capi.ROOT}/tests/golden/varlen_h4_kv2_d64.npz")
    q, k, v = (torch.from_numpy(z[n]).to(DEV) for n in ("q", "k", "v"))
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV)
    assert capi.flash_attn_varlen(q, k, v, torch.from_numpy(z["cu"]).to(DEV), 70, out) == capi.OK, capi.last_error()
    assert max_err(out, z["out"]) <= TOL[torch.float16]


# ------------------------------------------------------------------------------------------------
# dense prefill against the oracle: shapes, masks, dtypes, layouts
# ------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,Hq,Hkv,L,D,kind,views", [
    (1, 8, 2, 256, 64, "causal", False),     # benchmark configuration 1 shape
    (2, 8, 2, 320, 128, "causal", True),     # reference-style transposed views
    (2, 6, 2, 200, 128, "window", False),    # n_rep = 3, symmetric window (reference test case B)
    (2, 4, 4, 333, 128, "random", False),    # L % 4 != 0: mask rows at any byte, per-batch masks
    (1, 16, 2, 520, 64, "random", True),     # n_rep = 8
    (1, 12, 2, 136, 128, "blocky", False),   # n_rep = 6
    (1, 16, 1, 264, 128, "causal", False),   # n_rep = 16
    (1, 2, 2, 1, 128, "full", False),        # single token
    (1, 4, 2, 63, 64, "causal", False),
    (3, 4, 1, 65, 128, "full", False),
    (1, 4, 1, 1040, 128, "blocky", False),
    # above 1024 rows the pre-pass classifies the mask (few workgroups: two teams of four waves; eight waves are in the next test)
    (1, 6, 2, 1093, 128, "random", False),   # n_rep = 3
    (1, 8, 1, 1100, 64, "window", True),     # n_rep = 8, D = 64, transposed views
    (2, 4, 4, 1029, 128, "causal", False),   # n_rep = 1, a last tile of 5 rows
])
def test_dense_matches_oracle(dtype, B, Hq, Hkv, L, D, kind, views):
    gen = torch.Generator().manual_seed(1000 * L + D + Hq)
    q, k, v = workloads.dense_prefill(B, Hq, Hkv, L, D, dtype, seed=L + Hq, scale=0.5, views=views, device=DEV)
    q = q * 2 if dtype == torch.float16 else q   # fp16: logits with a wider spread
    mask = make_mask(kind, B, L, gen)
    out = run_prefill(q, k, v, mask.to(DEV))
    want = oracle.flash_attn(q, k, v, mask)
    assert not torch.isnan(out).any()
    assert max_err(out, want) <= TOL[dtype]


@pytest.mark.parametrize("kind", ["random", "full"])
@pytest.mark.parametrize("L", [2, 3, 4, 5, 66, 67, 127, 129])
def test_dense_mask_rows_end_inside_a_word(L, kind):
    """Mask rows whose last key tile ends one to four bytes into a word, and rows shorter than one word: the tile's words come from
    the row's end, shifted, and keys past it count for nothing, in mixed tiles and in tiles that every row attends."""
    q, k, v = workloads.dense_prefill(2, 4, 2, L, 128, torch.float16, seed=L, scale=0.5, device=DEV)
    mask = make_mask(kind, 2, L, torch.Generator().manual_seed(L))
    out = run_prefill(q, k, v, mask.to(DEV))
    assert max_err(out, oracle.flash_attn(q, k, v, mask)) <= TOL[torch.float16]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,Hq,Hkv,L,kind", [
    (3, 32, 8, 1093, "random"),    # n_rep = 4: 64 rows per workgroup, a last key tile of 5 rows
    (3, 32, 4, 1100, "window"),    # n_rep = 8: 32 rows
    (20, 4, 4, 1029, "causal"),    # n_rep = 1: 256 rows
    (13, 6, 2, 1111, "blocky"),    # n_rep = 3: 256 rows, key tiles that no row attends
])
def test_dense_eight_waves(dtype, B, Hq, Hkv, L, kind):
    """More than 384 workgroups of eight waves over more than 1024 rows, which is what takes them, at ragged sizes: every element
    against the fp32 evaluation on the GPU."""
    gen = torch.Generator().manual_seed(L)
    q, k, v = workloads.dense_prefill(B, Hq, Hkv, L, 128, dtype, seed=L, scale=0.5, device=DEV)
    mask = make_mask(kind, B, L, gen).to(DEV)
    out = run_prefill(q, k, v, mask)
    assert max_err(out, torch_ref(q, k, v, mask)) <= TOL[dtype]


@pytest.mark.parametrize("Hq,Hkv,Lmax,D", [
    (8, 2, 200, 128),     # one chunk: the workgroup's result is the output
    (4, 4, 257, 64),      # a second chunk of one row
    (40, 2, 1030, 128),   # 20 heads per KV head: two head groups; several chunks
    (8, 1, 16400, 64),    # as many chunks as a head's merge holds
    (64, 8, 3000, 128),   # 6 sequences: every unit has a chunk
])
def test_decode_chunks(Hq, Hkv, Lmax, D):
    """Decode problems small enough to be cut into one chunk of rows per workgroup, at contexts around a wave's, a group's and a
    chunk's edges: against the oracle, the same again on two streams at once (the arrival counters are the stream's own and
    end as they began), and bit-equal under graph capture, where a second launch merges.  Tolerance: that of every fp16
    attention result here."""
    edges = [0, 1, 16, 17, Lmax // 2 + 1, Lmax]
    q, kc, vc, _ = workloads.decode_cache(seed=Lmax, device=DEV, B=len(edges), Hq=Hq, Hkv=Hkv, Lmax=Lmax, D=D, ctx_lo=1, ctx_hi=1)
    ctx = torch.tensor(edges, dtype=torch.int32, device=DEV)
    streams = [torch.cuda.current_stream(), torch.cuda.Stream()]
    outs = [torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV) for _ in range(6)]
    torch.cuda.synchronize()
    for i, out in enumerate(outs):
        with torch.cuda.stream(streams[i % 2]):
            assert capi.flash_attn_decode(q, kc, vc, ctx, out) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert max_err(outs[0], oracle.flash_attn_decode(q, kc, vc, ctx)) <= TOL[torch.float16]
    assert all(torch.equal(o, outs[0]) for o in outs)
    out, ws = torch.empty_like(outs[0]), torch.empty(capi.lib().minfer_flash_attn_decode_workspace_bytes(len(edges), Hq, Lmax, D), dtype=torch.uint8, device=DEV)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert capi.flash_attn_decode(q, kc, vc, ctx, out, ws) == capi.OK, capi.last_error()
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, outs[0])


@pytest.mark.parametrize("Hq,Hkv,L,D,kind", [
    (32, 8, 1100, 64, "causal"),     # 280 workgroups of eight (batch, KV head) groups: each XCD's ids folded by themselves
    (32, 8, 1100, 128, "random"),
    (6, 2, 5600, 64, "causal"),      # 264 workgroups of six groups: all ids folded together
    (32, 8, 1100, 64, "blocky"),
    (36, 9, 930, 64, "causal"),      # 270, classified in the kernel
])
def test_dense_workgroups_in_folded_order(Hq, Hkv, L, D, kind):
    """Launches of more workgroups than units, all on the chip at once, take the second ones in the opposite order: every row is still
    computed, and as in a batch of copies too many for that, bit for bit."""
    q, k, v = workloads.dense_prefill(1, Hq, Hkv, L, D, torch.float16, seed=L, device=DEV)
    mask = make_mask(kind, 1, L, torch.Generator().manual_seed(L))
    out, outs = torch.full_like(q, float("nan")), torch.full((4, *q.shape[1:]), float("nan"), dtype=q.dtype, device=DEV)
    assert capi.flash_attn(q, k, v, mask.to(DEV), out) == capi.OK, capi.last_error()
    copies = [t.expand(4, *t.shape[1:]).contiguous() for t in (q, k, v, mask.to(DEV))]
    assert capi.flash_attn(*copies, outs) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert not torch.isnan(out).any()
    assert all(torch.equal(out[0], o) for o in outs)


@pytest.mark.parametrize("q8", [False, True])
@pytest.mark.parametrize("B,Hq,Hkv,Lmax,D", [
    (2, 4, 2, 40007, 64),      # four pairs of many pieces
    (12, 20, 1, 9001, 128),    # two head groups
    (40, 8, 8, 1101, 64),      # 320 pairs
    (64, 8, 8, 300, 128),      # 512 pairs, one or a few pieces each: as many as are taken
    (33, 4, 4, 2050, 128),
])
def test_decode_pieces(B, Hq, Hkv, Lmax, D, q8):
    """Pairs cut into pieces of their own: contexts from nothing to the capacity, around a group's and a piece's edges, against the
    oracle.  Tolerance: that of every fp16 attention result here."""
    lens = [Lmax, 0, 1, 16, 33, 127, 129, Lmax - 1, Lmax // 2 + 1, 257]
    q, kc, vc, _ = workloads.decode_cache(seed=B + Lmax, device=DEV, B=B, Hq=Hq, Hkv=Hkv, Lmax=Lmax, D=D, ctx_lo=1, ctx_hi=1)
    ctx = torch.tensor([lens[i % len(lens)] for i in range(B)], dtype=torch.int32, device=DEV)
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV)
    if q8:
        kc, vc = workloads.q8_0_rows(kc), workloads.q8_0_rows(vc)
        assert capi.flash_attn_decode_q8_0(q, kc, vc, ctx, out) == capi.OK, capi.last_error()
        want = oracle.flash_attn_decode_q8_0(q.cpu(), kc.cpu(), vc.cpu(), ctx.cpu())
    else:
        assert capi.flash_attn_decode(q, kc, vc, ctx, out) == capi.OK, capi.last_error()
        want = oracle.flash_attn_decode(q, kc, vc, ctx)
    torch.cuda.synchronize()
    assert max_err(out, want) <= TOL[torch.float16]


def test_merged_parts_on_every_kind_of_stream(monkeypatch):
    """The null stream, the per-thread one (handle 2) and a created one: whether a launch's last workgroups or a second launch
    merge the parts of a decode and add up the K slices of a projection, the bits are the same."""
    q, kc, vc, ctx = workloads.decode_cache(seed=3, device=DEV, B=2, Hq=8, Hkv=2, Lmax=3000, D=128, ctx_lo=2000, ctx_hi=3000)
    x, w = torch.randn(3, 4096, device=DEV).half(), torch.randn(4096, 1024, device=DEV).half()
    ws = torch.empty(capi.lib().minfer_gemm_workspace_bytes(3, 1024, 4096), dtype=torch.uint8, device=DEV)
    created = torch.cuda.Stream()
    got = []
    for handle in (0, 2, created.cuda_stream, 0):
        monkeypatch.setattr(capi, "_stream", lambda: ctypes.c_void_p(handle))
        out, y = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV), torch.full((3, 1024), float("nan"), dtype=q.dtype, device=DEV)
        torch.cuda.synchronize()
        assert capi.flash_attn_decode(q, kc, vc, ctx, out) == capi.OK, capi.last_error()
        assert capi.gemm_ws(x, w, None, y, 1.0, 0.0, ws) == capi.OK, capi.last_error()
        torch.cuda.synchronize()
        got.append((out, y))
    assert not any(torch.isnan(t).any() for t in got[0])
    assert all(torch.equal(a, b) for g in got[1:] for a, b in zip(g, got[0]))


@pytest.mark.parametrize("Hq,Hkv,Lmax,D,q8", [
    (8, 2, 200, 128, False),      # one chunk, merged by its workgroup
    (8, 2, 190, 64, True),
    (8, 2, 3000, 64, False),      # chunks merged by the last workgroup, a whole one without a number among them
    (8, 2, 3000, 128, True),
    (40, 40, 1700, 64, False),    # the line of equal shares
])
def test_decode_keeps_nan(Hq, Hkv, Lmax, D, q8):
    """A query row with a NaN, a KV head whose keys are all NaN and one whose first half of keys is: the rows that attend them
    are NaN throughout, and no other row changes by a bit.  The same from the merge of a second launch (under graph capture)."""
    n_rep = Hq // Hkv
    q, kc, vc, _ = workloads.decode_cache(seed=Lmax, device=DEV, B=4, Hq=Hq, Hkv=Hkv, Lmax=Lmax, D=D, ctx_lo=1, ctx_hi=1)
    ctx = torch.tensor([Lmax, Lmax, Lmax, Lmax - 7], dtype=torch.int32, device=DEV)
    call = capi.flash_attn_decode
    if q8:
        kc, vc, call = workloads.q8_0_rows(kc), workloads.q8_0_rows(vc), capi.flash_attn_decode_q8_0
    clean, out, replayed = (torch.zeros(q.shape, dtype=q.dtype, device=DEV) for _ in range(3))
    assert call(q, kc, vc, ctx, clean) == capi.OK, capi.last_error()
    assert not torch.isnan(clean).any()
    q[0, 1, 0, D // 3] = float("nan")
    nan_keys = kc[1, Hkv - 1], kc[2, 0, :Lmax // 2]
    for rows in nan_keys:
        (rows.view(-1, 34)[:, :2].view(torch.float16) if q8 else rows).fill_(float("nan"))   # (Q8_0: the blocks' scales)
    want_nan = torch.zeros(q.shape, dtype=torch.bool, device=DEV)
    want_nan[0, 1] = want_nan[1, (Hkv - 1) * n_rep:] = want_nan[2, :n_rep] = True
    assert call(q, kc, vc, ctx, out) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    ws = torch.empty(capi.lib().minfer_flash_attn_decode_workspace_bytes(4, Hq, Lmax, D), dtype=torch.uint8, device=DEV)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert call(q, kc, vc, ctx, replayed, ws) == capi.OK, capi.last_error()
    graph.replay()
    torch.cuda.synchronize()
    for o in (out, replayed):
        assert torch.equal(torch.isnan(o), want_nan), [(torch.isnan(o) != want_nan)[b].flatten(1).any(1).nonzero().flatten().tolist() for b in range(4)]
        assert torch.equal(o[~want_nan], clean[~want_nan])


@pytest.mark.parametrize("B,Hq,Hkv,Lmax,D,q8", [
    (33, 16, 8, 1536, 64, False),    # a workgroup per context, one round and a bit
    (33, 16, 16, 300, 64, False),    # more than two rounds
    (33, 16, 8, 890, 128, False),
    (60, 8, 8, 1500, 128, False),    # two rounds that come out full
    (33, 16, 8, 512, 128, True),
    (33, 16, 8, 760, 64, True),
    (33, 16, 8, 1537, 64, False),    # past those limits: the line of equal shares
    (40, 16, 8, 1101, 128, True),    # ... its shares between 128 and 256 rows
    (40, 16, 8, 1101, 128, False),
])
def test_decode_more_contexts_than_units(B, Hq, Hkv, Lmax, D, q8):
    """Contexts from nothing to the capacity, around a group's and a wave's edges, against the oracle.  Tolerance: that of every
    fp16 attention result here."""
    lens = [Lmax, 0, 1, 16, 31, 33, 127, 129, 255, 257, Lmax - 1, Lmax // 2 + 1]
    q, kc, vc, _ = workloads.decode_cache(seed=B + Lmax, device=DEV, B=B, Hq=Hq, Hkv=Hkv, Lmax=Lmax, D=D, ctx_lo=1, ctx_hi=1)
    ctx = torch.tensor([lens[i % len(lens)] for i in range(B)], dtype=torch.int32, device=DEV)
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV)
    if q8:
        kc, vc = workloads.q8_0_rows(kc), workloads.q8_0_rows(vc)
        assert capi.flash_attn_decode_q8_0(q, kc, vc, ctx, out) == capi.OK, capi.last_error()
        want = oracle.flash_attn_decode_q8_0(q.cpu(), kc.cpu(), vc.cpu(), ctx.cpu())
    else:
        assert capi.flash_attn_decode(q, kc, vc, ctx, out) == capi.OK, capi.last_error()
        want = oracle.flash_attn_decode(q, kc, vc, ctx)
    assert max_err(out, want) <= TOL[torch.float16]


def test_decode_with_the_partial_results_of_coarse_shares():
    """A workspace that holds the partial results of 256-row shares and no more, one byte less, and the allocation-free call on
    a problem whose finer shares its scratch does not hold.  Against the oracle."""
    B, Hq, Hkv, Lmax, D = 64, 64, 1, 5000, 128
    q, kc, vc, _ = workloads.decode_cache(seed=1, device=DEV, B=B, Hq=Hq, Hkv=Hkv, Lmax=Lmax, D=D, ctx_lo=1, ctx_hi=1)
    ctx = torch.tensor([[5000, 1, 300, 2047][i % 4] for i in range(B)], dtype=torch.int32, device=DEV)
    up = lambda n: (n + 255) // 256 * 256
    need = up(B * Hq * (Lmax // 256 + 3) * (D + 2) * 4) + up((B + 1) * 4) + 256
    assert need < 64 << 20 < capi.lib().minfer_flash_attn_decode_workspace_bytes(B, Hq, Lmax, D)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    out, out2 = (torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV) for _ in range(2))
    assert capi.flash_attn_decode(q, kc, vc, ctx, out, ws[:-1]) == capi.EWORKSPACE
    assert capi.flash_attn_decode(q, kc, vc, ctx, out, ws) == capi.OK, capi.last_error()
    assert capi.flash_attn_decode_noalloc(q, kc, vc, ctx, out2) == capi.OK, capi.last_error()
    some = [0, 1, 2, 3, 61, 62]
    want = oracle.flash_attn_decode(q[some], kc[some], vc[some], ctx[some])
    for o in (out, out2):
        assert not torch.isnan(o).any() and max_err(o[some], want) <= TOL[torch.float16]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,Hq,Hkv,L,D,kind", [
    (1, 8, 2, 512, 128, "causal"),     # the shortest; the workgroups classify their own rows
    (1, 3, 3, 640, 64, "random"),
    (2, 4, 4, 1000, 128, "window"),
    (1, 4, 1, 1025, 64, "random"),     # the pre-pass's classes; a last key tile of one row
    (1, 6, 2, 1111, 128, "causal"),
    (1, 2, 2, 1500, 128, "empty"),     # rows, whole tiles and one of the two teams without a key
])
def test_prefill_two_teams(B, Hq, Hkv, L, D, kind, dtype):
    """Few workgroups, whose two teams of waves take every other key tile, against the oracle.  Tolerance: that of every
    attention result here."""
    gen = torch.Generator().manual_seed(L)
    q, k, v = workloads.dense_prefill(B, Hq, Hkv, L, D, dtype, seed=L, scale=1.0, device=DEV)
    if kind == "empty":
        mask = torch.zeros(B, 1, L, L, dtype=torch.bool)
        mask[:, :, 64:128, 70:75] = True       # one tile of the list
        mask[:, :, 200:320, 64:192] = True     # two
        mask[:, :, 1400:, ::130] = True
    else:
        mask = workloads.causal_mask(B, L) if kind == "causal" else workloads.window_mask(B, L, 200) if kind == "window" else make_mask("random", B, L, gen)
    out = run_prefill(q, k, v, mask.to(DEV))
    assert max_err(out, oracle.flash_attn(q, k, v, mask)) <= TOL[dtype]


@pytest.mark.parametrize("Hq,Hkv,D,lens", [
    (8, 2, 128, [1, 0, 65, 700, 64, 513]),
    (4, 4, 64, [2100, 129, 33]),
])
def test_packed_two_teams(Hq, Hkv, D, lens):
    gen = torch.Generator().manual_seed(sum(lens))
    q, k, v = (torch.randn(1, H, sum(lens), D, generator=gen).half() for H in (Hq, Hkv, Hkv))
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32)
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV)
    assert capi.flash_attn_varlen(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), max(lens), out) == capi.OK, capi.last_error()
    assert max_err(out, oracle.flash_attn_varlen(q, k, v, cu)) <= TOL[torch.float16]


@pytest.mark.parametrize("D,lens", [(128, [100] * 12), (64, [90, 0, 70, 100, 33] * 5), (128, [513, 0, 700, 65])])
def test_packed_with_no_bound_of_the_lengths(D, lens):
    """max_seqlen 0 (not known), or one that says no more than the number of tokens does, does not make a batch of short sequences
    one for the kernel of two teams, whose sums meet in another order, nor keep a batch of long ones from it: the same bits as
    with the bound."""
    gen = torch.Generator().manual_seed(sum(lens))
    q, k, v = (torch.randn(1, H, sum(lens), D, generator=gen).half().to(DEV) for H in (8, 2, 2))
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device=DEV)
    outs = [torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV) for _ in range(3)]
    for bound, out in zip((max(lens), 0, sum(lens) + 1), outs):
        assert capi.flash_attn_varlen(q, k, v, cu, bound, out) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert max_err(outs[0], oracle.flash_attn_varlen(q.cpu(), k.cpu(), v.cpu(), cu.cpu())) <= TOL[torch.float16]
    assert torch.equal(outs[1], outs[0]) and torch.equal(outs[2], outs[0])


@pytest.mark.parametrize("offset", [0, 5])
@pytest.mark.parametrize("B,L,D", [(2, 1, 64), (3, 2, 128), (2, 3, 64), (2, 4, 128), (2, 5, 64), (2, 15, 128), (2, 16, 64), (3, 17, 128),
                                   (2, 63, 64), (2, 65, 128), (1, 129, 128), (2, 255, 64), (1, 1023, 64), (1, 1025, 128), (1, 1103, 64)])
def test_mask_rows_at_any_byte(B, L, D, offset):
    """Rows of the mask start at any byte (L odd, base address odd) and end inside a 16-column piece or a 4-column word; the
    bytes around the mask are True, so a column read past a row's end would show.  Self-classifying workgroups up to 1024
    rows, the pre-pass above.  Tolerance: the one every fp16 attention result here has."""
    gen = torch.Generator().manual_seed(L)
    q, k, v = workloads.dense_prefill(B, 4, 2, L, D, torch.float16, seed=L, scale=1.0, device=DEV)
    mask = make_mask("random", B, L, gen)
    buf = torch.ones(B * L * L + offset + 64, dtype=torch.bool, device=DEV)
    m = buf[offset:offset + B * L * L].view(B, 1, L, L)
    m.copy_(mask)
    out = run_prefill(q, k, v, m)
    assert max_err(out, oracle.flash_attn(q, k, v, mask)) <= TOL[torch.float16]


@pytest.mark.parametrize("B,Hq,Hkv,L,D,kind", [
    (1, 4, 4, 16, 128, "random"),      # n_rep = 1: four query blocks per workgroup, of which one has rows
    (2, 4, 2, 48, 64, "full"),         # n_rep = 2
    (1, 6, 2, 208, 128, "window"),     # n_rep = 3
    (2, 8, 2, 320, 128, "blocky"),     # n_rep = 4, key tiles that no row of a query block attends
    (1, 16, 2, 512, 64, "random"),     # n_rep = 8: two head groups
    (1, 16, 1, 1008, 128, "blocky"),   # n_rep = 16, a last key tile of 48 columns
    (1, 8, 2, 1024, 128, "random"),    # the longest mask whose rows one wave-wide load covers
    (3, 32, 8, 512, 128, "blocky"),    # more workgroups than fit on the chip at once: the pre-pass classifies
])
def test_short_dense_masks_classified_inside_the_kernel(B, Hq, Hkv, L, D, kind):
    """A short dense problem launches no classification pre-pass: each workgroup classifies its own mask rows.  Checked against
    the oracle, bit for bit against the same call with the mask at an odd address and, up to 511 rows (from there on few
    workgroups take two teams), bit for bit against a batch of copies, too many for the chip, which takes the pre-pass."""
    dtype = torch.float16
    gen = torch.Generator().manual_seed(77 * L + Hq)
    q, k, v = workloads.dense_prefill(B, Hq, Hkv, L, D, dtype, seed=L + Hq + 1, scale=0.5, device=DEV)
    mask = make_mask(kind, B, L, gen)
    md = mask.to(DEV)
    out = run_prefill(q, k, v, md)
    assert not torch.isnan(out).any()
    assert max_err(out, oracle.flash_attn(q, k, v, mask)) <= TOL[dtype]
    shifted = torch.zeros(md.numel() + 1, dtype=torch.bool, device=DEV)[1:].view(md.shape)
    shifted.copy_(md)
    assert shifted.data_ptr() % 16 == 1
    assert torch.equal(run_prefill(q, k, v, shifted), out)
    if L < 512:
        n = 512 // (B * Hkv) + 1                 # a workgroup per (batch entry, KV head) at least
        many = run_prefill(*(t.repeat(n, 1, 1, 1) for t in (q, k, v, md)))
        assert torch.equal(many.view(n, *out.shape), out.expand(n, *out.shape))


def test_cpu_plumbing_config_on_gpu():
    """benchmark configuration 1 (fp32 N(0,1) inputs, S=256, D=64): the same seeded inputs rounded to fp16."""
    q, k, v, mask = workloads.cpu_plumbing(seed=0)
    want = oracle.flash_attn(q.half(), k.half(), v.half(), mask)
    out = run_prefill(q.half().to(DEV), k.half().to(DEV), v.half().to(DEV), mask.to(DEV))
    assert out.shape == (1, 8, 256, 64)
    assert max_err(out, want) <= TOL[torch.float16]


def test_strided_out_and_determinism():
    B, Hq, Hkv, L, D = 2, 8, 2, 192, 128
    q, k, v = workloads.dense_prefill(B, Hq, Hkv, L, D, torch.float16, seed=5, views=True, device=DEV)
    mask = workloads.causal_mask(B, L, device=DEV)
    a = run_prefill(q, k, v, mask)
    out_t = torch.full((B, L, Hq, D), float("nan"), dtype=torch.float16, device=DEV).transpose(1, 2)
    b = run_prefill(q, k, v, mask, out=out_t)
    assert torch.equal(a, b)
    assert torch.equal(a, run_prefill(q, k, v, mask))
    assert max_err(a, oracle.flash_attn(q, k, v, mask)) <= TOL[torch.float16]


# ------------------------------------------------------------------------------------------------
# exact properties: masking and GQA mapping are bit-identical
# ------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_masking_and_gqa_mapping_exact(dtype):
    B, Hq, Hkv, L, D = 2, 8, 2, 200, 128
    gen = torch.Generator().manual_seed(9)
    q, k, v = workloads.dense_prefill(B, Hq, Hkv, L, D, dtype, seed=9, scale=1.0, device=DEV)
    n_rep = Hq // Hkv
    # one attended key per row: the output row is that V row, bit for bit
    sel = torch.randint(0, L, (B, L), generator=gen)
    onehot = torch.zeros(B, L, L, dtype=torch.bool)
    onehot.scatter_(2, sel[:, :, None], True)
    out = run_prefill(q, k, v, onehot[:, None].contiguous().to(DEV))
    for b in range(B):
        for h in range(Hq):
            assert torch.equal(out[b, h], v[b, h // n_rep, sel[b].to(DEV)])
    # causal: row 0 is V row 0
    out = run_prefill(q, k, v, workloads.causal_mask(B, L, device=DEV))
    for h in range(Hq):
        assert torch.equal(out[:, h, 0], v[:, h // n_rep, 0])
    # V constant per KV head: every row of query head h equals the constant of KV head h // n_rep
    vc = torch.empty_like(v)
    for g in range(Hkv):
        vc[:, g] = float(g + 1)
    out = run_prefill(q, k, vc, workloads.causal_mask(B, L, device=DEV))
    for h in range(Hq):
        assert torch.equal(out[:, h], torch.full_like(out[:, h], float(h // n_rep + 1)))
    # rows that attend nothing give zeros, their neighbours are unaffected
    m = workloads.causal_mask(B, L)
    m[:, :, 70, :] = False
    out2 = run_prefill(q, k, v, m.to(DEV))
    assert torch.all(out2[:, :, 70] == 0)
    ref = run_prefill(q, k, v, workloads.causal_mask(B, L, device=DEV))
    keep = torch.arange(L) != 70
    assert torch.equal(out2[:, :, keep], ref[:, :, keep])


# ------------------------------------------------------------------------------------------------
# the benchmark configurations at full size
# ------------------------------------------------------------------------------------------------
def sample_rows(L, n, gen):
    fixed = [0, 1, 31, 32, 63, 64, 65, L // 2, L - 65, L - 2, L - 1]
    extra = torch.randint(0, L, (n,), generator=gen).tolist()
    return sorted(set(r for r in fixed + extra if 0 <= r < L))


@pytest.mark.parametrize("views", [False, True])
def test_llama8b_prefill_full(views):
    """benchmark configuration 2: B=1, Hq=32, Hkv=8, S=4096, D=128, fp16, causal, 0.5*N(0,1)."""
    q, k, v, mask = workloads.llama8b_prefill(seed=0, device=DEV, views=views)
    out = run_prefill(q, k, v, mask)
    assert max_err(out, torch_ref(q, k, v, mask)) <= TOL[torch.float16]
    rows = sample_rows(4096, 150, torch.Generator().manual_seed(1))
    want = oracle.flash_attn_rows(q, k, v, mask[:, 0, rows].cpu(), rows)
    assert max_err(out[:, :, rows], want) <= TOL[torch.float16]
    assert torch.equal(out[0, :, 0], v[0].repeat_interleave(4, 0)[:, 0])


def test_long_context_prefill_full():
    """benchmark configuration 4: B=1, Hq=32, Hkv=8, S=32768, D=128, bf16, causal, 0.5*N(0,1)."""
    L = 32768
    q, k, v, mask = workloads.long_context_prefill(seed=0, device=DEV, L=L)
    out = run_prefill(q, k, v, mask)
    rows = sample_rows(L, 40, torch.Generator().manual_seed(2))
    want = oracle.flash_attn_rows(q, k, v, mask[:, 0, rows].cpu(), rows)
    assert max_err(out[:, :, rows], want) <= TOL[torch.bfloat16]
    assert torch.equal(out[0, :, 0], v[0].repeat_interleave(4, 0)[:, 0])
    assert max_err(out, torch_ref(q, k, v, mask, row_chunk=512)) <= TOL[torch.bfloat16]


def test_decode_full():
    """benchmark configuration 3: B=64, Hq=32, Hkv=8, D=128, fp16, ctx in [512, 8192], cache [B,Hkv,8192,128]."""
    q, kc, vc, ctx = workloads.decode_cache(seed=0, device=DEV)
    # rows beyond ctx are garbage that must not reach the result
    for b in range(0, 64, 7):
        kc[b, :, int(ctx[b]):] = float("nan")
        vc[b, :, int(ctx[b]):] = float("inf")
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV)
    assert capi.flash_attn_decode(q, kc, vc, ctx, out) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert not torch.isnan(out).any()
    want = oracle.flash_attn_decode(q, kc, vc, ctx)
    assert max_err(out, want) <= TOL[torch.float16]


def test_ragged_prefill_full():
    """benchmark configuration 5: 16 sequences, lengths in [128, 2048], Hq=64, Hkv=8, D=128, fp16, N(0,1)."""
    q, k, v, cu = workloads.ragged_prefill(seed=0, device=DEV)
    lens = (cu[1:] - cu[:-1]).tolist()
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV)
    assert capi.flash_attn_varlen(q, k, v, cu, max(lens), out) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert not torch.isnan(out).any()
    worst, lo = 0.0, 0
    for n in lens:
        m = workloads.causal_mask(1, n, device=DEV)
        worst = max(worst, max_err(out[:, :, lo:lo + n], torch_ref(q[:, :, lo:lo + n], k[:, :, lo:lo + n], v[:, :, lo:lo + n], m)))
        lo += n
    assert worst <= TOL[torch.float16]
    # the shortest sequence in full against the oracle
    s = int(np.argmin(lens))
    lo, hi = int(cu[s]), int(cu[s + 1])
    want = oracle.flash_attn(q[:, :, lo:hi], k[:, :, lo:hi], v[:, :, lo:hi], workloads.causal_mask(1, hi - lo))
    assert max_err(out[:, :, lo:hi], want) <= TOL[torch.float16]


# ------------------------------------------------------------------------------------------------
# decode and varlen edge cases against the oracle
# ------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,Hq,Hkv,Lmax,D,lo,hi", [
    (2, 8, 2, 256, 128, 1, 256),
    (5, 8, 2, 1000, 64, 0, 1000),      # ctx = 0 allowed, Lmax not a multiple of 16
    (2, 40, 2, 700, 128, 500, 700),    # n_rep = 20: two head groups
    (3, 6, 6, 1537, 128, 1537, 1537),  # ctx = Lmax, n_rep = 1, 4 chunks with a 1-row tail
    (4, 4, 1, 17, 64, 1, 17),
    (3, 8, 2, 0, 128, 0, 0),           # an empty cache: zeros, with the workspace size the library reports for it
])
def test_decode_matches_oracle(dtype, B, Hq, Hkv, Lmax, D, lo, hi):
    scale = 1.0 if dtype == torch.float16 else 0.5
    q, kc, vc, ctx = workloads.decode_cache(seed=Lmax, device="cpu", B=B, Hq=Hq, Hkv=Hkv, Lmax=Lmax, D=D, dtype=dtype,
                                            ctx_lo=lo, ctx_hi=hi)
    vc = (vc.float() * scale).to(dtype)
    out = torch.full(q.shape, float("nan"), dtype=dtype, device=DEV)
    assert capi.flash_attn_decode(q.to(DEV), kc.to(DEV), vc.to(DEV), ctx.to(DEV), out) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert max_err(out, oracle.flash_attn_decode(q, kc, vc, ctx)) <= TOL[dtype]
    assert torch.all(out[ctx.to(DEV) == 0] == 0)


@pytest.mark.parametrize("B,Hq,Hkv,Lmax,D,ctx", [
    (200, 8, 2, 64, 64, "tiny"),          # shares of the work span many short sequences, some empty; B > 64
    (1, 4, 1, 40000, 128, "full"),        # one (sequence, KV head) cut into ~57 shares: as many partials per row
    (70, 40, 2, 1000, 128, "gaps"),       # empty sequences at both ends and in between, two head groups
    (3, 16, 16, 5000, 64, "full"),
])
def test_decode_work_is_shared_out_evenly_whatever_the_lengths(B, Hq, Hkv, Lmax, D, ctx):
    g = torch.Generator().manual_seed(B + Lmax)
    q = torch.randn(B, Hq, 1, D, generator=g).half()
    kc = torch.randn(B, Hkv, Lmax, D, generator=g).half()
    vc = torch.randn(B, Hkv, Lmax, D, generator=g).half()
    if ctx == "tiny":
        lens = torch.randint(0, 41, (B,), generator=g, dtype=torch.int32)
    elif ctx == "full":
        lens = torch.full((B,), Lmax, dtype=torch.int32)
    else:
        lens = torch.randint(1, Lmax + 1, (B,), generator=g, dtype=torch.int32)
        lens[:3] = 0
        lens[-2:] = 0
        lens[10:40:7] = 0
    out = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV)
    assert capi.flash_attn_decode(q.to(DEV), kc.to(DEV), vc.to(DEV), lens.to(DEV), out) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert max_err(out, oracle.flash_attn_decode(q, kc, vc, lens)) <= TOL[torch.float16]
    assert torch.all(out[lens.to(DEV) == 0] == 0)
    # the same caches as Q8_0 blocks
    kq, vq = torch.from_numpy(oracle.quant_q8_0(kc.float())), torch.from_numpy(oracle.quant_q8_0(vc.float()))
    out8 = torch.full(q.shape, float("nan"), dtype=q.dtype, device=DEV)
    assert capi.flash_attn_decode_q8_0(q.to(DEV), kq.to(DEV), vq.to(DEV), lens.to(DEV), out8) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert max_err(out8, oracle.flash_attn_decode_q8_0(q, kq, vq, lens)) <= TOL[torch.float16]
    assert torch.all(out8[lens.to(DEV) == 0] == 0)


def test_decode_equals_last_prefill_row():
    """Splitting the KV range and merging by log-sum-exp must not change the result: the decode of
    position ctx-1 equals the last row of a causal prefill over the same ctx rows."""
    B, Hq, Hkv, Lmax, D = 1, 8, 2, 2048, 128
    q, k, v = workloads.dense_prefill(B, Hq, Hkv, Lmax, D, torch.float16, seed=21, device=DEV)
    pre = run_prefill(q, k, v, workloads.causal_mask(B, Lmax, device=DEV))
    for ctx_len in (1, 511, 512, 513, 2048):
        out = torch.empty(B, Hq, 1, D, dtype=torch.float16, device=DEV)
        ctx = torch.tensor([ctx_len], dtype=torch.int32, device=DEV)
        assert capi.flash_attn_decode(q[:, :, ctx_len - 1:ctx_len].contiguous(), k, v, ctx, out) == capi.OK
        assert max_err(out[:, :, 0], pre[:, :, ctx_len - 1]) <= 1e-3


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Hq,Hkv,D,lens", [
    (8, 2, 128, [5, 64, 100, 1, 257]),
    (8, 1, 64, [130, 31, 0, 77]),
    (6, 2, 128, [1, 1, 1]),
    (4, 4, 64, [300]),
    (8, 2, 128, [(7 * i) % 41 for i in range(150)]),      # more sequences than a wave has lanes, some empty
    (8, 2, 64, [700, 333, 0, 20, 64, 1]),
])
def test_varlen_matches_oracle_and_dense(dtype, Hq, Hkv, D, lens):
    g = torch.Generator().manual_seed(sum(lens))
    T = sum(lens)
    q = torch.randn(1, Hq, T, D, generator=g).to(dtype)
    k = torch.randn(1, Hkv, T, D, generator=g).to(dtype)
    v = (0.5 * torch.randn(1, Hkv, T, D, generator=g)).to(dtype)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    out = torch.full(q.shape, float("nan"), dtype=dtype, device=DEV)
    assert capi.flash_attn_varlen(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), max(lens), out) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert max_err(out, oracle.flash_attn_varlen(q, k, v, cu)) <= TOL[dtype]
    # max_seqlen sizes the launch and chooses the kernel (0, or one past T: not known): the same bits either way
    out0 = torch.full(q.shape, float("nan"), dtype=dtype, device=DEV)
    assert capi.flash_attn_varlen(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), 0, out0) == capi.OK, capi.last_error()
    out_big = torch.full(q.shape, float("nan"), dtype=dtype, device=DEV)
    assert capi.flash_attn_varlen(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), 5000, out_big) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert torch.equal(out0, out) and torch.equal(out_big, out)
    # same result as the reference-signature op under the block-diagonal causal mask
    blk = torch.zeros(T, T, dtype=torch.bool)
    for lo, hi in zip(cu[:-1].tolist(), cu[1:].tolist()):
        blk[lo:hi, lo:hi] = torch.ones(hi - lo, hi - lo, dtype=torch.bool).tril()
    dense = run_prefill(q.to(DEV), k.to(DEV), v.to(DEV), blk[None, None].contiguous().to(DEV))
    # (two bf16 results may round an element above 1 to neighbouring values, 2^-7 apart)
    one_ulp = float(dense.float().abs().max()) * 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    assert max_err(out, dense) <= TOL[dtype] / 2 + one_ulp


def test_varlen_malformed_cu_seqlens_stay_in_bounds():
    """cu_seqlens lives on the device and is never checked by the host: a decreasing entry, a negative one and one
    past T must not move any access outside q/k/v/out.  The tensors are views with guard rows on both sides of every
    head (NaN in q/k/v, which would poison any result that read them; a sentinel in out); sequences that are valid
    and overlap no other come out as the oracle computes them."""
    Hq, Hkv, D, T, G = 8, 2, 128, 600, 96
    g = torch.Generator().manual_seed(77)

    def guarded(H, fill, scale=1.0):
        buf = torch.full((1, H, T + 2 * G, D), fill, dtype=torch.float16)
        buf[:, :, G:G + T] = (scale * torch.randn(1, H, T, D, generator=g)).to(torch.float16)
        buf = buf.to(DEV)
        return buf, buf[:, :, G:G + T]

    qb, q = guarded(Hq, float("nan"))
    kb, k = guarded(Hkv, float("nan"))
    vb, v = guarded(Hkv, float("nan"), 0.5)
    ob = torch.full((1, Hq, T + 2 * G, D), 7.0, dtype=torch.float16, device=DEV)
    out = ob[:, :, G:G + T]
    # sequence 0 = rows [0,200); 1 ends before it starts (empty); 2 = [150,400) overlaps the end of 0; 3 starts at 400
    # and claims rows far past T (cut to [400,600)); 4 starts past T (empty); 5 has a negative start and end (empty)
    cu = torch.tensor([0, 200, 150, 400, 2_000_000_000, -5, -3], dtype=torch.int32, device=DEV)
    assert capi.flash_attn_varlen(q, k, v, cu, 0, out) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert torch.all(ob[:, :, :G] == 7.0) and torch.all(ob[:, :, G + T:] == 7.0)     # guard rows of out untouched
    assert not torch.isnan(out).any()                                                 # no guard row of q/k/v was read
    qc, kc, vc = q.cpu(), k.cpu(), v.cpu()
    for lo, hi, rows in [(0, 200, slice(0, 150)), (150, 400, slice(50, 250)), (400, 600, slice(0, 200))]:
        want = oracle.flash_attn(qc[:, :, lo:hi], kc[:, :, lo:hi], vc[:, :, lo:hi], workloads.causal_mask(1, hi - lo))
        assert max_err(out[:, :, lo:hi][:, :, rows], want[:, :, rows]) <= TOL[torch.float16]
    # the same with max_seqlen given: rows of a sequence past it are left alone, the others are as before
    ob.fill_(7.0)
    assert capi.flash_attn_varlen(q, k, v, cu, 100, out) == capi.OK, capi.last_error()
    torch.cuda.synchronize()
    assert torch.all(ob[:, :, :G] == 7.0) and torch.all(ob[:, :, G + T:] == 7.0)
    assert torch.all(out[:, :, 500:] == 7.0)                                          # rows 100.. of the last sequence
    want = oracle.flash_attn(qc[:, :, 400:500], kc[:, :, 400:500], vc[:, :, 400:500], workloads.causal_mask(1, 100))
    assert max_err(out[:, :, 400:500], want) <= TOL[torch.float16]


# ------------------------------------------------------------------------------------------------
# the registered torch ops (the reference's call path) give the same bits and the same errors
# ------------------------------------------------------------------------------------------------
def test_torch_ops_match_c_abi(kerns):
    from minfer.const import GGML_QUANT_SIZES, GGMLQuantizationType
    qt = GGMLQuantizationType.F16
    qb, qs = GGML_QUANT_SIZES[qt]
    B, Hq, Hkv, L, D = 2, 12, 2, 300, 128
    q, k, v = workloads.dense_prefill(B, Hq, Hkv, L, D, torch.float16, seed=31, views=True, device=DEV)
    mask = workloads.window_mask(B, L, 100, device=DEV)
    a = torch.zeros(B, Hq, L, D, dtype=torch.float16, device=DEV)
    kerns.flash_attn(qt, qb, qs, q, k, v, mask, a)           # reference call shape: test/kernels.py:246-248
    torch.cuda.synchronize()
    assert torch.equal(a, run_prefill(q, k, v, mask))

    qd, kc, vc, ctx = workloads.decode_cache(seed=3, device=DEV, B=4, Lmax=1024, ctx_lo=1, ctx_hi=1024)
    a = torch.zeros_like(qd)
    kerns.flash_attn_decode(qt, qb, qs, qd, kc, vc, ctx, a)
    b = torch.zeros_like(qd)
    assert capi.flash_attn_decode(qd, kc, vc, ctx, b) == capi.OK
    torch.cuda.synchronize()
    assert torch.equal(a, b)

    qv, kv, vv, cu = workloads.ragged_prefill(seed=3, device=DEV, n_seqs=4, len_lo=1, len_hi=200, Hq=8, Hkv=2)
    a = torch.zeros_like(qv)
    kerns.flash_attn_varlen(qt, qb, qs, qv, kv, vv, cu, 200, a)
    b = torch.zeros_like(qv)
    assert capi.flash_attn_varlen(qv, kv, vv, cu, 200, b) == capi.OK
    torch.cuda.synchronize()
    assert torch.equal(a, b)


def test_torch_op_validation(kerns):
    """The checks of the reference host function (flash_attn/op.cuh:32-96) raise RuntimeError."""
    B, Hq, Hkv, L, D = 1, 4, 2, 64, 128
    q, k, v = workloads.dense_prefill(B, Hq, Hkv, L, D, torch.float16, seed=1, device=DEV)
    mask = workloads.causal_mask(B, L, device=DEV)
    out = torch.empty_like(q)
    args = lambda **kw: [1, 1, 2] + [kw.get(n, d) for n, d in (("q", q), ("k", k), ("v", v), ("mask", mask), ("out", out))]
    with pytest.raises(RuntimeError):
        kerns.flash_attn(*args(q=q.float()))                                   # dtype
    with pytest.raises(RuntimeError):
        kerns.flash_attn(*args(mask=mask.to(torch.uint8)))                     # mask dtype
    with pytest.raises(RuntimeError):
        kerns.flash_attn(*args(mask=mask.expand(B, 1, L, L).transpose(2, 3)))  # mask not contiguous
    with pytest.raises(RuntimeError):
        kerns.flash_attn(*args(q=q[..., ::2].repeat_interleave(2, -1)[..., ::1].transpose(2, 3).transpose(2, 3)[:, :, :, :64]))  # head_dim 64 vs k 128
    with pytest.raises(RuntimeError):
        kerns.flash_attn(*args(k=k[:, :, :32]))                                # Lk != Lq
    with pytest.raises(RuntimeError):
        kerns.flash_attn(*args(out=out[0]))                                    # rank
    with pytest.raises(RuntimeError):
        kerns.flash_attn(*args(v=v.transpose(1, 2).contiguous().transpose(1, 2)))  # k/v strides differ
    with pytest.raises(RuntimeError):
        kerns.flash_attn(*args(mask=mask.cpu()))                               # device
    kerns.flash_attn(*args())                                                  # and the good call passes
    torch.cuda.synchronize()
