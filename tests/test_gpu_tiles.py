"""The tiled fp6 kernel (rq_gemm6.hip) by itself, at shapes that the router still sends to whole tiles and to K slices (most small
products go in units of 64 rows x 64 tokens now), and the tiles that it leaves over to the units in both of its tile orders. Every
case says which of them it means and asks the plan; outputs are pre-filled, and a few tokens of each token tile are compared bit
for bit with the oracle."""
import numpy as np
import pytest
import torch

import ruquant_amd as rq
from ruquant_amd import synth
from tests.gpu_util import bits_equal, first_mismatch
from tests.plan_util import plan

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def weights(N, K, seed, multipliers):
    """random codes; the first three rows all -8, all 7 and both in turn by groups of 64, with multipliers of 15 where there are
    any (1 .. 15 per 64 inputs elsewhere)"""
    blocks = synth.random_weight_blocks(N, K, seed, rq.TYPE_W4A4)
    qs = blocks["qs"].reshape(N, K // 8)
    qs[0], qs[1] = 0x88888888, 0x77777777
    qs[2] = np.where((np.arange(K // 8) // 8) % 2 == 0, 0x88888888, 0x77777777)
    blocks["qs"] = qs.reshape(blocks["qs"].shape)
    if multipliers:
        k = np.random.default_rng(seed).integers(1, 16, size=(N, K // 256, 4), dtype=np.uint32)
        k[:3] = 15
        head = (np.uint32(3 << 29) | k[..., 0] | k[..., 1] << 4 | k[..., 2] << 8 | k[..., 3] << 12).astype(np.uint32)
        blocks["sum"] = head.view(np.int32)
    else:
        blocks["sum"] = synth.signed_code_sums(qs).astype(np.int32)[:, None]
    return blocks


def tokens(M, K, seed):
    """rows of +1, -1 and both (q - z = +-15 with m = 255 in every group), then ordinary ones"""
    x = synth.activations("outlier_channels", M, K, seed)
    x[0], x[1] = 1.0, -1.0
    x[2] = np.where((np.arange(K) // 64) % 2 == 0, 1.0, -1.0)
    x[M - 1] = 0.5
    return x


def check(oracle, bl, ws, x, sample, workspace=None, repeats=2):
    M = x.shape[0]
    xd = torch.from_numpy(x).to(DEV)
    if workspace is None:
        workspace = rq.fused_workspace_bytes(ws, M)
    work = torch.full((workspace,), 0xA5, dtype=torch.uint8, device=DEV)
    want = [oracle.mul_mat(w.type, b, x[sample], w.clip) for b, w in zip(bl, ws)]
    for _ in range(repeats):   # the second call meets the arrival counters that the first one left
        outs = [torch.full((M, w.N + 3 * i + 1), float("nan"), dtype=torch.float32, device=DEV) for i, w in enumerate(ws)]
        views = [o[:, :w.N] for o, w in zip(outs, ws)]
        if len(ws) == 1:
            rq.mul_mat(ws[0], xd, out=views[0], workspace=work)
        else:
            rq.mul_mat_fused(ws, xd, outs=views, workspace=work)
        torch.cuda.synchronize()
        for o, w, v in zip(outs, ws, want):
            assert not torch.isnan(o[:, :w.N]).any() and torch.isnan(o[:, w.N:]).all()
            got = o[:, :w.N][sample].cpu().numpy()
            assert bits_equal(got, v), first_mismatch(got, v)


def sample_of(M):
    return sorted(t for t in {0, 1, 2, 63, 64, 65, M // 2, M - 2, M - 1} | set(range(100, M, 128)) if t < M)


@pytest.mark.parametrize("multipliers", [0, 1])
@pytest.mark.parametrize("K,N,M,whole,cut,slices", [
    (4352, 17000, 100, 0, 67, 3),      # 34 steps in slices of 11 and 12 (an odd count in some), ragged rows and tokens
    (4352, 4500, 2300, 256, 68, 3),    # the same behind a round of whole tiles
    (5120, 17100, 65, 0, 67, 3),       # one token in the tile's second half
    (5120, 17100, 128, 0, 67, 3),      # a full tile of tokens
    (5120, 8300, 256, 0, 66, 3),       # two, in turn
    (2560, 9300, 330, 0, 111, 2),
    (32768, 256, 1536, 0, 12, 13),     # the longest row: 19 and 20 steps, the float totals at 3.9 M of the 4.19 M of their window
    (1024, 8192, 1000, 256, 0, 1),     # a round of whole tiles in super-tiles, nothing left over
    (256, 4300, 700, 102, 0, 1),      # fewer steps (2) than stages of the ring
    (512, 4300, 700, 102, 0, 1),      # as many
    (768, 4300, 700, 102, 0, 1)],     # a step and a half of them
    ids=lambda v: str(v))
def test_whole_tiles_and_slices(oracle, K, N, M, whole, cut, slices, multipliers):
    p = plan(rq.TYPE_W4A4, K, N, M, multipliers)
    assert (p["launches"], p["whole"], p["cut"], p["slices"], p["units"]) == (1, whole, cut, slices, 0)
    b = weights(N, K, N + M, multipliers)
    check(oracle, [b], [rq.W4A4Weight(b, rq.TYPE_W4A4, DEV, keep_blocks=False)], tokens(M, K, M), sample_of(M))


@pytest.mark.parametrize("multipliers", [0, 1])
def test_without_slabs_every_tile_runs_whole(oracle, multipliers):
    K, N, M = 2560, 17100, 100
    assert plan(rq.TYPE_W4A4, K, N, M, multipliers)["cut"] == 67
    p = plan(rq.TYPE_W4A4, K, N, M, multipliers, slabs=False)
    assert (p["whole"], p["cut"], p["units"]) == (67, 0, 0)
    b = weights(N, K, 8, multipliers)
    w = rq.W4A4Weight(b, rq.TYPE_W4A4, DEV, keep_blocks=False)
    check(oracle, [b], [w], tokens(M, K, 4), sample_of(M), workspace=rq.fused_workspace_bytes([w], M) - 256)


@pytest.mark.parametrize("K,Ns,M,multipliers,known,cut,slices,launches", [
    (2560, (2300, 1000, 2800), 500, (0, 0, 0), True, 96, 2, 1),       # 9 + 4 + 11 row tiles in super-tiles over weights
    (2560, (2300, 1000, 2800), 500, (1, 1, 1), True, 96, 2, 1),
    (2560, (9000, 8400), 100, (1, 1), True, 69, 3, 1),                # two weights: the third slot selects nothing
    (2560, (9000, 4000, 4400), 100, (1, 1, 0), False, 70, 3, 1),      # copies planned as weights without multipliers
    (5120, (17100, 17408), 100, (1, 0), True, 67 + 68, 3, 2)],        # known to be of both kinds: a launch each
    ids=["super_tiles", "super_tiles_multipliers", "two_weights", "unknown_addresses", "both_kinds"])
def test_slices_of_sets(oracle, K, Ns, M, multipliers, known, cut, slices, launches):
    p = plan(rq.TYPE_W4A4, K, Ns, M, sum(m << i for i, m in enumerate(multipliers)) if known else 0)
    assert (p["launches"], p["whole"], p["cut"], p["slices"], p["units"]) == (launches, 0, cut, slices, 0)
    bl = [weights(N, K, 60 + i, m) for i, (N, m) in enumerate(zip(Ns, multipliers))]
    ws = [rq.W4A4Weight(b, rq.TYPE_W4A4, DEV, keep_blocks=False) for b in bl]
    if not known:
        for w in ws:
            copy = torch.empty(w.prepared.numel() + 4096, dtype=torch.uint8, device=DEV)[2048:2048 + w.prepared.numel()]
            copy.copy_(w.prepared)
            w.prepared = copy
    check(oracle, bl, ws, tokens(M, K, M), sample_of(M))


@pytest.mark.parametrize("K,Ns,M,multipliers,whole,units", [
    (1024, (6100,), 1500, 0, 256, 256),               # 24 x 12 tiles: a whole super-tile is left over
    (1024, (6100,), 1500, 1, 256, 256),
    (1024, (3000, 1400, 1536), 1500, 0, 256, 256),    # the same over weights, whose row tiles end inside super-tiles
    (512, (4300,), 2048, 0, 256, 128),                # 17 x 16: token tiles running fastest, the last row tile ragged
    (512, (8192,), 1100, 1, 256, 256)],               # 32 x 9
    ids=lambda v: str(v))
def test_tiles_left_over_to_the_units(oracle, K, Ns, M, multipliers, whole, units):
    """The units count through the left-over tiles in the tiled kernel's order: all of y is written, by one of the two."""
    p = plan(rq.TYPE_W4A4, K, Ns, M, 7 * multipliers)
    assert (p["launches"], p["whole"], p["cut"], p["units"]) == (1, whole, 0, units)
    bl = [weights(N, K, 40 + i, multipliers) for i, N in enumerate(Ns)]
    ws = [rq.W4A4Weight(b, rq.TYPE_W4A4, DEV, keep_blocks=False) for b in bl]
    check(oracle, bl, ws, tokens(M, K, M), sample_of(M), repeats=1)


def test_without_slabs_long_rows_go_in_units(oracle):
    K, N, M = 32768, 200, 100
    assert plan(rq.TYPE_W4A4, K, N, M)["cut"] == 1 and plan(rq.TYPE_W4A4, K, N, M, slabs=False)["units"] == 8
    b = weights(N, K, 8, 0)
    w = rq.W4A4Weight(b, rq.TYPE_W4A4, DEV, keep_blocks=False)
    check(oracle, [b], [w], tokens(M, K, 4), sample_of(M), workspace=rq.fused_workspace_bytes([w], M) - 256)


@pytest.mark.parametrize("N,M,units", [(8300, 40, 130), (8300, 64, 130), (6200, 64, 0)])
def test_static_workspace_at_33_to_64_tokens(oracle, N, M, units):
    """rq_w4a4_mul_mat_static from 129 panels up (units) and below (the skinny kernel), the two in turn on the one array."""
    K, type_ = 2560, rq.TYPE_W4A4
    assert plan(type_, K, N, M)["units"] == units
    b = weights(N, K, N, 0)
    w = rq.W4A4Weight(b, type_, DEV, keep_blocks=False)
    x = tokens(M, K, M)
    xd = torch.from_numpy(x).to(DEV)
    L = rq.load_library()
    want = oracle.mul_mat(type_, b, x, w.clip)
    for m in (M, 20, M):
        y = torch.full((m, N), float("nan"), dtype=torch.float32, device=DEV)
        rc = L.rq_w4a4_mul_mat_static(type_, w.prepared.data_ptr(), K, N, xd.data_ptr(), K, m, y.data_ptr(), N, w.clip, 0,
                                      torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        torch.cuda.synchronize()
        if m == M:
            got = y.cpu().numpy()
            assert bits_equal(got, want), first_mismatch(got, want)


@pytest.mark.parametrize("N,M", [(16449, 33), (16384, 64), (17408, 64)])
def test_filling_calls_keep_the_skinny_kernel(oracle, N, M):
    """More panels than compute units at 33 to 64 tokens, through the calls after which other weights may use the activations:
    whole panels and cut ones beside them, in a workspace full of rubbish, then a second weight on what the call left."""
    K, type_ = 1024, rq.TYPE_W4A4
    assert plan(type_, K, N, M)["units"] == (N + 63) // 64 and plan(type_, K, N, M, once=False)["units"] == 0
    L = rq.load_library()
    bl = [weights(N, K, 1, 0), weights(6000, K, 2, 1)]
    ws = [rq.W4A4Weight(b, type_, DEV, keep_blocks=False) for b in bl]
    x = tokens(M, K, M)
    xd = torch.from_numpy(x).to(DEV)
    work = torch.full((ws[0].workspace(M).numel(),), 0xA5, dtype=torch.uint8, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    for w, b, stages in ((ws[0], bl[0], 3), (ws[1], bl[1], 2), (ws[0], bl[0], 2)):
        y = torch.full((M, w.N), float("nan"), dtype=torch.float32, device=DEV)
        rc = L.rq_w4a4_mul_mat_stages(type_, w.prepared.data_ptr(), K, w.N, xd.data_ptr(), K, M, y.data_ptr(), w.N, w.clip, 0,
                                      work.data_ptr(), work.numel(), stream, stages)
        assert rc == 0
        torch.cuda.synchronize()
        want = oracle.mul_mat(type_, b, x, w.clip)
        got = y.cpu().numpy()
        assert bits_equal(got, want), first_mismatch(got, want)
