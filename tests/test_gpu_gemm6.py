"""Wide batches through the fp6 MFMA kernels, compared bit for bit with the oracle, by whichever of tiles, K slices and units the
router takes (test_gpu_tiles.py and test_gpu_block6.py mean one of them each); and the int8 MFMA kernel they replaced, which
RQ_GEMM_FP6=0 still selects, in a child process (the variable is read once per process)."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import ruquant_amd as rq
from ruquant_amd import synth
from tests.gpu_util import adversarial_weights, adversarial_activations, bits_equal, first_mismatch, run_gpu

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HERE = os.path.dirname(os.path.abspath(__file__))


def test_prepared_weight_carries_the_fp6_plane():
    L = rq.load_library()
    K, N = 5120, 1000
    compact = N * K // 2
    # padded to row tiles of 256: 1024 rows x 0.75 bytes per weight
    assert L.rq_w4a4_prepared_bytes(K, N) >= compact + 1024 * K * 3 // 4


@pytest.mark.parametrize("type_,wgroup", [(rq.TYPE_W4A4H, 0), (rq.TYPE_W4A4, 64), (rq.TYPE_W4A4, 256)],
                         ids=["w4a4h", "w4a4_wgroup64", "w4a4_wgroup256"])
def test_leftover_tiles_cut_along_k_uneven_slices(oracle, type_, wgroup):
    """8 row tiles x 33 token tiles = 264 tiles: 256 run whole, the last 8 (one row tile, eight token tiles) as 64 units.
    Ragged rows and tokens, with and without weight multipliers, K = 4352 = 68 x 64."""
    N, K, M = 2000, 4352, 4200
    blocks, wf = adversarial_weights(oracle, N, K, type_, wgroup=wgroup)
    W = rq.W4A4Weight(blocks, type_, DEV)
    x = adversarial_activations(M, K, type_, wf, seed=7)
    got = run_gpu(W, x)
    want = oracle.mul_mat(type_, blocks, x, W.clip, n_rot=max(W.n_rot, 0))
    assert bits_equal(got, want), first_mismatch(got, want)
    # twice
    got2 = run_gpu(W, x)
    assert bits_equal(got2, want), first_mismatch(got2, want)


def test_slices_longest_row_extreme_sums(oracle):
    """K = 32768 with every tile cut along K (1 row tile x 12 token tiles: 13 slices of 19 or 20 steps each), inputs
    that drive the sums to their ends: rows of all -8 / all +7 codes against tokens that quantize to q - z = +-15 with
    m = 255 in all 512 groups (without weight multipliers such rows do not go in units). Within a slice the biased fp32 accumulator moves by 122400 per group for 32 groups
    between two transfers to the int32 total (3.9 M of the 4.19 M its window allows), in both directions."""
    N, K, M, type_ = 256, 32768, 1536, rq.TYPE_W4A4
    blocks = synth.random_weight_blocks(N, K, 5, type_, clip=0.9)
    qs = blocks["qs"].reshape(N, -1)
    qs[0, :] = 0x88888888
    qs[1, :] = 0x77777777
    qs[2, ::2] = 0x88888888
    qs[2, 1::2] = 0x77777777
    blocks["qs"] = qs.reshape(blocks["qs"].shape)
    blocks["sum"] = synth.signed_code_sums(qs).astype(np.int32)[:, None]
    W = rq.W4A4Weight(blocks, type_, DEV)
    x = synth.activations("outlier_channels", M, K, 9)
    x[0, :] = 1.0
    x[1, :] = -1.0
    x[2, :] = np.where((np.arange(K) // 64) % 2 == 0, 1.0, -1.0)
    x[1535, :] = 0.5
    got = run_gpu(W, x)
    sample = [0, 1, 2, 3, 127, 128, 700, 1534, 1535]
    want = oracle.mul_mat(type_, blocks, x[sample], W.clip, n_rot=0)
    assert bits_equal(got[sample], want), first_mismatch(got[sample], want)
    clip = np.float32(0.9)
    unit = np.float32(np.float32(1.0) * clip) / np.float32(3825.0)
    expect = (np.float32(-122400 * 512) * np.float32(16.0)) * unit * blocks["d"][0, 0]
    assert got[0, 0] == np.float32(expect)


@pytest.mark.parametrize("per", [256, 64])
def test_weight_multipliers_extreme_sums(oracle, per):
    """The same extremes on a tensor with weight multipliers (rq.pack_groups, one per block or per 64 inputs): rows of
    all -8 / all +7 codes with multiplier 15 everywhere against q - z = +-15 with m = 255, both signs: 95 units, whose
    sums of bit patterns take 15 x 122400 = 1.836 M per group. (The tiled kernel, which transfers its float totals after
    every second group, has the same rows in test_gpu_tiles.py.)"""
    N, K, M, type_ = 300, 4352, 1200, rq.TYPE_W4A4
    rng = np.random.default_rng(17)
    codes = rng.integers(-8, 8, size=(N, K), dtype=np.int8)
    codes[0, :] = -8
    codes[1, :] = 7
    codes[2, :] = np.where((np.arange(K) // 64) % 2 == 0, -8, 7)
    units = np.abs(rng.normal(0.02, 0.005, size=N)).astype(np.float32)
    mults = rng.integers(1, 16, size=(N, K // per), dtype=np.int32)
    mults[0:3, :] = 15
    mults[5, :] = 1
    blocks = rq.pack_groups(codes, units, mults)
    W = rq.W4A4Weight(blocks, type_, DEV)
    x = synth.activations("outlier_channels", M, K, 9)
    x[0, :] = 1.0
    x[1, :] = -1.0
    x[2, :] = np.where((np.arange(K) // 64) % 2 == 0, 1.0, -1.0)
    got = run_gpu(W, x)
    sample = [0, 1, 2, 3, 127, 128, 640, 1199]
    want = oracle.mul_mat(type_, blocks, x[sample], W.clip, n_rot=0)
    assert bits_equal(got[sample], want), first_mismatch(got[sample], want)
    unit = np.float32(1.0) / np.float32(3825.0)
    expect = (np.float32(-15 * 122400 * (K // 64)) * np.float32(16.0)) * unit * units[0]
    assert got[0, 0] == np.float32(expect)


def test_weight_multipliers_at_an_address_the_library_has_not_seen(oracle):
    """The launcher picks the kernel for tensors with weight multipliers from what rq_w4a4_prepare saw. A copy of the
    prepared bytes at another address is unknown to it and takes the other kernel, which must give the same bits."""
    import ctypes
    import torch
    N, K, M, type_ = 520, 2560, 200, rq.TYPE_W4A4H
    blocks, wf = adversarial_weights(oracle, N, K, type_, wgroup=64)
    W = rq.W4A4Weight(blocks, type_, DEV)
    x_np = adversarial_activations(M, K, type_, wf)
    want = oracle.mul_mat(type_, blocks, x_np, W.clip, n_rot=K)
    assert bits_equal(run_gpu(W, x_np), want)
    L = rq.load_library()
    moved = torch.empty(W.prepared.numel() + 4096, dtype=torch.uint8, device=DEV)[2048:2048 + W.prepared.numel()]
    assert moved.data_ptr() % 256 == 0
    moved.copy_(W.prepared)
    x = torch.from_numpy(x_np).to(DEV)
    y = torch.full((M, N), float("nan"), dtype=torch.float32, device=DEV)
    ws = W.workspace(M)
    rc = L.rq_w4a4_mul_mat(type_, moved.data_ptr(), K, N, x.data_ptr(), K, M, y.data_ptr(), N, W.clip, K, ws.data_ptr(),
                           ws.numel(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert bits_equal(got, want), first_mismatch(got, want)


@pytest.mark.parametrize("in_place", [False, True], ids=["one_buffer", "plane_apart"])
@pytest.mark.parametrize("N,M", [(6200, 40), (8300, 40), (570, 200), (570, 1100), (300, 3)])
def test_a_moved_weight_needs_nothing_of_its_original(oracle, N, M, in_place):
    """Prepared bytes copied to another address, the original overwritten: every kernel that reads the fp6 plane (small
    units, tiles, K slices) or the int4 panels gives the same bits. (Of a weight prepared in place the plane is a buffer of
    its own, which the caller keeps.)"""
    K, type_ = 2560, rq.TYPE_W4A4
    blocks, wf = adversarial_weights(oracle, N, K, type_, seed=M)
    W = rq.W4A4Weight(blocks, type_, DEV, in_place=in_place)
    x = adversarial_activations(M, K, type_, wf, seed=M)
    want = oracle.mul_mat(type_, blocks, x, W.clip)
    original = W.prepared
    moved = torch.empty(original.numel() + 4096, dtype=torch.uint8, device=DEV)[2048:2048 + original.numel()]
    moved.copy_(original)
    original.fill_(0x5A)
    W.prepared = moved
    got = run_gpu(W, x)
    assert bits_equal(got, want), first_mismatch(got, want)


@pytest.mark.parametrize("M", [65, 128, 129, 300])
def test_token_counts_around_the_tile(oracle, M):
    """One and a few runs of 64 tokens, partly filled, K = 5120, few rows: units."""
    N, K, type_ = 520, 5120, rq.TYPE_W4A4H
    blocks, wf = adversarial_weights(oracle, N, K, type_)
    W = rq.W4A4Weight(blocks, type_, DEV)
    x = adversarial_activations(M, K, type_, wf, seed=M)
    got = run_gpu(W, x)
    want = oracle.mul_mat(type_, blocks, x, W.clip, n_rot=K)
    assert bits_equal(got, want), first_mismatch(got, want)


def test_workspace_without_slabs_runs_every_tile_whole(oracle):
    """A workspace that ends in front of the slabs of the K slices (what the static entry point has for wide batches)
    gives the same bits; these few rows go in units either way."""
    N, K, M, type_ = 520, 2560, 200, rq.TYPE_W4A4H
    blocks, wf = adversarial_weights(oracle, N, K, type_)
    W = rq.W4A4Weight(blocks, type_, DEV)
    x_np = adversarial_activations(M, K, type_, wf, seed=3)
    want = oracle.mul_mat(type_, blocks, x_np, W.clip, n_rot=K)
    L = rq.load_library()
    full = L.rq_w4a4_workspace_bytes(type_, K, N, M)
    slabs = 256 * 4 + 256 * 256 * 128 * 4
    assert full > slabs
    x = torch.from_numpy(x_np).to(DEV)
    for nbytes in (full, full - slabs + (1 << 20)):
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=DEV)
        y = torch.full((M, N), float("nan"), dtype=torch.float32, device=DEV)
        rc = L.rq_w4a4_mul_mat(type_, W.prepared.data_ptr(), K, N, x.data_ptr(), K, M, y.data_ptr(), N, W.clip, K,
                               ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, rc
        torch.cuda.synchronize()
        got = y.cpu().numpy()
        assert bits_equal(got, want), "%d bytes: %s" % (nbytes, first_mismatch(got, want))


def test_int8_gemm_under_rq_gemm_fp6_0():
    env = dict(os.environ)
    env["RQ_GEMM_FP6"] = "0"
    out = subprocess.run([sys.executable, "-u", os.path.join(HERE, "gemm_i8_case.py")], env=env, capture_output=True,
                         text=True, timeout=600)
    assert out.returncode == 0 and "ALL OK" in out.stdout, out.stdout[-3000:] + out.stderr[-2000:]


@pytest.mark.parametrize("wgroup", [0, 64], ids=["legacy", "wgroup64"])
@pytest.mark.parametrize("M,slabs", [(65, True), (200, True), (200, False), (4700, True)])
def test_several_weights_in_one_launch(oracle, M, slabs, wgroup):
    """Three weights of one kind whose row tiles (2 + 1 + 4, ragged) are counted through in one launch, rows too short to
    be cut along K: units at 65 and 200 tokens, a workspace without slabs, and a whole round with three tiles left over to the
    units (7 x 37 tiles). Outputs with row strides of their own; what lies beside them stays."""
    K, type_ = 512, rq.TYPE_W4A4
    ws, bl = [], []
    for i, N in enumerate([384, 98, 1000]):
        b, wf = adversarial_weights(oracle, N, K, type_, seed=30 + i, wgroup=wgroup)
        bl.append(b)
        ws.append(rq.W4A4Weight(b, type_, DEV))
    x = adversarial_activations(M, K, type_, wf, seed=M)
    xd = torch.from_numpy(x).to(DEV)
    outs = [torch.full((M, w.N + 3 * i), -7.0, dtype=torch.float32, device=DEV) for i, w in enumerate(ws)]
    # (without slabs: only the cells for 64 tokens' rows behind the activations, as for a call of the fewest bytes)
    nbytes = rq.fused_workspace_bytes(ws, M) - (0 if slabs else 30 << 20)
    work = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    for rep in range(2):   # the second call meets the counters the first one left
        rq.mul_mat_fused(ws, xd, outs=[o[:, :w.N] for o, w in zip(outs, ws)], workspace=work)
        torch.cuda.synchronize()
        for b, w, o in zip(bl, ws, outs):
            want = oracle.mul_mat(type_, b, x, w.clip)
            got = o.cpu().numpy()
            assert bits_equal(got[:, :w.N], want), first_mismatch(got[:, :w.N], want)
            assert (got[:, w.N:] == -7.0).all()


def _graph_nodes(call):
    """kernel launches of one call: nodes of the graph that captures it"""
    call()
    torch.cuda.synchronize()
    with open("/proc/self/maps") as f:   # (the copy that torch runs on)
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64.so" in line))
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g):
        call()
    n = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


@pytest.mark.parametrize("K,Ns,M,launches", [(17408, (4134, 2216), 525, 2), (17408, (10029, 6404), 234, 2),
                                             (17408, (8192, 16384), 256, 1), (5120, (4134, 2216), 525, 1),
                                             (5120, (6144, 1024, 1024), 512, 1)])
def test_one_launch_only_where_it_is_not_slower(K, Ns, M, launches):
    """Weights whose tiles can each be cut along K but not together (85 + 45 of 256, long rows) keep their own launches;
    either way the bits are those of the separate products."""
    type_ = rq.TYPE_W4A4
    ws = [rq.W4A4Weight(synth.random_weight_blocks(N, K, i, type_), type_, DEV) for i, N in enumerate(Ns)]
    x = torch.from_numpy(synth.activations("student_t4", M, K, 5)).to(DEV)
    outs = [torch.full((M, N), float("nan"), dtype=torch.float32, device=DEV) for N in Ns]
    work = torch.empty(rq.fused_workspace_bytes(ws, M), dtype=torch.uint8, device=DEV)
    assert _graph_nodes(lambda: rq.mul_mat_fused(ws, x, outs=outs, workspace=work)) == 1 + launches
    for w, o in zip(ws, outs):
        assert torch.equal(o, rq.mul_mat(w, x))


@pytest.mark.parametrize("K,M,Ns,wgroups,moved,launches", [
    (2560, 512, (500, 200, 1200), (0, 0, 0), False, 1),        # units over weights
    (512, 4096, (500, 200, 1200), (256, 256, 256), False, 1),  # 2 + 1 + 5 row tiles: super-tiles over weights, one whole round
    (2560, 200, (1000, 700), (64, 64), False, 1),              # two weights: the third slot selects nothing
    (2560, 200, (384, 98, 1000), (64, 0, 64), False, 3),       # with and without multipliers: a launch each
    (2560, 200, (384, 98, 1000), (64, 256, 0), True, 1)],      # copies the launcher knows nothing of: units read the flags
    ids=["units", "super_tiles_whole", "two_weights", "both_kinds", "unknown_addresses"])
def test_sets_of_weights(oracle, K, M, Ns, wgroups, moved, launches):
    """Sets in units and in whole super-tiles that straddle weights, against the oracle, with outputs of their own row
    strides (slices of sets: test_gpu_tiles.py)."""
    type_ = rq.TYPE_W4A4
    ws, bl = [], []
    for i, (N, g) in enumerate(zip(Ns, wgroups)):
        b, wf = adversarial_weights(oracle, N, K, type_, seed=60 + i, wgroup=g)
        w = rq.W4A4Weight(b, type_, DEV)
        if moved:
            copy = torch.empty(w.prepared.numel() + 4096, dtype=torch.uint8, device=DEV)[2048:2048 + w.prepared.numel()]
            copy.copy_(w.prepared)
            w.prepared = copy
        bl.append(b)
        ws.append(w)
    x = adversarial_activations(M, K, type_, wf, seed=M)
    xd = torch.from_numpy(x).to(DEV)
    outs = [torch.full((M, N + 3 * i), -7.0, dtype=torch.float32, device=DEV) for i, N in enumerate(Ns)]
    work = torch.full((rq.fused_workspace_bytes(ws, M),), 0xA5, dtype=torch.uint8, device=DEV)
    views = [o[:, :N] for o, N in zip(outs, Ns)]
    assert _graph_nodes(lambda: rq.mul_mat_fused(ws, xd, outs=views, workspace=work)) == 1 + launches
    for b, w, o in zip(bl, ws, outs):
        want = oracle.mul_mat(type_, b, x, w.clip)
        got = o.cpu().numpy()
        assert bits_equal(got[:, :w.N], want), first_mismatch(got[:, :w.N], want)
        assert (got[:, w.N:] == -7.0).all()
