"""The fp6 product in units of 64 rows x 64 tokens (rq_block6.hip), bit for bit against the oracle: where a wavefront has no
group, a few or enough to move its totals to LDS on the way; ragged rows, tokens and row strides; every kind of weight
multiplier; one round of the chip, two, and the tiles that the tiled kernel leaves over; and 33 .. 64 tokens, which take it only
in calls that share their activation with no other."""
import numpy as np
import pytest
import torch

import ruquant_amd as rq
from ruquant_amd import synth
from tests.gpu_util import adversarial_weights, adversarial_activations, bits_equal, first_mismatch, run_gpu
from tests.plan_util import FP6, SKINNY, plan

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("K,N,M,wgroup,units", [
    (256, 64, 65, 0, 2),             # four groups for eight wavefronts
    (512, 1, 128, 64, 2),            # one group each, one row
    (4352, 130, 190, 0, 9),          # eight or nine, ragged
    (4352, 130, 190, 256, 9),
    (15360, 70, 66, 0, 4),           # 30: past the 28 between two transfers
    (32768, 65, 67, 64, 0),          # the longest row: by price one tile in slices
    (17408, 70, 67, 64, 4),          # 34, with multipliers
    (512, 4096, 512, 0, 512),        # 512 units: two rounds
    (512, 4300, 2048, 0, 128),       # 17 x 16 tiles: 16 left over behind a round, the last row tile ragged
    (512, 8192, 1100, 256, 256),     # 32 x 9 tiles: 32 left over, in runs of nine token tiles
    (2560, 6200, 33, 0, 0),          # 97 panels: the skinny kernel
    (2560, 6200, 64, 64, 0),
    (3072, 6200, 40, 64, 97),        # with multipliers there too
    (17408, 6145, 41, 0, 0),
    (2560, 8300, 33, 0, 130),        # 130 panels: 33 .. 64 tokens in units
    (2560, 8300, 64, 64, 130),
    (17408, 8257, 41, 0, 130),
    (512, 16500, 57, 0, 258),        # two rounds
    (10240, 4096, 64, 0, 64),        # units in four pieces: as many as that takes
    (1024, 70, 33, 0, 2),            # ... without rows, and with one token
    (1280, 2050, 70, 64, 66),        # one more: in two pieces, the last panel's second without rows
    (1280, 4070, 128, 0, 128),       # as many as that takes
    (512, 4100, 97, 256, 130),       # one more: whole
    (11264, 70, 40, 0, 0)])          # few panels of longer rows: the skinny kernel
def test_units_of_64_rows_and_tokens(oracle, K, N, M, wgroup, units):
    type_ = rq.TYPE_W4A4 if K in (256, 512, 32768) else rq.TYPE_W4A4H
    blocks, wf = adversarial_weights(oracle, N, K, type_, seed=N + M, wgroup=wgroup)
    W = rq.W4A4Weight(blocks, type_, DEV)
    assert plan(type_, K, N, M, wgroup != 0)["units"] == units
    x = adversarial_activations(M, K, type_, wf, seed=M)
    want = oracle.mul_mat(type_, blocks, x, W.clip, n_rot=max(W.n_rot, 0))
    got = run_gpu(W, x)
    assert bits_equal(got, want), first_mismatch(got, want)
    # rows of y that are no multiple of four floats apart, and nothing written between them
    out = torch.full((M, N + 3), -7.0, dtype=torch.float32, device=DEV)
    rq.mul_mat(W, torch.from_numpy(x).to(DEV), out=out[:, :N])
    got = out.cpu().numpy()
    assert bits_equal(got[:, :N], want), first_mismatch(got[:, :N], want)
    assert (got[:, N:] == -7.0).all()


@pytest.mark.parametrize("K", [17408, 32768])
def test_extreme_sums_between_two_transfers(oracle, K):
    """K = 17408, the longest row without multipliers that goes in units: 34 groups per wavefront, rows of all -8 / all 7 against
    tokens of q - z = +-15 with m = 255, so that the float totals move by 122,400 per group, 28 groups and a tile of one more
    between two transfers: 3.55 M of their 4.19 M. (The same at K = 32768 in K slices.)"""
    N, M, type_ = 64, 80, rq.TYPE_W4A4
    p = plan(type_, K, N, M)
    assert (p["units"], p["cut"]) == ((2, 0) if K == 17408 else (0, 1))
    blocks = synth.random_weight_blocks(N, K, 5, type_)
    qs = blocks["qs"].reshape(N, -1)
    qs[0, :] = 0x88888888
    qs[1, :] = 0x77777777
    qs[2, ::2] = 0x88888888
    qs[2, 1::2] = 0x77777777
    blocks["qs"] = qs.reshape(blocks["qs"].shape)
    x = np.ones((M, K), dtype=np.float32)
    x[1::2] = -1.0
    x[2::4, ::2] = -1.0
    W = rq.W4A4Weight(blocks, type_, DEV)
    want = oracle.mul_mat(type_, blocks, x, W.clip)
    got = run_gpu(W, x)
    assert bits_equal(got, want), first_mismatch(got, want)


def test_extreme_sums_with_weight_multipliers(oracle):
    """The longest row with a multiplier of 15 on every group: 64 groups per wavefront, whose terms of up to 1.836 M each are
    added as bit patterns, modulo 2^32, the bias of every one still on it. Rows of all -8 / all 7 / both in turn against tokens
    of q - z = +-15 with m = 255: totals of 117.5 M per wavefront and 940 M per output, both signs."""
    K, M, panels, type_ = 32768, 40, 129, rq.TYPE_W4A4
    assert plan(type_, K, 64 * panels, M, multipliers=1)["units"] == panels
    rng = np.random.default_rng(3)
    codes = rng.integers(-8, 8, size=(64, K), dtype=np.int8)
    codes[0] = -8
    codes[1] = 7
    codes[2] = np.where((np.arange(K) // 64) % 2 == 0, -8, 7)
    units = np.abs(rng.normal(0.02, 0.005, size=64)).astype(np.float32)
    mults = rng.integers(1, 16, size=(64, K // 64), dtype=np.int32)
    mults[:3] = 15
    panel = rq.pack_groups(codes, units, mults)
    W = rq.W4A4Weight(np.tile(panel, (panels, 1)), type_, DEV, keep_blocks=False)
    x = synth.activations("outlier_channels", M, K, 9)
    x[0] = 1.0
    x[1] = -1.0
    x[2] = np.where((np.arange(K) // 64) % 2 == 0, 1.0, -1.0)
    x[39] = 0.5
    want = oracle.mul_mat(type_, panel, x, W.clip)
    got = run_gpu(W, x).reshape(M, panels, 64)
    for p in (0, 1, 64, 128):
        assert bits_equal(got[:, p], want), first_mismatch(got[:, p], want)
    assert (got == got[:, :1]).all()
    unit = np.float32(1.0) / np.float32(3825.0)
    expect = (np.float32(-15 * 122400 * (K // 64)) * np.float32(16.0)) * unit * units[0]
    assert got[0, 0, 0] == np.float32(expect)


@pytest.mark.parametrize("M,Ns", [(40, (3000, 2100, 1500)), (70, (3000, 2100, 1500)), (40, (4000, 2100, 2500))],
                         ids=["skinny", "70_tokens", "40_tokens"])
def test_a_set_of_weights(oracle, M, Ns):
    """Three weights, with and without multipliers, whose panels do not end with a row tile, in one launch (40 tokens, 136
    panels) or one each (70, where the two kinds go apart); 104 panels at 40 tokens are the skinny kernel's."""
    K, type_ = 1024, rq.TYPE_W4A4H
    ws, want = [], []
    x = None
    p = plan(type_, K, Ns, M, multipliers=2)
    assert (p["kernel"], p["launches"]) == ((SKINNY, 1) if sum(Ns) == 6600 and M == 40 else (FP6, 1 if M == 40 else 3))
    assert p["whole"] == p["cut"] == 0
    for i, (N, g) in enumerate(zip(Ns, (0, 64, 0))):
        blocks, wf = adversarial_weights(oracle, N, K, type_, seed=i, wgroup=g)
        w = rq.W4A4Weight(blocks, type_, DEV)
        if x is None:
            x = adversarial_activations(M, K, type_, wf, seed=3)
        ws.append(w)
        want.append(oracle.mul_mat(type_, blocks, x, w.clip, n_rot=w.n_rot))
    outs = rq.mul_mat_fused(ws, torch.from_numpy(x).to(DEV))
    for o, v in zip(outs, want):
        assert bits_equal(o.cpu().numpy(), v), first_mismatch(o.cpu().numpy(), v)
