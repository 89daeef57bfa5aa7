"""Which kernels a call runs (rq_w4a4_product_plan: the function that the entry points themselves ask), without a GPU."""
import ctypes

import pytest

import ruquant_amd as rq
from tests.plan_util import DECODE, FP6, GEMV, SKINNY, plan

W4A4, W4A4H = rq.TYPE_W4A4, rq.TYPE_W4A4H


@pytest.mark.parametrize("M,kernel", [(1, DECODE), (2, GEMV), (4, GEMV), (5, SKINNY), (32, SKINNY), (65, FP6), (2048, FP6)])
def test_kernel_by_token_count(M, kernel):
    p = plan(W4A4H, 5120, 5120, M)
    assert p["kernel"] == kernel and p["launches"] == 1


@pytest.mark.parametrize("K,N,multipliers,kernel", [
    (5120, 8192, 0, SKINNY), (5120, 8193, 0, FP6), (17408, 12288, 0, FP6), (18432, 12288, 0, SKINNY), (32768, 17408, 0, SKINNY),
    (5120, 17408, 0, FP6), (5376, 17408, 0, SKINNY), (10240, 17408, 0, SKINNY), (10240, 24576, 0, FP6), (10240, 34816, 0, SKINNY),
    (12288, 24576, 0, SKINNY), (17408, 17408, 0, SKINNY), (5120, 34816, 0, FP6),
    (1024, 8192, 1, SKINNY), (2816, 8192, 1, SKINNY), (3072, 6080, 1, SKINNY), (3072, 6081, 1, FP6), (10240, 8192, 1, FP6),
    (10496, 8192, 1, SKINNY), (10240, 8192, 0, SKINNY), (1024, 8256, 1, FP6), (32768, 12288, 1, FP6), (17408, 17408, 1, FP6), (32768, 17408, 1, SKINNY)])
@pytest.mark.parametrize("M", [33, 64])
def test_33_to_64_tokens(K, N, multipliers, kernel, M):
    """Units of the fp6 product only where they are no slower on weights that come from memory either (6 % at most)."""
    p = plan(W4A4, K, N, M, multipliers)
    assert p["kernel"] == kernel and p["launches"] == 1
    assert p["units"] == (-(-N // 64) if kernel == FP6 else 0) and p["whole"] == p["cut"] == 0
    # a call whose activations others may use keeps the form that all weights can read
    assert plan(W4A4, K, N, M, multipliers, once=False)["kernel"] == SKINNY
    assert plan(W4A4, K, N, 32, multipliers)["kernel"] == SKINNY


@pytest.mark.parametrize("type_,K,N,M,kernel", [
    (W4A4H, 5632, 64, 64, FP6), (W4A4H, 6144, 64, 33, SKINNY), (W4A4H, 6144, 768, 64, SKINNY), (W4A4H, 6144, 769, 64, FP6),
    (W4A4H, 8192, 64, 33, FP6), (W4A4, 5888, 512, 33, FP6), (W4A4, 6144, 1024, 48, SKINNY), (W4A4, 7936, 1025, 33, FP6),
    (W4A4, 8192, 2304, 64, SKINNY), (W4A4, 8192, 2305, 33, FP6), (W4A4, 9216, 64, 64, SKINNY), (W4A4, 9216, 2305, 64, FP6),
    (W4A4H, 9216, 2048, 64, SKINNY), (W4A4H, 9216, 2049, 64, FP6), (W4A4H, 9216, 2049, 40, SKINNY), (W4A4, 10240, 1792, 40, SKINNY),
    (W4A4H, 10240, 1792, 40, SKINNY), (W4A4H, 10240, 512, 41, FP6), (W4A4, 10240, 1793, 33, FP6), (W4A4, 10496, 4096, 64, SKINNY)])
@pytest.mark.parametrize("multipliers", [0, 1])
def test_33_to_64_tokens_of_few_panels(type_, K, N, M, multipliers, kernel):
    """A few panels of rows from K = 6144 up: where the units were up to 14 % slower than the skinny kernel on weights from memory."""
    assert plan(type_, K, N, M, multipliers)["kernel"] == kernel


def test_33_to_64_tokens_launch_by_launch():
    """With room for the largest weight only, every weight's own launch has to be one that the units are faster for."""
    Ns = (6144, 6144, 6144)
    room = rq.load_library().rq_w4a4_workspace_bytes(W4A4, 5120, 6144, 64)
    assert plan(W4A4, 5120, Ns, 64)["kernel"] == FP6 and plan(W4A4, 5120, Ns, 64)["launches"] == 1
    p = plan(W4A4, 5120, Ns, 64, workspace=room)
    assert p["kernel"] == SKINNY and p["launches"] == 3
    Ns = (12288, 9000, 6144)
    room = rq.load_library().rq_w4a4_workspace_bytes(W4A4, 1024, 12288, 64)
    assert plan(W4A4, 1024, Ns, 64, workspace=room)["kernel"] == SKINNY
    Ns = (12288, 9000, 8256)
    p = plan(W4A4, 1024, Ns, 64, workspace=room)
    assert p["kernel"] == FP6 and p["launches"] == 3 and p["units"] == 192 + 141 + 129


@pytest.mark.parametrize("K,N,M,multipliers,units", [
    (17408, 1000, 128, 0, True), (17664, 1000, 128, 0, False), (32768, 256, 1536, 0, False), (32768, 3000, 65, 0, False),
    (5120, 3000, 400, 0, True), (6144, 3000, 400, 0, True), (8192, 3000, 400, 0, False), (10240, 6000, 256, 0, False),
    (22528, 1000, 128, 1, True), (32768, 6000, 128, 1, True), (5120, 6000, 200, 1, True)])
def test_long_rows_above_64_tokens(K, N, M, multipliers, units):
    """Few tiles of long rows without multipliers are cut along K: units get weights from memory too slowly."""
    p = plan(W4A4, K, N, M, multipliers)
    assert (p["units"] > 0) == units and (p["cut"] > 0) == (not units) and p["whole"] == 0
    # without room for slices the other choice is whole tiles, a workgroup each: units
    assert plan(W4A4, K, N, M, multipliers, slabs=False)["units"] > 0


def test_every_tile_is_counted_once():
    """Tiles whole, cut, or in units (eight a tile where whole tiles run beside them)."""
    for N, M in [(17408, 65), (17408, 2048), (6100, 1500), (3000, 700), (256, 5000)]:
        p = plan(W4A4, 2560, N, M)
        tiles = -(-N // 256) * -(-M // 128)
        if p["whole"] + p["cut"] == 0:
            assert p["units"] == -(-N // 64) * -(-M // 64)
        else:
            assert p["whole"] + p["cut"] + p["units"] // 8 == tiles
        assert (p["slices"] > 1) == (p["cut"] > 0)


def test_no_tile_is_cut_without_slabs():
    assert plan(W4A4, 5120, 17408, 65)["cut"] == 68
    p = plan(W4A4, 5120, 17408, 65, slabs=False)
    assert p["cut"] == 0 and p["whole"] + p["units"] > 0


def test_refused_arguments():
    L = rq.load_library()
    out, N = (ctypes.c_int64 * 6)(), (ctypes.c_int64 * 1)(64)
    ask = lambda type_, n, K, M, ws, rot=0: L.rq_w4a4_product_plan(type_, n, K, N, M, rot, 0, 0, ws, out)
    assert ask(W4A4, 1, 512, 1, 1 << 24) == 0
    assert ask(W4A4, 0, 512, 1, 1 << 24) == -3 and ask(W4A4, 4, 512, 1, 1 << 24) == -3
    assert ask(W4A4, 1, 500, 1, 1 << 24) == -1 and ask(W4A4, 1, 512, 0, 1 << 24) == -1 and ask(12, 1, 512, 1, 1 << 24) == -1
    assert ask(W4A4H, 1, 512, 1, 1 << 24, 300) == -3
    assert ask(W4A4, 1, 512, 100, 1 << 10) == -2
