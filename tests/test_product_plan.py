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
