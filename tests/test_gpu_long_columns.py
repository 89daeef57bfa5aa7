"""Rows of at least 256 columns of a long Paley stage, whose columns four threads share (paley_row): the rotation and, with the
transposed signs, the dequantizer, bit for bit against the oracle. 256 columns (one run of the workgroup), 512 (two), and 256 of
several rotation blocks, whose chunks are shorter than a run."""
import numpy as np
import pytest
import torch

import ruquant_amd as rq
from tests.gpu_util import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("K,n_rot", [(11264, 11264), (17408, 17408), (17408, 4352), (22528, 22528), (22528, 5632), (30720, 30720),
                                     (21504, 21504), (26624, 26624), (27648, 6912)])
@pytest.mark.parametrize("M", [1, 3])
def test_rotation_and_its_inverse(oracle, K, n_rot, M):
    rng = np.random.default_rng(K + n_rot + M)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[:, ::97] = -0.0
    got = rq.hadamard(torch.from_numpy(x).to(DEV), n_rot).cpu().numpy()
    want = np.stack([np.concatenate([oracle.hadamard(x[t, o:o + n_rot]) for o in range(0, K, n_rot)]) for t in range(M)])
    assert bits_equal(got, want), first_mismatch(got, want)
    blocks = oracle.quantize_rows_w(x, hadamard=True, n_rot=n_rot)
    back = rq.dequantize(blocks, rq.TYPE_W4A4H).cpu().numpy()
    want = np.stack([oracle.dequantize_row_w(blocks[t], hadamard=True) for t in range(M)])
    assert bits_equal(back, want), first_mismatch(back, want)
