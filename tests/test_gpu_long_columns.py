"""Rows of at least 256 columns of a long Paley stage, bit for bit against the oracle: the rotation alone, the rotation with the
quantizer and, with the transposed signs, the dequantizer. 256 columns go to four threads each (paley_row), in one chunk or in
many down to four columns; more columns to four threads or to one each, by the order of the Paley matrix, the token count and
what follows (takes_wide), whole runs of 256 and ragged ones."""
import numpy as np
import pytest
import torch

import ruquant_amd as rq
from tests.gpu_util import bits_equal, first_mismatch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("K,n_rot", [(11264, 11264), (17408, 17408), (17408, 4352), (22528, 22528), (22528, 5632), (30720, 30720),
                                     (21504, 21504), (26624, 26624), (27648, 6912),
                                     # 256 columns in chunks shorter than 16 and of 16
                                     (11264, 176), (15360, 480), (17408, 272), (17408, 1088), (26624, 832), (27648, 432),
                                     # more columns, in chunks of 4 to 256
                                     (30976, 352), (14080, 2816), (22528, 11264), (19200, 3840), (30720, 240), (30720, 15360),
                                     (30464, 272), (30464, 4352), (20736, 2304), (26880, 5376), (29952, 832), (32256, 1344)])
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


@pytest.mark.parametrize("K,n_rot", [(22528, 22528), (30720, 15360), (16896, 5632), (19712, 2816), (30464, 4352), (27648, 9216),
                                     (29952, 3328), (32256, 5376), (26112, 544)])
@pytest.mark.parametrize("M", [2, 45, 130])
def test_rotation_and_quantizer(oracle, K, n_rot, M):
    """The same stage in front of the quantizer, up to 40 tokens, more, and from 129 (a few of which are compared)."""
    rng = np.random.default_rng(K + n_rot + M)
    x = rng.standard_normal((M, K)).astype(np.float32)
    got = rq.quantize_act(torch.from_numpy(x).to(DEV), 0.9, hadamard_=True, n_rot=n_rot)
    rot = rq.hadamard(torch.from_numpy(x).to(DEV), n_rot).cpu().numpy()
    for t in {0, 1, M // 2, M - 1}:
        want = oracle.quantize_row_a4h(x[t], 0.9, n_rot=n_rot)
        assert got[t].tobytes() == want.tobytes(), t
        want = np.concatenate([oracle.hadamard(x[t, o:o + n_rot]) for o in range(0, K, n_rot)])
        assert bits_equal(rot[t], want), first_mismatch(rot[t], want)
