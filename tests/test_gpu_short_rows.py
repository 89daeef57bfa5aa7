"""Activations of short rows, bit for bit against the oracle, where the rotation kernel changes its form: up to 512 tokens and
more (256 threads a token; with twenty chunks also below, by what follows the rotation), rows without a Paley stage up to 256 tokens and more (the first eight Sylvester stages on the load),
and chunks that those stages use up, do not fill, or of a single float (where the scale needs a pass of its own)."""
import numpy as np
import pytest
import torch

import ruquant_amd as rq
from tests.gpu_util import adversarial_weights, adversarial_activations, bits_equal, first_mismatch, run_gpu

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("K,M", [(256, 5), (512, 64), (4096, 256), (4096, 257), (1024, 513), (1536, 513), (1280, 65), (3072, 512),
                                 (5120, 65), (5120, 513), (8192, 16), (8192, 200), (32768, 33)])
def test_product(oracle, K, M):
    type_, N = rq.TYPE_W4A4H, 40
    blocks, wf = adversarial_weights(oracle, N, K, type_, seed=K + M)
    W = rq.W4A4Weight(blocks, type_, DEV)
    x = adversarial_activations(M, K, type_, wf, seed=M)
    got, want = run_gpu(W, x), oracle.mul_mat(type_, blocks, x, W.clip, n_rot=W.n_rot)
    assert bits_equal(got, want), first_mismatch(got, want)


@pytest.mark.parametrize("M", [5, 257])
@pytest.mark.parametrize("n_rot", [1, 2, 8, 16, 32, 256, 512, 1024, 12, 192, 20, 320])
def test_rotation(oracle, n_rot, M):
    K = 1024 if n_rot & (n_rot - 1) == 0 else 3072 if n_rot % 12 == 0 else 5120
    x = np.random.default_rng(n_rot).standard_normal((M, K)).astype(np.float32)
    got = rq.hadamard(torch.from_numpy(x).to(DEV), n_rot).cpu().numpy()
    want = np.concatenate([oracle.hadamard(b) for b in x.reshape(-1, n_rot)]).reshape(M, K)
    assert bits_equal(got, want), first_mismatch(got, want)


@pytest.mark.parametrize("K,n_rot,M", [(1280, 1280, 65), (1280, 20, 512), (2560, 2560, 384), (2560, 2560, 385), (5120, 20, 65),
                                       (5120, 320, 100), (5120, 320, 385), (5120, 5120, 65), (5120, 2560, 512), (5120, 5120, 513)])
def test_rows_of_twenty_chunks(oracle, K, n_rot, M):
    rows = np.random.default_rng(K + n_rot).standard_normal((7, K)).astype(np.float32)
    rows[3] = 0.0
    token = np.arange(M) % 7
    x = torch.from_numpy(rows[token]).to(DEV)
    want = np.concatenate([oracle.hadamard(b) for b in rows.reshape(-1, n_rot)]).reshape(7, K)[token]
    got = rq.hadamard(x, n_rot).cpu().numpy()
    assert bits_equal(got, want), first_mismatch(got, want)
    clip = float(np.float32(0.9))
    want = [oracle.quantize_row_a4h(r, clip, n_rot).tobytes() for r in rows]
    got = rq.quantize_act(x, clip, hadamard_=True, n_rot=n_rot)
    assert all(got[t].tobytes() == want[t % 7] for t in range(M))
