"""Kernels at the sizes where they can go wrong: remainders of tiles, first and last sizes of a range, against the CPU oracle.

Bounds: max|got - want| / max|want| <= 1e-3 for fp32 activations (fp16 operands), 2e-2 for bfloat16 ones, as in test_parity_gpu.py.
"""
import numpy as np
import pytest

from gomlx_amd import ggml, nn, synth
from gomlx_amd.nn import Activation, Quantization
from oracle import ggml_oracle as oracle

pytestmark = pytest.mark.gpu

TOL_F32, TOL_BF16 = 1e-3, 2e-2


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def rel(got, want):
    return float(np.max(np.abs(got - want))) / (float(np.max(np.abs(want))) or 1.0)


@pytest.mark.parametrize("slice_sb", [1, 7, 8])
@pytest.mark.parametrize("M", [33, 64, 97, 128, 129])
def test_q4_k_several_tiles_over_every_slice_length(gpu, monkeypatch, M, slice_sb):
    """One to four tiles of 32 batch rows against slices of one, seven and eight super-blocks (K is nine of them: the slices are uneven)."""
    monkeypatch.setenv("GOMLX_HIPQ_Q4K_SLICE_SB", str(slice_sb))
    monkeypatch.setenv("GOMLX_HIPQ_Q4K_TILES_TOGETHER", "2")
    K, N = 9 * 256, 2 * 256 + 36
    W, W2, x = synth.weights(ggml.Q4_K, 3, N, K), synth.weights(ggml.Q4_K, 4, N, K), synth.activations(5 + M, M, K)
    q = Quantization(ggml_type=ggml.Q4_K)
    xd, wd = dev(gpu, x), dev(gpu, W)
    want = oracle.c_qdense(ggml.Q4_K, x, W, None, oracle.ACT_NONE)
    assert rel(nn.quantized_dense(xd, wd, q).cpu().numpy(), want) < TOL_F32
    up = oracle.c_qdense(ggml.Q4_K, x, W2, None, oracle.ACT_NONE)
    got = nn.gated_feed_forward(xd, wd, dev(gpu, W2), q, Activation.RELU).cpu().numpy()
    assert np.max(np.abs(got - np.maximum(want, 0) * up)) < 2 * TOL_F32 * np.max(np.abs(want)) * np.max(np.abs(up))
