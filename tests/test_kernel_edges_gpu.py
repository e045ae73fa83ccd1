"""Kernels at the sizes where they can go wrong: remainders of tiles, first and last sizes of a range, against the CPU oracle.

Bounds: max|got - want| / max|want| <= 1e-3 for fp32 activations (fp16 operands), 2e-2 for bfloat16 ones, as in test_parity_gpu.py.
"""
import ctypes

import numpy as np
import pytest

from gomlx_amd import _lib, ggml, nn, synth
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


GEMM_TYPES = [ggml.Q4_K, ggml.Q8_0, ggml.Q4_0, ggml.IQ4_NL]


@pytest.mark.parametrize("t", GEMM_TYPES)
@pytest.mark.parametrize("tm,slices,M,K,N", [
    (4, 1, 17, 256, 257),      # a single unit of K, one partly filled tile, N odd: element-wise stores
    (4, 3, 129, 768, 260),     # one row into the second tile, a slice per unit, four columns into the second workgroup
    (6, 1, 193, 1280, 36),     # one row over, N inside the first wavefront's tiles
    (8, 2, 255, 1280, 516),    # one row short, uneven slices
    (8, 1, 288, 512, 320),     # a whole tile and a whole 32-row part of the second
    (4, 1, 130, 512, 259),     # three columns that are no whole four, in the second workgroup's first wavefront
    (6, 1, 191, 512, 94),      # two, in the second wavefront
])
def test_gemm_with_weights_converted_in_registers(gpu, monkeypatch, t, tm, slices, M, K, N):
    """Every epilogue of gemm_wreg.hip (plain, bias and activation, residual behind a norm, gated pair, q / k / v of one input) at the edges of
    its tiles, fp32 and bfloat16 activations."""
    torch = gpu
    monkeypatch.setenv("GOMLX_HIPQ_GEMM_WREG", f"{tm},{slices}")
    W, W2, x = synth.weights(t, 3, N, K), synth.weights(t, 4, N, K), synth.activations(5 + M, M, K)
    rng = np.random.default_rng(M)
    bias, res = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
    q, wd, w2d, xd = Quantization(ggml_type=t), dev(torch, W), dev(torch, W2), dev(torch, x)
    gate, up = (oracle.c_qdense(t, x, w, None, oracle.ACT_NONE) for w in (W, W2))
    peak = float(np.max(np.abs(gate))) * float(np.max(np.abs(up)))
    assert rel(nn.quantized_dense(xd, wd, q).cpu().numpy(), gate) < TOL_F32
    got = nn.quantized_dense(xd, wd, q, dev(torch, bias), Activation.RELU).cpu().numpy()
    assert np.max(np.abs(got - np.maximum(gate + bias, 0))) < TOL_F32 * np.max(np.abs(gate))
    for act, f in ((Activation.SILU, lambda v: v / (1 + np.exp(-v))), (Activation.RELU, lambda v: np.maximum(v, 0))):
        got = nn.gated_feed_forward(xd, wd, w2d, q, act).cpu().numpy()
        assert np.max(np.abs(got - f(gate.astype(np.float64)) * up)) < 2 * TOL_F32 * peak
    norm = nn.RMSNorm(gain=dev(torch, np.ones(K, np.float32)), epsilon=1e-5)
    scale = np.sqrt(np.mean(x.astype(np.float64) ** 2, axis=1, keepdims=True) + 1e-5)
    got = nn.quantized_dense(xd, wd, q, norm=norm, residual=dev(torch, res)).cpu().numpy()
    assert np.max(np.abs(got - res - gate / scale)) < TOL_F32 * np.max(np.abs(gate / scale)) + 1e-6 * np.max(np.abs(res))
    if N % 32 == 0:
        outs = nn.quantized_dense_batch([(xd, w, q, None, None) for w in (wd, w2d, wd)], norm=norm)
        for o, w in zip(outs, (gate, up, gate)):
            assert rel(o.cpu().numpy(), w / scale) < TOL_F32
    xb = xd.to(torch.bfloat16)
    want = oracle.c_qdense(t, xb.float().cpu().numpy(), W, bias, oracle.ACT_NONE)
    assert rel(nn.quantized_dense(xb, wd, q, dev(torch, bias)).cpu().numpy(), want) < TOL_BF16


@pytest.mark.parametrize("t", GEMM_TYPES)
@pytest.mark.parametrize("tm,slices,M", [(4, 2, 130), (6, 3, 200), (8, 2, 257)])
def test_matrices_of_one_input_in_slices_with_weights_converted_in_registers(gpu, monkeypatch, t, tm, slices, M):
    """Three matrices of different widths, the last workgroup of each partly filled, K in slices: each one's columns of the shared sums."""
    torch, K, Ns = gpu, 5 * 256, (544, 288, 32)
    monkeypatch.setenv("GOMLX_HIPQ_GEMM_WREG", f"{tm},{slices}")
    x, Ws = synth.activations(5 + M, M, K), [synth.weights(t, 3 + i, n, K) for i, n in enumerate(Ns)]
    gain = 1 + 0.1 * np.random.default_rng(M).standard_normal(K).astype(np.float32)
    biases = [dev(torch, np.linspace(-1, 1, n, dtype=np.float32)) for n in Ns]
    norm = nn.RMSNorm(gain=dev(torch, gain), epsilon=1e-5)
    h = x * gain / np.sqrt(np.mean(x.astype(np.float64) ** 2, axis=1, keepdims=True) + 1e-5)
    xd, q = dev(torch, x), Quantization(ggml_type=t)
    outs = nn.quantized_dense_batch([(xd, dev(torch, w), q, b, None) for w, b in zip(Ws, biases)], norm=norm)
    for out, w, b in zip(outs, Ws, biases):
        want = oracle.c_qdense(t, h.astype(np.float32), w, None, oracle.ACT_NONE)
        assert np.max(np.abs(out.cpu().numpy() - want - b.cpu().numpy())) < TOL_F32 * np.max(np.abs(want))


@pytest.mark.parametrize("t", GEMM_TYPES)
@pytest.mark.parametrize("bf16", [False, True])
def test_gemm_with_weights_converted_in_registers_and_infinite_activations(gpu, monkeypatch, t, bf16):
    """Rows with +inf, with -inf and with both, as in 64 bits on weights rounded to the operands' 16 bits, where a zero makes a NaN; the other rows stay finite."""
    torch, M, K, N = gpu, 300, 512, 260
    monkeypatch.setenv("GOMLX_HIPQ_GEMM_WREG", "8,1")
    W = synth.weights(t, 77, N, K)
    x = np.random.default_rng(M).standard_normal((M, K)).astype(np.float32)
    x[1, K - 3], x[130, 5], x[299, 17], x[299, K - 300] = np.inf, -np.inf, np.inf, -np.inf
    xd, w = dev(torch, x), torch.from_numpy(oracle.c_dequantize(t, W, K))
    w = w.to(torch.bfloat16 if bf16 else torch.float16).double().numpy()
    got = nn.quantized_dense(xd.to(torch.bfloat16) if bf16 else xd, dev(torch, W), Quantization(ggml_type=t)).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.T
    for m in (1, 130, 299):
        assert not np.isfinite(want[m]).any()
        np.testing.assert_array_equal(got[m], want[m])
    assert np.isfinite(np.delete(got, (1, 130, 299), axis=0)).all()


def test_gemm_with_weights_converted_in_registers_keeps_infinities(gpu, monkeypatch):
    """A block of infinite scale in one weight row: that output column is infinite or NaN as the reference's, every other one untouched."""
    torch = gpu
    K, N, M = 512, 63, 40
    monkeypatch.setenv("GOMLX_HIPQ_SPLIT_K_TO", "16")
    for t in GEMM_TYPES:
        W = synth.weights(t, 3, N, K)
        W[5, 0:2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
        bpb = ggml.bytes_per_block(t)
        # largest code (and sub-block scale) everywhere: no infinity meets a zero or its opposite inside the block
        W[5, 4 if t == ggml.Q4_K else 2:bpb] = 0x7F if t == ggml.Q8_0 else 0xFF
        x = np.abs(synth.activations(9, M, K)) + 0.1
        monkeypatch.setenv("GOMLX_HIPQ_GEMM_WREG", "4")
        got = nn.quantized_dense(dev(torch, x), dev(torch, W), Quantization(ggml_type=t)).cpu().numpy()
        want = oracle.c_qdense(t, x, W, None, oracle.ACT_NONE)
        assert np.all(np.isposinf(want[:, 5])) and np.all(np.isposinf(got[:, 5]))
        ok = np.arange(N) != 5
        assert rel(got[:, ok], want[:, ok]) < TOL_F32


@pytest.mark.parametrize("t,M,K,N", [
    (ggml.Q4_K, 6, 5120, 2305), (ggml.Q4_K, 12, 4096, 3075), (ggml.Q4_K, 32, 4096, 3074), (ggml.Q4_K, 77, 4096, 3073), (ggml.Q4_K, 128, 4096, 3077),
    (ggml.Q8_0, 17, 4096, 1601), (ggml.Q8_0, 66, 4096, 1603), (ggml.Q4_0, 33, 4096, 2891), (ggml.IQ4_NL, 12, 5120, 2337), (ggml.Q6_K, 20, 4096, 2051),
    (ggml.Q6_K, 5, 8192, 1025),
])
def test_split_k_rows_of_any_length(gpu, t, M, K, N):
    """The split-K routes with N off every multiple of four (their sums' rows are padded, the outputs stored element by element): plain with
    bias, behind a norm with a residual, a gated pair, q / k / v of one input, outputs that are not 16-byte aligned, bfloat16 rows. Up to 16 rows
    such calls stay on the GEMV (16-bit fixed point per 32 values: a step of 2^-15 of their maximum, about 2.5 sigma, is 2.2e-5 sigma rms) and the
    few-row kernel (20 bits); one fp16, a step of 2^-11 of each value, is 1e-4 rms.  Over a sum both stay in that proportion to the output's
    rms, and the largest error to the largest output about so: 5e-5 lies between."""
    torch = gpu
    W, W2, x = synth.weights(t, 3, N, K), synth.weights(t, 4, N, K), synth.activations(5 + M, M, K)
    rng = np.random.default_rng(M)
    bias, res = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
    q, wd, w2d, xd = Quantization(ggml_type=t), dev(torch, W), dev(torch, W2), dev(torch, x)
    gate, up = (oracle.c_qdense(t, x, w, None, oracle.ACT_NONE) for w in (W, W2))
    peak = float(np.max(np.abs(gate)))
    got = nn.quantized_dense(xd, wd, q, dev(torch, bias), Activation.RELU).cpu().numpy()
    assert np.max(np.abs(got - np.maximum(gate + bias, 0))) < TOL_F32 * peak
    if M <= 16:
        assert rel(nn.quantized_dense(xd, wd, q).cpu().numpy(), gate) < 5e-5
    got = nn.quantized_dense(xd, wd, q, dev(torch, np.concatenate([bias, bias]))[1:N + 1]).cpu().numpy()  # a bias off 16 bytes
    assert np.max(np.abs(got - gate - np.concatenate([bias, bias])[1:N + 1])) < TOL_F32 * peak
    norm = nn.RMSNorm(gain=dev(torch, np.ones(K, np.float32)), epsilon=1e-5)
    scale = np.sqrt(np.mean(x.astype(np.float64) ** 2, axis=1, keepdims=True) + 1e-5)
    got = nn.quantized_dense(xd, wd, q, norm=norm, residual=dev(torch, res)).cpu().numpy()
    assert np.max(np.abs(got - res - gate / scale)) < TOL_F32 * np.max(np.abs(gate / scale)) + 1e-6 * np.max(np.abs(res))
    got = nn.gated_feed_forward(xd, wd, w2d, q, Activation.RELU).cpu().numpy()
    assert np.max(np.abs(got - np.maximum(gate, 0) * up)) < 2 * TOL_F32 * peak * np.max(np.abs(up))
    outs = nn.quantized_dense_batch([(xd, w, q, None, None) for w in (wd, w2d, wd)], norm=norm)
    for o, w in zip(outs, (gate, up, gate)):
        assert rel(o.cpu().numpy(), w / scale) < TOL_F32
    xb = xd.to(torch.bfloat16)
    want = oracle.c_qdense(t, xb.float().cpu().numpy(), W, bias, oracle.ACT_NONE)
    assert rel(nn.quantized_dense(xb, wd, q, dev(torch, bias)).cpu().numpy(), want) < TOL_F32


@pytest.mark.parametrize("t", GEMM_TYPES + [ggml.Q6_K])
@pytest.mark.parametrize("K,N", [(2048, 131), (2048, 1150), (4608, 509)])
def test_small_matrices_with_rows_of_any_length_keep_their_weights_exact(gpu, t, K, N):
    """Less than 2.4 million values with N off every multiple of four: unit vectors return the weights themselves, which the split-K kernels
    contract as they are (a 16-bit image would round them)."""
    W = np.tile(synth.weights(t, 77 + t, 67, K), (-(-N // 67), 1))[:N]
    cols = np.linspace(0, K - 1, 20).astype(int)
    x = np.zeros((20, K), np.float32)
    x[np.arange(20), cols] = 1.0
    got = nn.quantized_dense(dev(gpu, x), dev(gpu, W), Quantization(ggml_type=t)).cpu().numpy()
    want = np.tile(oracle.c_dequantize(t, W[:67], K), (-(-N // 67), 1))[:N, cols].T
    assert np.array_equal(got, want)


def off16(torch, a):
    """A copy of a float32 array on the GPU that starts 4 bytes behind a multiple of 16."""
    buf = torch.empty(a.size + 1, dtype=torch.float32, device="cuda")
    view = buf[1:].view(a.shape)
    view.copy_(torch.from_numpy(a))
    assert view.data_ptr() % 16 == 4
    return view


@pytest.mark.parametrize("t,M,K,N", [
    (ggml.Q4_K, 17, 2048, 1024), (ggml.Q4_K, 96, 2048, 1024), (ggml.Q8_0, 40, 4096, 512), (ggml.Q4_0, 128, 2048, 1024), (ggml.IQ4_NL, 70, 2048, 8192),
    (ggml.Q6_K, 33, 2048, 1024), (ggml.Q6_K, 96, 2048, 1024), (ggml.Q4_K, 300, 14336, 4096),
    (ggml.Q8_0, 8, 8192, 1024), (ggml.Q4_K, 12, 14336, 4096),  # few rows: two launches of the few-row kernel, three of the split-K ones
])
@pytest.mark.parametrize("bf16", [False, True])
def test_residual_and_up_bias_off_16_bytes_keep_the_route(gpu, t, M, K, N, bf16):
    """A residual or an up bias off 16 bytes is read element by element: the same bits as an aligned one, on the split-K kernels, whose weights are exact,
    up to the same row counts.  Up to 16 rows an up bias off 16 bytes keeps the pair on routes with more bits of the activations instead: within those of
    the split-K kernels' fp16 (2^-11 of each value, 1e-4 rms of the largest output and a tenth of the bound of 1e-3 in either factor)."""
    torch = gpu
    reps = -(-N // 97)
    wd, w2d = (dev(torch, np.tile(synth.weights(t, s, 97, K), (reps, 1))[:N]) for s in (3, 4))
    x = dev(torch, synth.activations(5 + M, M, K))
    x = x.to(torch.bfloat16) if bf16 else x
    rng = np.random.default_rng(M)
    res, bias = rng.standard_normal((M, N)).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    q, norm = Quantization(ggml_type=t), nn.RMSNorm(gain=dev(torch, 1 + 0.1 * rng.standard_normal(K).astype(np.float32)), epsilon=1e-5)
    for n in (None, norm):
        a, b = (nn.quantized_dense(x, wd, q, dev(torch, bias), norm=n, residual=r) for r in (dev(torch, res), off16(torch, res)))
        assert torch.equal(a, b)
        a, b = (nn.gated_feed_forward(x, wd, w2d, q, Activation.RELU, dev(torch, bias), u, norm=n) for u in (dev(torch, bias), off16(torch, bias)))
        if M > 16:
            assert torch.equal(a, b)
        else:
            assert float((a - b).abs().max()) < 2 * TOL_F32 * float(a.abs().max())


@pytest.mark.parametrize("t,M,K,N,wreg", [
    (ggml.Q4_K, 40, 4096, 1024, None), (ggml.Q8_0, 17, 4096, 1028, None), (ggml.Q4_0, 66, 4096, 1024, None), (ggml.Q6_K, 20, 4096, 1024, None),  # split-K
    (ggml.Q8_0, 129, 512, 260, "4,1"), (ggml.Q4_K, 255, 512, 516, "8,1"), (ggml.IQ4_NL, 193, 768, 36, "6,1"),  # the GEMM that converts weights in registers
    (ggml.Q4_0, 257, 512, 289, "8,1"), (ggml.Q8_0, 190, 512, 34, "6,1"), (ggml.Q4_K, 129, 512, 3, "4,1"),
])
def test_outputs_off_16_bytes(gpu, monkeypatch, t, M, K, N, wreg):
    """y off 16 bytes, N a multiple of four and not: the same bits as at an aligned address - plain, a residual stream updated in place, a gated pair - and
    no element outside y."""
    torch = gpu
    if wreg:
        monkeypatch.setenv("GOMLX_HIPQ_GEMM_WREG", wreg)
    L, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    W, W2, x = synth.weights(t, 3, N, K), synth.weights(t, 4, N, K), synth.activations(5 + M, M, K)
    rng = np.random.default_rng(M)
    bias, res = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
    wd, w2d, xd, bd, rd = dev(torch, W), dev(torch, W2), dev(torch, x), dev(torch, bias), dev(torch, res)
    def calls(y):
        yp = y.data_ptr()
        yield lambda: L.gq_qdense_f32(t, xd.data_ptr(), M, K, wd.data_ptr(), N, bd.data_ptr(), oracle.ACT_RELU, yp, stream)
        yield lambda: L.gq_qdense_block_f32(t, xd.data_ptr(), M, K, None, wd.data_ptr(), N, bd.data_ptr(), oracle.ACT_NONE, yp, yp, stream)
        yield lambda: L.gq_qdense_gated_f32(t, xd.data_ptr(), M, K, None, wd.data_ptr(), bd.data_ptr(), w2d.data_ptr(), None, N, oracle.ACT_RELU, yp, stream)
    buf = torch.full((M * N + 8,), 7.0, device="cuda")
    y, odd = torch.empty(M, N, device="cuda"), buf[5:5 + M * N].view(M, N)
    gate, up = (oracle.c_qdense(t, x, w, b, oracle.ACT_NONE) for w, b in ((W, bias), (W2, None)))
    wants = [np.maximum(gate, 0), gate + res, np.maximum(gate, 0) * up]
    for a, b, want in zip(calls(y), calls(odd), wants):
        for out, call in ((y, a), (odd, b)):
            out.copy_(rd)
            _lib.check(call())
        assert torch.equal(y, odd)
        assert np.max(np.abs(y.cpu().numpy() - want)) < 2 * TOL_F32 * np.max(np.abs(want))
        assert bool((buf[:5] == 7).all()) and bool((buf[5 + M * N:] == 7).all())


@pytest.mark.parametrize("recorded", [False, True])
def test_split_k_without_room_falls_back(gpu, recorded):
    """N off every multiple of four at 128 rows: the split-K kernels' scratch memory (23 MiB here) does not fit the static array, or what the stream holds when
    a recording begins; the call goes on to the two passes (16 MiB), whose weights are rounded to 16 bits."""
    torch, t, M, K, N = gpu, ggml.Q4_K, 128, 16384, 351
    L = _lib.lib()
    W, x = synth.weights(t, 3, N, K), synth.activations(4, 129, K)
    wd, xd = dev(torch, W), dev(torch, x)
    want = oracle.c_qdense(t, x[:M], W, None, oracle.ACT_NONE)
    y = torch.zeros(M, N, device="cuda")
    split = nn.quantized_dense(xd[:M], wd, Quantization(ggml_type=t)).cpu().numpy()
    assert rel(split, want) < TOL_F32
    if not recorded:
        _lib.check(L.gq_qdense_f32_static(t, xd.data_ptr(), M, K, wd.data_ptr(), N, None, 0, y.data_ptr(), torch.cuda.current_stream().cuda_stream))
        got = y.cpu().numpy()
    else:
        torch.cuda.synchronize()
        sp = ctypes.c_void_p()
        _lib.check(L.gq_stream_create(ctypes.byref(sp)))
        dense = lambda rows, out: _lib.check(L.gq_qdense_f32(t, xd.data_ptr(), rows, K, wd.data_ptr(), N, None, 0, out.data_ptr(), sp))
        one_more = torch.zeros(129, N, device="cuda")
        torch.cuda.synchronize()
        dense(129, one_more)  # two passes: the stream holds what they need
        _lib.check(L.gq_sync(sp))
        _lib.check(L.gq_graph_begin(sp))
        dense(M, y)
        g = ctypes.c_void_p()
        _lib.check(L.gq_graph_end(sp, ctypes.byref(g)))
        for _ in range(3):
            y.fill_(float("nan"))
            torch.cuda.synchronize()
            dense(129, one_more)
            _lib.check(L.gq_graph_launch(g, sp))
            _lib.check(L.gq_sync(sp))
            got = y.cpu().numpy()
            assert np.array_equal(got, one_more[:M].cpu().numpy())
        _lib.check(L.gq_graph_destroy(g))
        _lib.check(L.gq_stream_destroy(sp))
    assert rel(got, want) < TOL_F32 and not np.array_equal(got, split)


@pytest.mark.parametrize("t", GEMM_TYPES + [ggml.Q6_K])
@pytest.mark.parametrize("M,K,N", [(20, 4096, 2051), (40, 4096, 1602), (96, 8192, 1025), (64, 2048, 1024)])
@pytest.mark.parametrize("bf16", [False, True])
def test_infinite_activations_of_batches_with_rows_of_any_length(gpu, t, M, K, N, bf16):
    """The split-K kernels, N off every multiple of four and not: rows with +inf, with -inf and with both are the infinities and NaN of 64 bits, the other
    rows finite, as on the routes these calls had before.  (Q4_K's sub-block minima are a second sum, in which an infinity meets its opposite: several
    infinities in one slice of K are NaN there, one is not.)"""
    torch = gpu
    W = np.tile(synth.weights(t, 77, 131, K), (-(-N // 131), 1))[:N]
    x = np.random.default_rng(M + K).standard_normal((M, K)).astype(np.float32)
    x[1, K - 3], x[3, 5], x[4, 17], x[4, K - 300] = np.inf, -np.inf, np.inf, -np.inf
    x[6, 700:702], x[8, 9], x[8, 600] = np.inf, -np.inf, np.nan
    xd = dev(torch, x)
    if bf16:
        xd = xd.to(torch.bfloat16)
        x = xd.float().cpu().numpy()
    got = nn.quantized_dense(xd, dev(torch, W), Quantization(ggml_type=t)).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = np.tile(x.astype(np.float64) @ oracle.c_dequantize(t, W[:131], K).astype(np.float64).T, (1, -(-N // 131)))[:, :N]
    for m in (1, 3, 4, 6, 8):
        assert not np.isfinite(want[m]).any()
        nan = np.isnan(got[m]) & (t == ggml.Q4_K and m in (4, 6))
        np.testing.assert_array_equal(got[m][~nan], want[m][~nan])
    assert np.isfinite(np.delete(got, (1, 3, 4, 6, 8), axis=0)).all()


@pytest.mark.parametrize("count", [1, 1024, 1025, 16385])
def test_gather_finds_a_bad_index_wherever_it_is(gpu, count):
    """First, middle and last index, alone on the stream and behind other work."""
    torch = gpu
    K, vocab = 32, 50
    table = synth.weights(ggml.Q8_0, 3, vocab, K)
    q, td = Quantization(ggml_type=ggml.Q8_0), dev(torch, table)
    idx = (np.arange(count, dtype=np.int32) * 7 % vocab).reshape(-1, 1)
    want = oracle.c_dequantize(ggml.Q8_0, table, K)[idx[:, 0]]
    idx_d = dev(torch, idx)
    for ahead in (0, 10_000_000):
        torch.cuda._sleep(ahead)
        assert np.array_equal(nn.quantized_gather(td, idx_d, q).cpu().numpy().view(np.uint32), want.view(np.uint32))
    for bad, at in ((vocab, count - 1), (-1, 0), (vocab, count // 2)):
        wrong = idx.copy()
        wrong[at] = bad
        with pytest.raises(IndexError):
            nn.quantized_gather(td, dev(torch, wrong), q)


@pytest.mark.parametrize("bad", [False, True])
def test_gather_returns_with_its_rows_written(gpu, bad):
    """256 MiB of rows, some 50 us of writing: the stream has nothing left to do when the call returns or raises, so that a reader on another
    stream needs no event and memory of another stream may be released."""
    torch = gpu
    K, vocab, count = 4096, 64, 16384
    td = dev(torch, synth.weights(ggml.Q8_0, 3, vocab, K))
    idx = torch.arange(count, dtype=torch.int32, device="cuda").remainder_(vocab).view(-1, 1)
    if bad:
        idx[count - 1] = vocab
    torch.cuda.synchronize()
    if bad:
        with pytest.raises(IndexError):
            nn.quantized_gather(td, idx, Quantization(ggml_type=ggml.Q8_0))
    else:
        nn.quantized_gather(td, idx, Quantization(ggml_type=ggml.Q8_0))
    assert torch.cuda.current_stream().query()


@pytest.mark.parametrize("t", [ggml.Q4_0, ggml.Q8_0, ggml.IQ4_NL])
@pytest.mark.parametrize("K,N", [(4352, 16420), (2048, 33290)])
def test_32_value_blocks_over_long_slices(gpu, t, K, N):
    """Several tiles of batch rows over slices of more than 1024 values: three of 1536 or 2048 whose last is cut short, and one of 2048; with
    a normalisation, whose sums of squares come from four wavefronts per slice then."""
    torch, M = gpu, 40
    W = synth.weights(t, 3, 131, K)
    x = synth.activations(5, M, K)
    want = oracle.c_qdense(t, x, W, None, oracle.ACT_NONE)
    reps = -(-N // 131)
    q, xd = Quantization(ggml_type=t), dev(torch, x)
    wd = dev(torch, np.tile(W, (reps, 1))[:N])
    assert rel(nn.quantized_dense(xd, wd, q).cpu().numpy(), np.tile(want, (1, reps))[:, :N]) < TOL_F32
    norm = nn.RMSNorm(gain=dev(torch, np.ones(K, np.float32)), epsilon=1e-5)
    want = want / np.sqrt(np.mean(x.astype(np.float64) ** 2, axis=1, keepdims=True) + 1e-5)
    assert rel(nn.quantized_dense(xd, wd, q, norm=norm).cpu().numpy(), np.tile(want, (1, reps))[:, :N]) < TOL_F32
