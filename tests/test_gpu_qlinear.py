"""GPU parity of the affine-quantized projections against the oracle's
restatement of MLX's format: y = x @ dequantize(W).T (the reference test's
dense comparison, tests/test_qwen3_5_linear_attention.py:59-86)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import mlx_lean_moe_amd as gdn
from mlx_lean_moe_amd import _lib
from mlx_lean_moe_amd.quant import _f32_matmul, decode_kernel_takes, quantized_linear_split
from oracle import quant_ref as Q
from oracle import gated_delta_ref as R
from tests.helpers import assert_bf16_out_close, layer_inputs, layer_params

pytestmark = pytest.mark.gpu

_TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _weights(rng, N, K, bits, gs, sb):
    words, s, b = Q.quantize(rng.standard_normal((N, K)) * 0.05, bits, gs, sb=sb)
    return words, s, b


def _dev_weights(gpu, words, s, b, sb):
    return {"weight": torch.tensor(words.view(np.int32), device=gpu),
            "scales": torch.tensor(s, dtype=torch.float32, device=gpu).to(_TORCH[sb]),
            "biases": torch.tensor(b, dtype=torch.float32, device=gpu).to(_TORCH[sb])}


def _decode_kernel_takes(M, K, bits, gs, sb):
    return decode_kernel_takes(M, K, bits, gs, _TORCH[sb])


@pytest.mark.parametrize("M,N,K,bits,gs,sb", [
    (1, 40, 128, 4, 64, "bf16"),
    (7, 96, 256, 4, 32, "f16"),
    (64, 12352, 2048, 4, 64, "bf16"),   # the layer's stacked input projection at decode
    (33, 2048, 4096, 4, 64, "bf16"),    # out_proj at decode (value_dim 4096 -> hidden)
    (5, 70, 1024, 8, 32, "f16"),
    (200, 130, 512, 8, 128, "f32"),     # quantized_linear: dense; the ABI: the kernel for 65-511 rows
    (300, 2048, 1024, 4, 64, "bf16"),   # the same, ragged last row tile
    (2, 78, 256, 4, 64, "bf16"),        # decode kernel: 4 groups per column, last block partial
    (3, 77, 256, 4, 64, "bf16"),        # scales span not whole 16-byte pieces: tiled kernel
    (16, 200, 1024, 4, 32, "f32"),      # decode kernel with float32 scales
    (64, 100, 4096, 8, 32, "f32"),      # scales exceed the decode kernel's LDS: tiled kernel
    (9, 64, 4096, 8, 128, "bf16"),      # 8-bit codes past the decode kernel's registers: tiled
    (1, 4096, 2048, 4, 64, "bf16"),     # decode kernel, one row
    (2, 78, 512, 4, 64, "bf16"),        # decode kernel, one step, last block partial
    (17, 130, 2048, 8, 64, "f16"),      # decode kernel, 8-bit codes, 64-k slices
    (48, 96, 1024, 4, 128, "f32"),      # decode kernel, two slices per group
    (600, 256, 512, 4, 64, "bf16"),     # quantized_linear: dequantize + BLAS; the ABI: tiled kernel
])
def test_quantized_matmul_matches_oracle(gpu, M, N, K, bits, gs, sb):
    rng = np.random.default_rng(M + N + K)
    words, s, b = _weights(rng, N, K, bits, gs, sb)
    x = R.bf16_round(rng.standard_normal((M, K)))
    # bf16 activations: the decode kernel applies scales and biases to float
    # partial sums (exact weights); the tiled kernels dequantize the weights
    # to bf16 whatever the scales' dtype (gdn_quantized_matmul's contract)
    exact = _decode_kernel_takes(M, K, bits, gs, sb)
    ref = Q.quantized_matmul(x, words, s, b, bits, gs, w_round="f32" if exact else "bf16")
    scheme = gdn.QuantScheme(bits, gs)
    W = _dev_weights(gpu, words, s, b, sb)
    xt = torch.tensor(x, dtype=torch.float32, device=gpu).to(torch.bfloat16)
    y = gdn.quantized_linear(xt, W, scheme)
    assert y.dtype == torch.bfloat16 and tuple(y.shape) == (M, N)
    assert_bf16_out_close(y.float().cpu().numpy(), ref)
    # float32 output: the accumulation alone (no output rounding)
    y32 = torch.empty(M, N, device=gpu)
    _lib.call("gdn_quantized_matmul", _lib.ptr(xt), _lib.GDN_BF16, _lib.ptr(W["weight"]),
              _lib.ptr(W["scales"]), _lib.ptr(W["biases"]), _lib.dtype_code(W["scales"].dtype),
              _lib.ptr(y32), _lib.GDN_F32, None, M, N, K, bits, gs, None, 0, _lib.stream_ptr(xt.device))
    err = np.abs(y32.cpu().numpy() - ref).max()
    assert err <= 1e-5 * np.abs(ref).max() + 1e-6, err


@pytest.mark.parametrize("M,N,K,bits,gs,sb", [
    (1, 4096, 2048, 4, 64, "bf16"),     # one decode row, as the reference runs (float32 activations)
    (16, 200, 1024, 4, 32, "f32"),
    (17, 130, 2048, 8, 64, "f16"),      # 17-32 rows: 64-column workgroups
    (32, 78, 512, 4, 64, "bf16"),
])
def test_float32_activations_on_the_decode_kernel(gpu, M, N, K, bits, gs, sb):
    """float32 x (split into bf16 hi + lo, ~16 significant bits) against the
    exact weights: what mx.quantized_matmul computes for float32 x."""
    assert decode_kernel_takes(M, K, bits, gs, _TORCH[sb])
    rng = np.random.default_rng(M * 7 + N)
    words, s, b = _weights(rng, N, K, bits, gs, sb)
    x = rng.standard_normal((M, K)).astype(np.float32)
    ref = Q.quantized_matmul(x, words, s, b, bits, gs, w_round="f32")
    W = _dev_weights(gpu, words, s, b, sb)
    y = gdn.quantized_linear(torch.tensor(x, device=gpu), W, gdn.QuantScheme(bits, gs))
    assert y.dtype == torch.float32
    err = np.abs(y.cpu().numpy() - ref).max()
    assert err <= 1e-4 * np.abs(ref).max() + 1e-6, err
    # more than 32 float32 rows: the C entry declines, quantized_linear dequantizes
    assert _lib.load().gdn_quantized_matmul(
        None, _lib.GDN_F32, _lib.ptr(W["weight"]), _lib.ptr(W["scales"]), _lib.ptr(W["biases"]),
        _lib.dtype_code(W["scales"].dtype), None, _lib.GDN_F32, None, 33, N, K, bits, gs,
        None, 0, None) == _lib.GDN_EUNSUPPORTED


@pytest.mark.parametrize("N,K,gs,sb,x32", [
    (12352, 2048, 64, "bf16", False),   # the stacked input projection, one sequence
    (12352, 2048, 64, "bf16", True),
    (2048, 4096, 64, "bf16", False),    # out_proj: two rounds of lane chunks
    (2047, 4096, 128, "bf16", True),    # odd N: the last wave's second column is idle
    (777, 1024, 32, "f16", False),      # half the lanes hold a chunk
    (130, 512, 128, "f32", True),       # a quarter of them; f32 scales
])
def test_one_row_runs_the_matrix_vector_kernel_exactly(gpu, N, K, gs, sb, x32):
    """One row of x and 4-bit codes (a single sequence's decode step) take
    the matrix-vector kernel: products against the exact weights s q + b,
    accumulated in float (bf16 x as bf16 pairs against 1 + q / 16; float32
    x in float32), within 1e-5 of the float64 product."""

    assert _decode_kernel_takes(1, K, 4, gs, sb)
    assert _lib.load().gdn_quantized_matmul_workspace_size(
        _lib.GDN_F32 if x32 else _lib.GDN_BF16, _lib.dtype_code(_TORCH[sb]), 1, N, K, 4, gs) == 0
    rng = np.random.default_rng(N + K)
    words, s, b = _weights(rng, N, K, 4, gs, sb)
    x = rng.standard_normal((1, K)).astype(np.float32)
    if not x32:
        x = R.bf16_round(x)
    ref = Q.quantized_matmul(x, words, s, b, 4, gs, w_round="f32")
    W = _dev_weights(gpu, words, s, b, sb)
    xt = torch.tensor(x, device=gpu).to(torch.float32 if x32 else torch.bfloat16)
    y = torch.empty(1, N, device=gpu)
    _lib.call("gdn_quantized_matmul", _lib.ptr(xt), _lib.dtype_code(xt.dtype), _lib.ptr(W["weight"]),
              _lib.ptr(W["scales"]), _lib.ptr(W["biases"]), _lib.dtype_code(W["scales"].dtype),
              _lib.ptr(y), _lib.GDN_F32, None, 1, N, K, 4, gs, None, 0, _lib.stream_ptr(gpu))
    err = np.abs(y.cpu().numpy() - ref).max()
    assert err <= 1e-5 * np.abs(ref).max() + 1e-6, err
    # a 1-D x through quantized_linear gives the same bits in x's dtype
    y1 = gdn.quantized_linear(xt[0], W, gdn.QuantScheme(4, gs))
    assert tuple(y1.shape) == (N,)
    np.testing.assert_array_equal(y1.float().cpu().numpy(), y[0].to(xt.dtype).float().cpu().numpy())


@pytest.mark.parametrize("M,N,K,bits,gs,sb,x32,splits", [
    (64, 8192, 2048, 8, 64, "bf16", False, 2),   # 128 column tiles of 64
    (16, 2048, 4096, 4, 64, "bf16", False, 4),   # out_proj at 16 rows: 64 tiles of 32
    (1, 1000, 2048, 8, 32, "f16", False, 8),     # ragged last tile
    (40, 100, 2048, 8, 64, "f32", False, 4),
    (5, 300, 1024, 4, 32, "bf16", True, 4),      # float32 x
])
def test_split_k_matches_the_unsplit_kernel_and_the_oracle(gpu, M, N, K, bits, gs, sb, x32, splits):
    """Few column tiles: with the workspace the decode kernel splits K over
    workgroups (float32 partial blocks, added in a fixed order). Both the
    split and the unsplit result meet the oracle's bound, they agree to
    float32 rounding, and two split runs agree bit for bit."""

    rng = np.random.default_rng(M * 31 + N)
    words, s, b = _weights(rng, N, K, bits, gs, sb)
    x = rng.standard_normal((M, K)).astype(np.float32)
    if not x32:
        x = R.bf16_round(x)
    ref = Q.quantized_matmul(x, words, s, b, bits, gs, w_round="f32")
    W = _dev_weights(gpu, words, s, b, sb)
    xdt = torch.float32 if x32 else torch.bfloat16
    xt = torch.tensor(x, device=gpu).to(xdt)
    lib = _lib.load()
    ws_bytes = lib.gdn_quantized_matmul_workspace_size(_lib.dtype_code(xdt), _lib.dtype_code(_TORCH[sb]),
                                                       M, N, K, bits, gs)
    assert ws_bytes == splits * M * N * 4
    ws = torch.full((ws_bytes // 4,), float("nan"), device=gpu)  # every partial is written
    outs = []
    for w_ptr, w_len in ((None, 0), (_lib.ptr(ws), ws_bytes), (_lib.ptr(ws), ws_bytes),
                         (_lib.ptr(ws), ws_bytes // 2)):
        y = torch.empty(M, N, device=gpu)
        _lib.call("gdn_quantized_matmul", _lib.ptr(xt), _lib.dtype_code(xdt), _lib.ptr(W["weight"]),
                  _lib.ptr(W["scales"]), _lib.ptr(W["biases"]), _lib.dtype_code(W["scales"].dtype),
                  _lib.ptr(y), _lib.GDN_F32, None, M, N, K, bits, gs, w_ptr, w_len, _lib.stream_ptr(gpu))
        outs.append(y.cpu().numpy())
    tol = (1e-4 if x32 else 1e-5) * np.abs(ref).max() + 1e-6
    for y in outs:
        assert np.abs(y - ref).max() <= tol
    assert np.array_equal(outs[1], outs[2])
    assert np.abs(outs[1] - outs[0]).max() <= 1e-5 * np.abs(ref).max() + 1e-6
    # through quantized_linear (its own workspace), in x's dtype
    y = gdn.quantized_linear(xt, W, gdn.QuantScheme(bits, gs))
    np.testing.assert_array_equal(y.float().cpu().numpy(), torch.tensor(outs[1]).to(xdt).float().numpy())


@pytest.mark.parametrize("M,N,K,sb", [
    (64, 2048, 4096, "bf16"),   # the layer's out_proj: 64 column tiles x 4 row blocks
    (40, 2048, 4096, "f16"),    # ragged last row block (8 rows)
    (17, 100, 4096, "f32"),     # one row in the second block; ragged last column tile
])
def test_row_blocks_match_the_oracle_in_one_launch(gpu, M, N, K, sb):
    """17-64 rows of 4-bit group-64 codes with few column tiles run as
    16-row blocks of the 16-row kernel in one launch: no workspace is asked
    for or used (the same bits with and without one), every row block
    meets the oracle's bound, and the residual is added in the store as the
    unfused add of two bf16 arrays."""

    bits, gs = 4, 64
    rng = np.random.default_rng(M * 7 + N)
    words, s, b = _weights(rng, N, K, bits, gs, sb)
    x = R.bf16_round(rng.standard_normal((M, K)).astype(np.float32))
    ref = Q.quantized_matmul(x, words, s, b, bits, gs, w_round="f32")
    W = _dev_weights(gpu, words, s, b, sb)
    xt = torch.tensor(x, device=gpu).to(torch.bfloat16)
    lib = _lib.load()
    assert lib.gdn_quantized_matmul_workspace_size(_lib.GDN_BF16, _lib.dtype_code(_TORCH[sb]), M, N, K,
                                                   bits, gs) == 0
    ws = torch.full((1 << 20,), float("nan"), device=gpu)
    outs = []
    for w_ptr, w_len in ((None, 0), (_lib.ptr(ws), 4 << 20)):
        y = torch.empty(M, N, device=gpu)
        _lib.call("gdn_quantized_matmul", _lib.ptr(xt), _lib.GDN_BF16, _lib.ptr(W["weight"]),
                  _lib.ptr(W["scales"]), _lib.ptr(W["biases"]), _lib.dtype_code(W["scales"].dtype),
                  _lib.ptr(y), _lib.GDN_F32, None, M, N, K, bits, gs, w_ptr, w_len, _lib.stream_ptr(gpu))
        outs.append(y.cpu().numpy())
    assert np.array_equal(outs[0], outs[1])
    assert torch.isnan(ws).all()  # untouched
    tol = 1e-5 * np.abs(ref).max() + 1e-6
    for r0 in range(0, M, 16):
        assert np.abs(outs[0][r0:r0 + 16] - ref[r0:r0 + 16]).max() <= tol, r0
    # bf16 y with a residual: the product rounded, then the sum rounded
    res = torch.randn(M, N, device=gpu).to(torch.bfloat16)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=gpu)
    _lib.call("gdn_quantized_matmul", _lib.ptr(xt), _lib.GDN_BF16, _lib.ptr(W["weight"]),
              _lib.ptr(W["scales"]), _lib.ptr(W["biases"]), _lib.dtype_code(W["scales"].dtype),
              _lib.ptr(y), _lib.GDN_BF16, _lib.ptr(res), M, N, K, bits, gs, None, 0, _lib.stream_ptr(gpu))
    unfused = (torch.tensor(outs[0], device=gpu).to(torch.bfloat16) + res).cpu()
    assert torch.equal(y.cpu(), unfused)


@pytest.mark.parametrize("bits,gs,sb,out", [(4, 64, "bf16", "bf16"), (8, 32, "f16", "f32"),
                                             (4, 128, "f32", "f32")])
def test_dequantize_is_bit_exact(gpu, bits, gs, sb, out):
    rng = np.random.default_rng(bits * gs)
    words, s, b = _weights(rng, 33, 256, bits, gs, sb)
    W = _dev_weights(gpu, words, s, b, sb)
    dense = gdn.dequantize(W, gdn.QuantScheme(bits, gs), _TORCH[out])
    np.testing.assert_array_equal(dense.float().cpu().numpy(),
                                  Q.dequantize(words, s, b, bits, gs, out=out))


def test_non_bf16_activations_use_dense_weights(gpu):
    rng = np.random.default_rng(4)
    words, s, b = _weights(rng, 48, 128, 4, 64, "bf16")
    W = _dev_weights(gpu, words, s, b, "bf16")
    x = rng.standard_normal((5, 128)).astype(np.float32)
    y = gdn.quantized_linear(torch.tensor(x, device=gpu), W, gdn.QuantScheme(4, 64))
    assert y.dtype == torch.float32
    ref = x.astype(np.float64) @ Q.dequantize(words, s, b, 4, 64, out="f32").T
    assert np.abs(y.cpu().numpy() - ref).max() < 1e-4


@pytest.mark.parametrize("M", [64, 600, 2100])
def test_stacked_projection_blocks_match_the_oracle(gpu, M):
    """quantized_linear_split: one quantized launch split into column views
    below 512 rows, one dequantized product split into views below 2048,
    a GEMM per block (packed) from 2048 rows on; either way each block is
    x @ W_block.T."""

    from mlx_lean_moe_amd.quant import concat_quantized, quantized_linear_split

    rng = np.random.default_rng(M)
    sizes, K = [96, 64, 16], 512
    parts = [_weights(rng, n, K, 4, 64, "bf16") for n in sizes]
    stacked = gdn.LinearWeights(concat_quantized([_dev_weights(gpu, *p, "bf16") for p in parts]),
                                gdn.QuantScheme(4, 64))
    x = R.bf16_round(rng.standard_normal((M, K)))
    xt = torch.tensor(x, dtype=torch.float32, device=gpu).to(torch.bfloat16)
    blocks = quantized_linear_split(xt, stacked, sizes)
    exact = _decode_kernel_takes(M, K, 4, 64, "bf16")
    for blk, (words, s, b), n in zip(blocks, parts, sizes):
        assert tuple(blk.shape) == (M, n) and blk.dtype == torch.bfloat16
        assert blk.is_contiguous() == (M >= 2048)
        ref = Q.quantized_matmul(x, words, s, b, 4, 64, w_round="f32" if exact else "bf16")
        assert_bf16_out_close(blk.float().cpu().numpy(), ref)


@pytest.mark.parametrize("T", [70, 600])
def test_layer_with_quantized_projections_matches_dense_weights(gpu, T):
    """The reference's layer test setup: quantized projections against the
    same layer on the dequantized dense weights, decode and prefill (600
    prompt tokens: the stacked input projection as one GEMM per block)."""

    dims = gdn.LinearAttentionDims(2, 4, 128, 128, 4)
    dt = (2, 4, 128, 128)
    H = 256
    rng = np.random.default_rng(21)
    conv_w, A_log, dt_bias, norm_w = layer_params(rng, dt)
    scheme = gdn.QuantScheme(4, 64)
    shapes = {"qkv": dims.conv_dim, "z": dims.value_dim, "a": 4, "b": 4}
    quant, dense = {}, {}
    for name, n in shapes.items():
        words, s, b = _weights(rng, n, H, 4, 64, "bf16")
        quant[name] = _dev_weights(gpu, words, s, b, "bf16")
        dense[name] = torch.tensor(Q.dequantize(words, s, b, 4, 64), dtype=torch.float32,
                                   device=gpu).to(torch.bfloat16)
    words, s, b = _weights(rng, H, dims.value_dim, 4, 64, "bf16")
    quant["out"] = _dev_weights(gpu, words, s, b, "bf16")
    dense["out"] = torch.tensor(Q.dequantize(words, s, b, 4, 64), dtype=torch.float32,
                                device=gpu).to(torch.bfloat16)
    f32 = lambda x: torch.tensor(np.asarray(x, np.float32), device=gpu)
    common = (f32(conv_w)[:, :, None], f32(A_log), f32(dt_bias), f32(norm_w))

    def make(w, q):
        return gdn.Qwen3_5LinearAttention(dims, w["qkv"], w["z"], w["a"], w["b"], common[0],
                                          common[1], common[2], common[3], w["out"], quant=q)

    lq, ld = make(quant, scheme), make(dense, None)
    assert lq._in_stacked is not None  # one launch for the four input projections
    x = torch.tensor(R.bf16_round(rng.standard_normal((T, H))), dtype=torch.float32,
                     device=gpu).to(torch.bfloat16)
    cq, cd = lq.new_cache(torch.bfloat16), ld.new_cache(torch.bfloat16)
    oq, od = lq(x, cq), ld(x, cd)
    assert_bf16_out_close(oq.float().cpu().numpy(), od.float().cpu().numpy().astype(np.float64))
    for t in range(3):
        xt = x[t]
        oq, od = lq(xt, cq), ld(xt, cd)
        assert_bf16_out_close(oq.float().cpu().numpy(), od.float().cpu().numpy().astype(np.float64))


@pytest.mark.parametrize("M,N,K,gs,dt", [
    (1, 2048, 4096, 64, "bf16"),      # the one-row matrix-vector kernel
    (16, 2048, 4096, 64, "bf16"),     # decode kernel, K split (sum kernel stores)
    (32, 12352, 2048, 64, "f32"),     # decode kernel, float32 x and result
    (100, 300, 512, 64, "bf16"),      # dequantize + BLAS, then the add
    (600, 256, 512, 64, "bf16"),      # the same
])
def test_residual_is_the_unfused_add(gpu, M, N, K, gs, dt):
    """residual + x W^T, the product rounded to the result dtype first: bit
    for bit the unfused add of the two arrays (the decoder layer's
    h = rows + attention(...))."""

    rng = np.random.default_rng(M + 3 * N)
    words, s, b = _weights(rng, N, K, 4, gs, "bf16")
    W = _dev_weights(gpu, words, s, b, "bf16")
    xdt = _TORCH[dt]
    x = torch.tensor(rng.standard_normal((M, K)), dtype=torch.float32, device=gpu).to(xdt)
    r = torch.tensor(rng.standard_normal((M, N)), dtype=torch.float32, device=gpu).to(xdt)
    scheme = gdn.QuantScheme(4, gs)
    want = gdn.quantized_linear(x, W, scheme) + r
    got = gdn.quantized_linear(x, W, scheme, residual=r)
    assert torch.equal(got, want)
    if M < 512 and dt == "bf16":
        # through the C ABI, residual aliasing y: y = x W^T + y
        y = r.clone()
        nb = _lib.load().gdn_quantized_matmul_workspace_size(_lib.GDN_BF16, _lib.GDN_BF16, M, N, K, 4, gs)
        ws = torch.empty(max(nb, 16), dtype=torch.uint8, device=gpu)
        _lib.call("gdn_quantized_matmul", _lib.ptr(x), _lib.GDN_BF16, _lib.ptr(W["weight"]),
                  _lib.ptr(W["scales"]), _lib.ptr(W["biases"]), _lib.GDN_BF16, _lib.ptr(y), _lib.GDN_BF16,
                  _lib.ptr(y), M, N, K, 4, gs, _lib.ptr(ws), nb, _lib.stream_ptr(gpu))
        assert torch.equal(y, want)
    with pytest.raises(ValueError, match="residual"):
        gdn.quantized_linear(x, W, scheme, residual=r[:, :-1])


@pytest.mark.parametrize("bits,gs,sb,out", [(2, 64, "bf16", "bf16"), (3, 32, "bf16", "f32"),
                                             (5, 128, "f16", "f16"), (6, 32, "f32", "bf16"),
                                             (6, 64, "bf16", "f32")])
def test_dequantize_every_affine_width_is_bit_exact(gpu, bits, gs, sb, out):
    """2-, 3-, 5- and 6-bit codes (the 3/5/6-bit ones straddle word
    boundaries) against the oracle: s * q + b in float32, one rounding."""

    rng = np.random.default_rng(bits * 1000 + gs)
    words, s, b = _weights(rng, 33, 256, bits, gs, sb)
    W = _dev_weights(gpu, words, s, b, sb)
    dense = gdn.dequantize(W, gdn.QuantScheme(bits, gs), _TORCH[out])
    np.testing.assert_array_equal(dense.float().cpu().numpy(),
                                  Q.dequantize(words, s, b, bits, gs, out=out))


def _fp_weights(rng, gpu, N, K, mode, gs):
    bits = 8 if mode == "mxfp8" else 4
    q = rng.integers(0, 2 ** bits, (N, K))
    if mode == "mxfp8":
        q[(q & 0x7F) == 0x7F] = 0x7E  # no NaN codes
    if mode == "nvfp4":
        scales = rng.integers(0x08, 0x7F, (N, K // gs))  # positive e4m3, none NaN
    else:
        scales = rng.integers(110, 140, (N, K // gs))
    W = {"weight": torch.tensor(Q.pack(q, bits).view(np.int32), device=gpu),
         "scales": torch.tensor(scales.astype(np.uint8), device=gpu)}
    return W, Q.dequantize_fp(Q.pack(q, bits), scales, mode, gs)


@pytest.mark.parametrize("mode,gs,K", [("mxfp4", 32, 256), ("mxfp8", 32, 256), ("nvfp4", 16, 256),
                                        ("nvfp4", 16, 240)])
def test_dequantize_float_schemes_is_bit_exact(gpu, mode, gs, K):
    """mxfp4, mxfp8 and nvfp4 codes (nvfp4 with a row of 240: a 16-code
    tail) against the oracle: value times scale, exact in bf16 and float32."""

    rng = np.random.default_rng(K + gs + len(mode))
    W, ref = _fp_weights(rng, gpu, 37, K, mode, gs)
    scheme = gdn.QuantScheme(8 if mode == "mxfp8" else 4, gs, mode)
    for dt in (torch.bfloat16, torch.float32):
        dense = gdn.dequantize(W, scheme, dt)
        np.testing.assert_array_equal(dense.float().cpu().numpy(), ref)


@pytest.mark.parametrize("M", [1, 64, 600])
@pytest.mark.parametrize("scheme", [(3, 64, "affine"), (6, 32, "affine"), (2, 128, "affine"),
                                    (4, 32, "mxfp4"), (8, 32, "mxfp8"), (4, 16, "nvfp4")])
def test_quantized_linear_every_scheme_matches_oracle(gpu, scheme, M, monkeypatch):
    """The schemes outside gdn_quantized_matmul's kernels through
    quantized_linear, bf16 x, with and without the residual, against x @ W.T
    in float64. Up to 64 rows gdn_quantized_matmul_scheme multiplies the
    packed codes (nothing is dequantized; the exact weights s * q + b, float32
    sums: within the output's bf16 rounding); above, the weights are
    dequantized to bf16 for the vendor BLAS."""

    bits, gs, mode = scheme
    rng = np.random.default_rng(bits + gs + M)
    N, K = 96, 512
    if mode == "affine":
        words, s, b = _weights(rng, N, K, bits, gs, "bf16")
        W = _dev_weights(gpu, words, s, b, "bf16")
        # the exact weights (decode sizes) or the bf16 ones the BLAS multiplies
        w = Q.dequantize(words, s, b, bits, gs, out="f32" if M <= 64 else "bf16")
    else:
        W, w = _fp_weights(rng, gpu, N, K, mode, gs)  # exact in bf16
    calls = []
    call = _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    x = R.bf16_round(rng.standard_normal((M, K)).astype(np.float32))
    xt = torch.tensor(x, device=gpu).to(torch.bfloat16)
    q = gdn.QuantScheme(bits, gs, mode)
    y = gdn.quantized_linear(xt, gdn.LinearWeights(W, q))
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    assert y.dtype == torch.bfloat16 and y.shape == (M, N)
    err = np.abs(y.float().cpu().numpy() - ref)
    if M <= 64:
        assert calls == ["gdn_quantized_matmul_scheme"], calls
        assert (err <= 2.0 ** -8 * np.abs(ref) + 1e-4 * np.abs(ref).max()).all(), err.max()
    else:
        assert "gdn_dequantize" in calls
        assert err.max() <= 1e-2 * np.abs(ref).max()
    r = torch.randn(M, N, device=gpu).to(torch.bfloat16)
    yr = gdn.quantized_linear(xt, gdn.LinearWeights(W, q), residual=r)
    assert torch.equal(yr, y + r)
    parts = quantized_linear_split(xt, gdn.LinearWeights(W, q), [40, 56])
    assert torch.equal(torch.cat(parts, dim=-1), y)


@pytest.mark.parametrize("M", [1, 5, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("scheme,N,K", [((5, 32, "affine"), 200, 480), ((3, 128, "affine"), 70, 768),
                                        ((8, 64, "affine"), 64, 256), ((4, 32, "affine"), 33, 2048),
                                        ((2, 32, "affine"), 96, 352), ((3, 32, "affine"), 80, 224),
                                        ((3, 64, "affine"), 65, 2560), ((5, 64, "affine"), 40, 640),
                                        ((6, 64, "affine"), 48, 192), ((2, 64, "affine"), 17, 4096),
                                        ((6, 128, "affine"), 64, 1024), ((8, 128, "affine"), 96, 512),
                                        ((4, 16, "nvfp4"), 130, 288), ((4, 32, "mxfp4"), 64, 1056),
                                        ((8, 32, "mxfp8"), 129, 320), ((4, 16, "nvfp4"), 24, 4096),
                                        ((8, 32, "mxfp8"), 2048, 1024)])
def test_scheme_matmul_shapes_and_outputs(gpu, scheme, N, K, M):
    """gdn_quantized_matmul_scheme through the C ABI at ragged sizes: every
    row-tile kernel (1-16 rows, 17-64 rows), each code width with runs of
    1, 2 and 4 MFMA blocks per lane (group sizes 32, 64, 128: runs starting
    on a word and runs shifted into place), K split over workgroups (long K,
    few columns), column counts that leave a block part-empty, and the output
    in bfloat16, float16 and float32 with the residual aliasing y; against
    the exact weights in float64 (float32 output: float32 sums)."""

    bits, gs, mode = scheme
    rng = np.random.default_rng(M * 7 + N + K)
    if mode == "affine":
        words, s, b = _weights(rng, N, K, bits, gs, "f16" if bits == 5 else "bf16")
        W = _dev_weights(gpu, words, s, b, "f16" if bits == 5 else "bf16")
        w = Q.dequantize(words, s, b, bits, gs, out="f32")
        sb = _lib.dtype_code(W["scales"].dtype)
    else:
        W, w = _fp_weights(rng, gpu, N, K, mode, gs)
        sb = 0
    x = R.bf16_round(rng.standard_normal((M, K)).astype(np.float32))
    xt = torch.tensor(x, device=gpu).to(torch.bfloat16)
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    mode_code = {"affine": 0, "mxfp4": 1, "mxfp8": 2, "nvfp4": 3}[mode]
    nb = _lib.load().gdn_quantized_matmul_scheme_workspace_size(M, N, K)
    ws = torch.empty(max(nb, 16), dtype=torch.uint8, device=gpu)
    for dt in (torch.float32, torch.bfloat16, torch.float16):
        if dt == torch.float16 and np.abs(ref).max() > 3e4:
            continue  # beyond float16's range (the float formats' large scales)
        r = torch.randn(M, N, device=gpu).to(dt)
        y = r.clone()
        _lib.call("gdn_quantized_matmul_scheme", _lib.ptr(xt), _lib.ptr(W["weight"]), _lib.ptr(W["scales"]),
                  _lib.ptr(W.get("biases")), sb, _lib.ptr(y), _lib.dtype_code(dt), _lib.ptr(y), M, N, K,
                  bits, gs, mode_code, _lib.ptr(ws), nb, _lib.stream_ptr(gpu))
        got = (y.double() - r.double()).cpu().numpy()
        rel = 2.0 ** -20 if dt == torch.float32 else 2.0 ** -7
        assert (np.abs(got - ref) <= rel * (np.abs(ref) + np.abs(r.double().cpu().numpy()))
                + 1e-5 * np.abs(ref).max()).all(), (dt, np.abs(got - ref).max())


@pytest.mark.parametrize("mode,gs,M", [("mxfp4", 32, 1), ("mxfp4", 32, 40), ("mxfp8", 32, 1), ("nvfp4", 16, 64)])
def test_scheme_matmul_special_scale_codes(gpu, mode, gs, M):
    """Scale codes at the ends of their formats through
    gdn_quantized_matmul_scheme: e8m0 255 (NaN) and e4m3 0x7F (NaN) make
    their column NaN, as x times a NaN weight does in the oracle; e8m0 0
    (2^-127) and 1 (2^-126) give their groups weights of at most 6 * 2^-126
    or 448 * 2^-126, whose products vanish beside the other groups'; mxfp8's
    NaN weight codes (0x7F, 0xFF) make their column NaN."""

    rng = np.random.default_rng(17 + M)
    N, K = 64, 256
    bits = 8 if mode == "mxfp8" else 4
    q = rng.integers(0, 2 ** bits, (N, K))
    if mode == "mxfp8":
        q[(q & 0x7F) == 0x7F] = 0x7E
        q[9, 100] = 0x7F
        q[10, 3] = 0xFF
    if mode == "nvfp4":
        scales = rng.integers(0x20, 0x40, (N, K // gs))
        scales[3, 2], scales[4, 0] = 0x7F, 0xFF  # NaN
        scales[5, 1], scales[6, 7] = 0x00, 0x01  # zero, the smallest subnormal
    else:
        scales = rng.integers(120, 130, (N, K // gs))
        scales[3, 2] = 255  # NaN
        scales[5, 1], scales[6, 7] = 0, 1
    scales = scales.astype(np.uint8)
    words = Q.pack(q, bits)
    w = Q.dequantize_fp(words, scales, mode, gs)
    x = R.bf16_round(rng.standard_normal((M, K)).astype(np.float32))
    with np.errstate(invalid="ignore", over="ignore"):
        ref = x.astype(np.float64) @ w.T
    xt = torch.tensor(x, device=gpu).to(torch.bfloat16)
    y = torch.empty(M, N, dtype=torch.float32, device=gpu)
    wt = torch.tensor(words.view(np.int32), device=gpu)
    st = torch.tensor(scales, device=gpu)
    mode_code = {"mxfp4": 1, "mxfp8": 2, "nvfp4": 3}[mode]
    _lib.call("gdn_quantized_matmul_scheme", _lib.ptr(xt), _lib.ptr(wt), _lib.ptr(st), None, 0, _lib.ptr(y),
              _lib.GDN_F32, None, M, N, K, bits, gs, mode_code, None, 0, _lib.stream_ptr(gpu))
    got = y.cpu().numpy()
    nan_cols = np.isnan(ref).any(axis=0)
    assert nan_cols.sum() >= (3 if mode == "mxfp8" else 1)
    assert np.isnan(got[:, nan_cols]).all()
    ok = ~nan_cols
    err = np.abs(got[:, ok] - ref[:, ok])
    assert (err <= 2.0 ** -20 * np.abs(ref[:, ok]) + 1e-5 * np.abs(ref[:, ok]).max()).all(), err.max()


def _f32_kernel(x, W, q, residual=None):
    """gdn_quantized_matmul_f32 as quantized_linear calls it, whatever the size
    (small weights stay on the library there)."""
    return _f32_matmul(x, W["weight"], W["scales"], W["biases"], q, W["weight"].shape[0], x.shape[-1], residual)


def _f32_bound(x, words, s, b, bits, gs):
    """Worst-case rounding of gdn_quantized_matmul_f32: its products are
    exact, and every value passes at most 3 gs + 2 float32 sums inside a group
    and 2 G + 20 across the groups (the scaled sum, the bias term, split
    blocks), each off by 2^-24 of the magnitudes it adds."""
    K = x.shape[1]
    centre = 2.0 ** (bits - 1)
    bp = np.repeat(b + centre * s, gs, axis=1).astype(np.float64)
    w = Q.dequantize(words, s, b, bits, gs, out="f32").astype(np.float64)
    mass = np.abs(x).astype(np.float64) @ (np.abs(w - bp) + np.abs(bp)).T
    return (3 * gs + 2 * K // gs + 22) * 2.0 ** -24 * mass


@pytest.mark.parametrize("M,N,K,bits,gs,sb", [
    (33, 300, 512, 4, 64, "bf16"),      # the first count past the decode kernel; ragged columns
    (777, 520, 2048, 4, 64, "bf16"),
    (81, 257, 384, 8, 128, "f32"),      # half a group a step, one row past five tiles
    (200, 2048, 4096, 4, 64, "bf16"),   # K split
    (130, 96, 1024, 4, 32, "f16"),      # an MFMA's k a group
    (64, 40, 64, 8, 32, "f32"),         # a single step
    (3, 512, 192, 4, 64, "bf16"),       # few rows of a K the decode kernel does not take
    (1, 17, 64, 4, 64, "f16"),
])
def test_float32_rows_in_three_bf16_pieces(gpu, M, N, K, bits, gs, sb):
    rng = np.random.default_rng(M * 5 + N)
    words, s, b = _weights(rng, N, K, bits, gs, sb)
    W = _dev_weights(gpu, words, s, b, sb)
    x = (rng.standard_normal((M, K)) * np.exp(rng.uniform(-6, 6, (M, K))) + 0.5).astype(np.float32)
    ref = Q.quantized_matmul(x, words, s, b, bits, gs, w_round="f32")
    assert _lib.load().gdn_quantized_matmul_f32_workspace_size(M, N, K, bits, gs) > 0
    y = _f32_kernel(torch.tensor(x, device=gpu), W, gdn.QuantScheme(bits, gs))
    assert y.dtype == torch.float32
    assert (np.abs(y.cpu().numpy() - ref) <= _f32_bound(x, words, s, b, bits, gs) + 1e-30).all()
    r = torch.tensor(rng.standard_normal((M, N)), dtype=torch.float32, device=gpu)
    got = _f32_kernel(torch.tensor(x, device=gpu), W, gdn.QuantScheme(bits, gs), residual=r)
    assert torch.equal(got, y + r)


@pytest.mark.parametrize("N,K", [(300, 512), (256, 4096)])  # K unsplit and split
def test_float32_rows_outside_the_pieces_range(gpu, N, K):
    """Rows with infinities, NaN, values near the ends of float32's range:
    the float32 weights' sums, element for element as float64 gives them
    (finite where it is finite, the same infinities and NaN)."""
    rng = np.random.default_rng(N)
    words, s, b = _weights(rng, N, K, 4, 64, "bf16")
    W = _dev_weights(gpu, words, s, b, "bf16")
    x = rng.standard_normal((70, K)).astype(np.float32)
    x[3, 5] = np.inf
    x[10, 7], x[10, 9] = np.inf, -np.inf
    x[20, 1] = np.nan
    x[33] = 0
    x[33, 4] = 3.3e38
    x[40] *= np.float32(1e-37)
    x[50] = 0
    x[69] *= np.float32(2.0 ** 99)
    w = Q.dequantize(words, s, b, 4, 64, out="f32").astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref = x.astype(np.float64) @ w.T
    y = _f32_kernel(torch.tensor(x, device=gpu), W, gdn.QuantScheme(4, 64)).cpu().numpy()
    finite = np.isfinite(x).all(axis=1)
    mass = np.abs(x[finite]).astype(np.float64) @ np.abs(w).T
    assert (np.abs(y[finite] - ref[finite]) <= 2 * K * 2.0 ** -24 * mass + 1e-38 * K).all()
    np.testing.assert_array_equal(np.isnan(y[~finite]), np.isnan(ref[~finite]))
    inf = np.isinf(ref)
    np.testing.assert_array_equal(y[inf], ref[inf].astype(np.float32))


@pytest.mark.parametrize("M,N,K,bits,gs,sb", [
    (65, 300, 256, 4, 64, "bf16"),      # one step; ragged columns; the fewest rows
    (112, 128, 512, 4, 32, "f16"),      # a whole 112-row tile, two groups a lane quarter pair
    (113, 130, 768, 4, 128, "bf16"),    # an odd step count, half a group a wave
    (200, 2048, 4096, 4, 64, "bf16"),   # K split over the grid
    (130, 257, 1024, 8, 64, "f32"),
    (220, 100, 2048, 8, 32, "bf16"),    # the most groups the LDS holds
    (100, 64, 1024, 4, 32, "f32"),      # the same in float32
])
def test_rows_above_the_decode_sizes(gpu, M, N, K, bits, gs, sb):
    """65 to 511 bf16 rows: x times the weights rounded to bf16, with and
    without a workspace to split K in, within float32 sums of the float64
    product: at most K + 20 roundings of 2^-24 of the magnitudes added."""
    from mlx_lean_moe_amd.quant import _mid_rows, workspace_bytes

    assert _mid_rows(M, N, K, gs, _TORCH[sb])
    rng = np.random.default_rng(M * 3 + N)
    words, s, b = _weights(rng, N, K, bits, gs, sb)
    W = _dev_weights(gpu, words, s, b, sb)
    x = R.bf16_round(rng.standard_normal((M, K)))
    w = Q.dequantize(words, s, b, bits, gs, out="bf16").astype(np.float64)
    ref = x.astype(np.float64) @ w.T
    bound = (K + 20) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T)
    xt = torch.tensor(x, dtype=torch.float32, device=gpu).to(torch.bfloat16)
    nbytes = workspace_bytes(torch.bfloat16, _TORCH[sb], M, N, K, bits, gs)
    assert nbytes > 0 or N != 2048
    for ws in (None, torch.empty(nbytes, dtype=torch.uint8, device=gpu) if nbytes else None):
        y = torch.empty(M, N, device=gpu)
        _lib.call("gdn_quantized_matmul_rows", _lib.ptr(xt), _lib.GDN_BF16, _lib.ptr(W["weight"]), _lib.ptr(W["scales"]),
                  _lib.ptr(W["biases"]), _lib.dtype_code(W["scales"].dtype), _lib.ptr(y), _lib.GDN_F32, None, M, N, K,
                  bits, gs, _lib.ptr(ws), nbytes if ws is not None else 0, _lib.stream_ptr(xt.device))
        assert (np.abs(y.cpu().numpy() - ref) <= bound).all()
    r = torch.tensor(rng.standard_normal((M, N)), dtype=torch.float32, device=gpu).to(torch.bfloat16)
    y = gdn.quantized_linear(xt, W, gdn.QuantScheme(bits, gs))
    assert (np.abs(y.float().cpu().numpy() - ref) <= bound + 2.0 ** -8 * np.abs(ref)).all()
    assert torch.equal(gdn.quantized_linear(xt, W, gdn.QuantScheme(bits, gs), residual=r), y + r)


@pytest.mark.parametrize("mode,bits,gs", [("mxfp4", 4, 32), ("mxfp8", 8, 32), ("nvfp4", 4, 16), ("affine", 3, 32),
                                          ("affine", 5, 64), ("affine", 6, 32), ("affine", 2, 128)])
@pytest.mark.parametrize("out", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("shift", [0, 1])
def test_dequantize_into_any_alignment(gpu, mode, bits, gs, out, shift):
    """Every code under every scale code (NaN and the smallest among them),
    rows that end inside a word pair, outputs on and off 16 bytes, and nothing
    written beyond the output."""
    rng = np.random.default_rng(bits + gs + shift)
    K, N = 3 * max(gs, 32), 256
    q = rng.integers(0, 2 ** bits, (N, K))
    q[:, :2 ** min(bits, 4)] = np.arange(2 ** min(bits, 4))
    if mode == "affine":
        s = R.bf16_round(rng.standard_normal((N, K // gs)))
        b = R.bf16_round(rng.standard_normal((N, K // gs)))
        ref = Q.dequantize(Q.pack(q, bits), s, b, bits, gs, out=out)
        scales, biases = (torch.tensor(v, dtype=torch.float32, device=gpu) for v in (s, b))
    else:
        s = np.repeat(np.arange(256)[:, None], K // gs, 1)
        with np.errstate(all="ignore"):
            ref = torch.tensor(Q.dequantize_fp(Q.pack(q, bits), s, mode, gs)).float().to(_TORCH[out]).float().numpy()
        scales, biases = torch.tensor(s.astype(np.uint8), device=gpu), None
    w = torch.tensor(Q.pack(q, bits).view(np.int32), device=gpu)
    buf = torch.full((N * K + 16,), 7.0, dtype=_TORCH[out], device=gpu)
    _lib.call("gdn_dequantize", _lib.ptr(w), _lib.ptr(scales), _lib.ptr(biases), _lib.GDN_F32, _lib.ptr(buf[shift:]),
              _lib.dtype_code(buf.dtype), N, K, bits, gs, {"affine": 0, "mxfp4": 1, "mxfp8": 2, "nvfp4": 3}[mode],
              _lib.stream_ptr(buf.device))
    got = buf.float().cpu().numpy()
    np.testing.assert_array_equal(got[shift:shift + N * K].reshape(N, K), ref)
    assert (got[:shift] == 7).all() and (got[shift + N * K:] == 7).all()


def test_products_under_transforms_stay_on_torch(gpu):
    """float32 rows and narrow bf16 products that are differentiated, run
    under vmap or carry a tangent give what torch's product of the
    dequantized weights gives there, as calls the kernels do not see."""
    rng = np.random.default_rng(9)
    words, s, b = _weights(rng, 48, 256, 4, 64, "bf16")
    W = _dev_weights(gpu, words, s, b, "bf16")
    scheme = gdn.QuantScheme(4, 64)
    for dtype in (torch.float32, torch.bfloat16):
        dense = gdn.dequantize(W, scheme, dtype)
        x = torch.tensor(rng.standard_normal((100, 256)), dtype=dtype, device=gpu)
        xg = x.clone().requires_grad_()
        gdn.quantized_linear(xg, W, scheme).float().sum().backward()
        want = dense.float().sum(0).expand(100, 256)
        assert (xg.grad.float() - want).abs().max() <= (2 ** -7 if dtype is torch.bfloat16 else 1e-5) * want.abs().max()
        with torch.no_grad():
            assert gdn.quantized_linear(xg, W, scheme).grad_fn is None
        with torch.autograd.forward_ad.dual_level():
            y = gdn.quantized_linear(torch.autograd.forward_ad.make_dual(x, x), W, scheme)
            assert torch.equal(torch.autograd.forward_ad.unpack_dual(y).tangent, x @ dense.T)
    x = torch.tensor(rng.standard_normal((3, 40, 256)), dtype=torch.float32, device=gpu)
    got = torch.vmap(lambda r: gdn.quantized_linear(r, W, scheme))(x)
    ref = x @ gdn.dequantize(W, scheme, torch.float32).T
    assert (got - ref).abs().max() <= 1e-5 * ref.abs().max()


@pytest.mark.parametrize("N,K", [(300, 512), (256, 4096)])
def test_float32_rows_times_scales_out_of_range(gpu, N, K):
    """Infinite, NaN and huge float32 scales and biases reach exactly the
    columns they belong to, with the infinities and NaN of the float32
    weights."""
    rng = np.random.default_rng(N + 1)
    words, s, b = _weights(rng, N, K, 4, 64, "f32")
    s, b = np.array(s, np.float32), np.array(b, np.float32)
    s[3, 1], s[70, 0], b[100, 2], s[N - 1, 0], b[N - 1, 0] = np.inf, np.nan, -np.inf, 1e30, 1e30
    W = _dev_weights(gpu, words, s, b, "f32")
    x = rng.standard_normal((70, K)).astype(np.float32)
    q = Q.unpack(words, 4).astype(np.float64)
    with np.errstate(all="ignore"):
        w = (np.repeat(s, 64, 1).astype(np.float64) * q + np.repeat(b, 64, 1)).astype(np.float32).astype(np.float64)
        ref = x.astype(np.float64) @ w.T
    y = _f32_kernel(torch.tensor(x, device=gpu), W, gdn.QuantScheme(4, 64)).cpu().numpy()
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    np.testing.assert_array_equal(np.isposinf(y), np.isposinf(ref))
    np.testing.assert_array_equal(np.isneginf(y), np.isneginf(ref))
    ok = np.isfinite(w).all(axis=1)
    mass = np.abs(x).astype(np.float64) @ np.abs(w[ok]).T
    assert (np.abs(y[:, ok] - ref[:, ok]) <= 2 * K * 2.0 ** -24 * mass).all()


@pytest.mark.parametrize("rows", [65, 128, 224, 384, 448])
@pytest.mark.parametrize("N,K", [(2048, 4096), (4096, 4096), (12352, 4096)])
def test_kept_copies_are_multiplied_above_the_decode_sizes(gpu, rows, N, K, monkeypatch):
    """Narrow or deep weights whose bf16 copy is kept: no call reads the codes
    above 64 rows, and the result is the library's product of the copy."""
    rng = np.random.default_rng(rows)
    scheme = gdn.QuantScheme(4, 64)
    W = {"weight": torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), dtype=torch.int32, device=gpu),
         "scales": torch.full((N, K // 64), 0.01, dtype=torch.bfloat16, device=gpu),
         "biases": torch.full((N, K // 64), -0.08, dtype=torch.bfloat16, device=gpu)}
    kept = gdn.LinearWeights(W, scheme).with_dense()
    x = torch.tensor(rng.standard_normal((rows, K)), dtype=torch.float32, device=gpu).to(torch.bfloat16)
    with monkeypatch.context() as m:
        m.setattr(_lib, "call", lambda name, *a: pytest.fail(f"{name} called"))
        y = gdn.quantized_linear(x, kept)
        blocks = quantized_linear_split(x, kept, [N - 64, 64])
    assert torch.equal(y, x @ kept.dense.T)
    assert torch.equal(torch.cat(blocks, dim=-1), y)
    # the codes' result: the same weights in float32 sums of another order
    plain = gdn.quantized_linear(x, W, scheme).double()
    mass = x.double().abs() @ kept.dense.double().abs().T
    assert ((y.double() - plain).abs() <= 2.0 ** -8 * plain.abs() + 2 * (K + 20) * 2.0 ** -24 * mass).all()


@pytest.mark.parametrize("M,N,K,bits,gs", [(66, 2048, 4096, 4, 64), (200, 2048, 4096, 8, 64), (130, 1000, 2048, 4, 32),
                                           (448, 2048, 4096, 4, 64)])
def test_rows_above_the_decode_sizes_split_k_only_where_asked(gpu, M, N, K, bits, gs):
    """gdn_quantized_matmul_rows splits K in a workspace (every partial block
    is written, the sum is the same each time, half a workspace splits less);
    gdn_quantized_matmul and gdn_quantized_matmul_noalloc do not, and agree bit
    for bit whatever workspace the first one is given."""
    rng = np.random.default_rng(M + K)
    words, s, b = _weights(rng, N, K, bits, gs, "bf16")
    W = _dev_weights(gpu, words, s, b, "bf16")
    x = R.bf16_round(rng.standard_normal((M, K)))
    w = Q.dequantize(words, s, b, bits, gs, out="bf16").astype(np.float64)
    ref = x.astype(np.float64) @ w.T
    bound = (K + 20) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T)
    xt = torch.tensor(x, dtype=torch.float32, device=gpu).to(torch.bfloat16)
    nbytes = _lib.load().gdn_quantized_matmul_rows_workspace_size(_lib.GDN_BF16, M, N, K, bits, gs)
    assert nbytes >= 2 * M * N * 4

    def run(name, ws_bytes):
        y = torch.empty(M, N, device=gpu)
        ws = torch.full((max(ws_bytes, 4) // 4,), float("nan"), device=gpu)
        tail = () if name.endswith("noalloc") else (_lib.ptr(ws) if ws_bytes else None, ws_bytes)
        _lib.call(name, _lib.ptr(xt), _lib.GDN_BF16, _lib.ptr(W["weight"]), _lib.ptr(W["scales"]),
                  _lib.ptr(W["biases"]), _lib.GDN_BF16, _lib.ptr(y), _lib.GDN_F32, None, M, N, K, bits, gs, *tail,
                  _lib.stream_ptr(xt.device))
        assert (np.abs(y.cpu().numpy() - ref) <= bound).all()
        return y

    whole = run("gdn_quantized_matmul_noalloc", 0)
    for ws_bytes in (0, nbytes, 4 * nbytes):
        assert torch.equal(run("gdn_quantized_matmul", ws_bytes), whole)
    assert torch.equal(run("gdn_quantized_matmul_rows", 0), whole)
    split = run("gdn_quantized_matmul_rows", nbytes)
    assert torch.equal(run("gdn_quantized_matmul_rows", nbytes), split) and not torch.equal(split, whole)
    run("gdn_quantized_matmul_rows", nbytes // 2)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("edge", [79, 80, 99, 126])
def test_float32_rows_at_the_ends_of_their_range_do_not_overflow(gpu, bits, edge):
    """Rows of +-2^edge against scales and biases just inside their limits and
    codes whose weights s q + b cancel to zero, or to one scale: the partial
    sums s (q - c) x and b' x must not overflow where the product does not."""
    N, K, gs = 70, 4096, 128
    s = 2.0 ** 15
    top = 2 ** bits - 1
    rng = np.random.default_rng(edge)
    q0 = np.array([0, top, 8])[np.arange(N) % 3]
    q = np.repeat(q0[:, None], K, 1)
    q[:, 5] += np.where(q0 == top, -1, 1)  # one weight of a row is a scale, the others zero
    W = {"weight": torch.tensor(Q.pack(q, bits).view(np.int32), device=gpu),
         "scales": torch.full((N, K // gs), s, device=gpu),
         "biases": torch.tensor(np.repeat(-q0[:, None] * s, K // gs, 1), dtype=torch.float32, device=gpu)}
    x = np.ldexp(np.where(rng.random((40, K)) < 0.3, -1.0, 1.0), edge).astype(np.float32)
    x[::2] = np.abs(x[::2])
    x[:, 5] = np.ldexp(1.0, edge - 20)
    y = _f32_kernel(torch.tensor(x, device=gpu), W, gdn.QuantScheme(bits, gs)).cpu().numpy()
    want = np.ldexp(np.where(q0 == top, -1.0, 1.0), edge - 5)
    # float32 sums of the cancelling terms |q0| s |x| of each of K elements
    assert np.isfinite(y).all()
    if edge >= 80:
        np.testing.assert_array_equal(y, np.repeat(want[None], 40, 0).astype(np.float32))
    else:
        assert (np.abs(y - want) <= K * 2.0 ** -24 * K * s * 2 * 2 ** bits * 2.0 ** edge).all()


@pytest.mark.parametrize("N,K,bits,gs,exact_zero", [(300, 2048, 4, 64, True), (130, 1024, 8, 64, True),
                                                    (130, 1024, 4, 32, False), (70, 4096, 8, 128, False)])
def test_float32_rows_with_outlying_activations_against_small_weights(gpu, N, K, bits, gs, exact_zero):
    """A few activations 10^9 times the rest where the weights are zero (or the
    codes nearest to zero): within float32 sums of |x| |w|. A group's two terms
    s (q - c) and b' = b + c s are at most 3 |w| together for c = round(-b / s)
    (test_float32_rows_in_three_bf16_pieces counts the sums)."""
    rng = np.random.default_rng(N + K)
    M, G = 50, K // gs
    s = R.bf16_round(rng.uniform(0.005, 0.01, (N, G))) * np.where(rng.random((N, G)) < 0.5, -1, 1)
    q0 = rng.integers(0, 2 ** bits, (N, G))
    b = -q0 * s if exact_zero else -(q0 + rng.uniform(-0.5, 0.5, (N, G))) * s
    s, b = s.astype(np.float32), b.astype(np.float32)
    q = rng.integers(0, 2 ** bits, (N, K))
    big = rng.choice(K, 5, replace=False)
    q[:, big] = q0[:, big // gs]
    W = {"weight": torch.tensor(Q.pack(q, bits).view(np.int32), device=gpu), "scales": torch.tensor(s, device=gpu),
         "biases": torch.tensor(b, device=gpu)}
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[:, big] *= np.float32(1e9)
    w = np.repeat(s, gs, 1).astype(np.float64) * q + np.repeat(b, gs, 1)
    if exact_zero:
        assert (w[:, big] == 0).all()
    y = _f32_kernel(torch.tensor(x, device=gpu), W, gdn.QuantScheme(bits, gs)).cpu().numpy()
    mass = np.abs(x).astype(np.float64) @ np.abs(w).T
    bound = (3 * gs + 2 * G + 22) * 2.0 ** -24 * 3 * mass
    assert (np.abs(y - x.astype(np.float64) @ w.T) <= bound).all()


@pytest.mark.parametrize("M,N,K,bits,gs,sb", [
    (33, 300, 512, 4, 64, "bf16"),      # ragged rows and columns
    (81, 257, 384, 8, 128, "f32"),      # one row past five tiles
    (200, 2048, 4096, 4, 64, "bf16"),   # K split
    (50, 96, 1024, 4, 32, "f16"),
    (16, 40, 64, 8, 32, "f32"),         # a single step
])
def test_whole_prompts_of_float32_rows_outside_the_pieces_range(gpu, M, N, K, bits, gs, sb):
    """Every row (and one column block) out of the pieces' range: infinities,
    NaN, and rows of 2^85 (at most 2^2 of them a value, times 2^28 and 128 of
    the column block's weights: below 2^127) and 2^-125, whose products are
    subnormal, within float32 sums of the float64 product."""
    rng = np.random.default_rng(M + N)
    words, s, b = _weights(rng, N, K, bits, gs, sb)
    if sb == "f32":
        s[0, 0], b[0, 0] = np.float32(2.0 ** 20), np.float32(-3 * 2.0 ** 20)
    W = _dev_weights(gpu, words, s, b, sb)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[0::4] *= np.float32(2.0 ** 85)
    x[1::4] *= np.float32(2.0 ** -125)
    x[2::4, 3] = np.inf
    x[3::4, 5] = np.nan
    w = Q.dequantize(words, s, b, bits, gs, out="f32").astype(np.float64)
    with np.errstate(invalid="ignore"):
        ref = x.astype(np.float64) @ w.T
        mass = np.abs(x).astype(np.float64) @ np.abs(w).T
    y = _f32_kernel(torch.tensor(x, device=gpu), W, gdn.QuantScheme(bits, gs)).cpu().numpy()
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    np.testing.assert_array_equal(y[2::4], ref[2::4].astype(np.float32))
    for rows in (slice(0, None, 4), slice(1, None, 4)):
        assert (np.abs(y[rows] - ref[rows]) <= 2 * K * 2.0 ** -24 * mass[rows] + K * 2.0 ** -149).all()


def test_float32_rows_outside_the_pieces_range_cost_a_bounded_multiple(gpu):
    """A prompt whose rows all hold an infinity takes about 4 times an ordinary
    one's time (the float32 matrix cores have a quarter of the bf16 ones' rate
    for a piece), not a serial chain a row: 20 times leaves room for noise."""
    M, N, K = 300, 2048, 2048
    rng = np.random.default_rng(1)
    words, s, b = _weights(rng, N, K, 4, 64, "bf16")
    W = _dev_weights(gpu, words, s, b, "bf16")
    x = torch.randn(M, K, device=gpu)
    far = x.clone()
    far[:, 3] = float("inf")
    times = []
    for t in (x, far):
        best = float("inf")
        for _ in range(5):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(4):
                _f32_kernel(t, W, gdn.QuantScheme(4, 64))
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end))
        times.append(best)
    assert times[1] < 20 * times[0], times


def test_dequantize_of_more_threads_than_a_grid_dimension_holds(gpu):
    """2^35 2-bit codes, 8 a thread: 2^32 threads, the first count that one grid
    dimension does not hold, checked in blocks over the whole output."""
    N, K, gs = 1 << 20, 1 << 15, 128
    if torch.cuda.mem_get_info(gpu)[0] < 100 << 30:
        pytest.skip("needs 75 GB of device memory")
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 16), dtype=torch.int32, device=gpu)
    s = torch.rand(N, K // gs, device=gpu).to(torch.bfloat16)
    out = gdn.dequantize({"weight": w, "scales": s, "biases": s}, gdn.QuantScheme(2, gs), torch.bfloat16)
    shifts = torch.arange(0, 32, 2, device=gpu, dtype=torch.int32)
    for n0 in range(0, N, N // 64):
        for n in (n0, n0 + N // 64 - 8):
            q = ((w[n:n + 8, :, None] >> shifts) & 3).reshape(8, K).float()
            sc = s[n:n + 8].float().repeat_interleave(gs, 1)
            assert torch.equal(out[n:n + 8], (sc * q + sc).to(torch.bfloat16)), n
    del w, s, out, q, sc
    torch.cuda.empty_cache()  # 75 GB that no other test needs


@pytest.mark.parametrize("M,N,K,bits,gs,sb", [
    # the 128 x 128 tiles: K not in steps of 256 (quantized_linear sends N >= 4096 there)
    (100, 300, 320, 4, 64, "bf16"),
    (130, 4100, 320, 8, 64, "f32"),
    (129, 4160, 1088, 4, 32, "f16"),
    (511, 4097, 192, 8, 32, "bf16"),
    # the same where the 112-row tiles would need a second round of workgroups
    (256, 12352, 256, 4, 64, "bf16"),
    (385, 12352, 512, 8, 128, "bf16"),
    (449, 12352, 1024, 8, 32, "bf16"),
    # the 112-row tiles, up to their last row count; two rounds of them
    (225, 1000, 512, 4, 64, "bf16"),
    (300, 4096, 256, 8, 32, "f16"),
    (511, 700, 768, 8, 128, "f32"),
    (300, 12352, 1024, 4, 128, "bf16"),
    # K split over the grid
    (448, 2048, 4096, 4, 64, "bf16"),
    (511, 1000, 4096, 8, 64, "f16"),
])
def test_every_kernel_of_65_to_511_rows(gpu, M, N, K, bits, gs, sb):
    """x times the bf16-rounded weights, whichever kernel takes the rows: the
    float32 result within K + 20 roundings of the magnitudes added, a float16 and
    a bfloat16 one with a residual in y itself as the unfused add of the rounded
    product, and quantized_linear's with the residual bit for bit that add."""
    rng = np.random.default_rng(M + N + K)
    words, s, b = _weights(rng, N, K, bits, gs, sb)
    W = _dev_weights(gpu, words, s, b, sb)
    x = R.bf16_round(rng.standard_normal((M, K)))
    xt = torch.tensor(x, dtype=torch.float32, device=gpu).to(torch.bfloat16)
    w = torch.tensor(Q.dequantize(words, s, b, bits, gs, out="bf16"), dtype=torch.float64, device=gpu)
    ref = xt.double() @ w.T
    bound = (K + 20) * 2.0 ** -24 * (xt.double().abs() @ w.abs().T)
    lib = _lib.load()
    nbytes = lib.gdn_quantized_matmul_rows_workspace_size(_lib.dtype_code(_TORCH[sb]), M, N, K, bits, gs)
    ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=gpu)

    def run(y, residual=None):
        _lib.call("gdn_quantized_matmul_rows", _lib.ptr(xt), _lib.GDN_BF16, _lib.ptr(W["weight"]),
                  _lib.ptr(W["scales"]), _lib.ptr(W["biases"]), _lib.dtype_code(_TORCH[sb]), _lib.ptr(y),
                  _lib.dtype_code(y.dtype), _lib.ptr(residual), M, N, K, bits, gs, _lib.ptr(ws), nbytes,
                  _lib.stream_ptr(gpu))
        return y

    y32 = run(torch.empty(M, N, device=gpu))
    assert ((y32.double() - ref).abs() <= bound).all()
    for dt in (torch.float16, torch.bfloat16):
        r = torch.randn(M, N, device=gpu).to(dt)
        y = r.clone()
        assert torch.equal(run(y, y), y32.to(dt) + r)
    q = gdn.QuantScheme(bits, gs)
    y = gdn.quantized_linear(xt, W, q)
    assert ((y.double() - ref).abs() <= bound + 2.0 ** -8 * ref.abs()).all()
    assert torch.equal(gdn.quantized_linear(xt, W, q, residual=r), y + r)


@pytest.mark.parametrize("M,N,K,kernel", [(100, 256, 1024, False), (513, 2048, 1024, True), (512, 2048, 1024, False),
                                          (40, 1024, 4096, True)])
def test_float32_rows_take_the_kernel_by_the_weights_size(gpu, M, N, K, kernel, monkeypatch):
    rng = np.random.default_rng(M)
    words, s, b = _weights(rng, N, K, 4, 64, "bf16")
    W = _dev_weights(gpu, words, s, b, "bf16")
    x = rng.standard_normal((M, K)).astype(np.float32)
    calls = []
    call = _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    y = gdn.quantized_linear(torch.tensor(x, device=gpu), W, gdn.QuantScheme(4, 64)).cpu().numpy()
    assert calls == ["gdn_quantized_matmul_f32" if kernel else "gdn_dequantize"]
    w = Q.dequantize(words, s, b, 4, 64, out="f32").astype(np.float64)
    assert (np.abs(y - x.astype(np.float64) @ w.T) <= K * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).T)).all()
