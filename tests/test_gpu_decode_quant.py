"""The decode GEMM that quantizes its own activations (1-4 tokens): bitwise the
GEMM on the quantizer's codes, over row-major and tiled weights, k ranges with
short, missing and whole bursts per wave, strided rows, a bias, rows of zeros,
infinities and NaNs, and the fused SwiGLU; at the edges of its dispatch (four
and five tokens, weights of more rounds, narrow weights that split K) both
sides give the same bits."""

from __future__ import annotations

import pytest
import torch

from jeeves_amd import synthetic
from jeeves_amd.fp8 import (FP8Linear, FP8SwiGLU, fp8_matmul, fp8_matmul_quantized, gate_up_swiglu, quantize_swiglu_output,
                            swiglu_quantize, tile_weight)
from jeeves_amd.fp8_weights import quantize_rows

pytestmark = pytest.mark.gpu


def same(a: torch.Tensor, b: torch.Tensor) -> bool:
    return torch.equal(torch.nan_to_num(a.float()), torch.nan_to_num(b.float())) and torch.equal(a.isnan(), b.isnan())


# 128 and 640: waves without steps and with one or two; 2560 and 4224: short
# bursts; 16384: the longest row; 4112 rows up: two tiles per wave, with each
# chunk count (4096 to 16384 columns); 256: a K split and 70000: far more than
# one round of short rows, on the general path.
@pytest.mark.parametrize("N,K", [(1024, 128), (1600, 640), (1040, 2560), (1024, 4096), (5000, 4096), (24576, 4096),
                                 (4112, 4224), (4096, 12288), (1008, 16384), (70000, 512), (256, 4096), (16384, 1024),
                                 (4112, 8192), (4112, 12288), (4112, 16384)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5])
def test_quantizing_gemm_equals_quantizer_and_gemm(N, K, M):
    print(f"quantizing decode GEMM N={N} K={K} M={M}", flush=True)
    wq, sw = quantize_rows(synthetic.weight(min(N, 5000), K, 60 + K).repeat(-(-N // 5000), 1)[:N].cuda())
    bias = synthetic.weight(1, N, 61)[0].cuda()
    x = torch.zeros(M, K + 24, dtype=torch.bfloat16, device="cuda")[:, :K]  # 16-byte aligned rows, not contiguous
    x.copy_(synthetic.activations_outliers(M, K, 62 + M))
    codes, scales = quantize_rows(x)
    for b in (None, bias):
        want = fp8_matmul_quantized(codes, scales, wq, sw, bias=b)
        assert torch.equal(fp8_matmul(x, wq, sw, bias=b), want)
        if N % 16 == 0:
            assert torch.equal(fp8_matmul(x, tile_weight(wq), sw, bias=b, tiled=True), want)


def test_quantizing_gemm_special_rows():
    N, K = 1040, 4096
    wq, sw = quantize_rows(synthetic.weight(N, K, 70).cuda())
    x = synthetic.activations_outliers(4, K, 71)
    x[0, 9] = float("inf")
    x[1] = 0.0
    x[2, K - 1] = float("nan")
    x[3] *= 1e-20
    x = x.cuda()
    for rows in ([0, 1, 2, 3], [1, 3], [2], [0]):
        xs = x[rows].contiguous()
        want = fp8_matmul_quantized(*quantize_rows(xs), wq, sw)
        assert same(fp8_matmul(xs, tile_weight(wq), sw, tiled=True), want), rows


@pytest.mark.parametrize("hidden,inter", [(4096, 12288), (2560, 1152), (640, 256)])
@pytest.mark.parametrize("M", [1, 2, 4, 5])
def test_swiglu_block_of_a_few_tokens(hidden, inter, M):
    gate_up, down = FP8Linear(hidden, 2 * inter, device="cuda"), FP8Linear(inter, hidden, device="cuda")
    gate_up.load_weight(synthetic.weight(2 * inter, hidden, 80).cuda())
    down.load_weight(synthetic.weight(hidden, inter, 81).cuda())
    x = synthetic.activations_outliers(M, hidden, 82 + M).cuda()
    gu = fp8_matmul_quantized(*quantize_rows(x), gate_up.weight, gate_up.scale)
    h = swiglu_quantize(gu[:, :inter], gu[:, inter:], return_h=True)[-1]
    assert torch.equal(gate_up_swiglu(x, gate_up.kernel_weight()[0], gate_up.scale, tiled=True), h)
    codes, scales = quantize_swiglu_output(h, packed=False)
    want = fp8_matmul_quantized(codes, scales, down.weight, down.scale)
    assert torch.equal(FP8SwiGLU(gate_up, down)(x), want)
