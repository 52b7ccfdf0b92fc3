"""One row given for every token (``row.expand(M, K)``, row stride 0): bitwise
the call on its contiguous copy, in both arithmetic modes, over the kernels of
1-128 tokens -- decode with and without a K split, packed activations,
batch-decode and prefill tiles."""

from __future__ import annotations

import pytest
import torch

from jeeves_amd import synthetic
from jeeves_amd.fp8 import FP8Linear, FP8SwiGLU, fp8_matmul, fp8_matmul_quantized, fp8_matmul_w8a16, tile_weight
from jeeves_amd.fp8_weights import quantize_rows

pytestmark = pytest.mark.gpu


def row(K: int, seed: int) -> torch.Tensor:
    return synthetic.activations_outliers(1, K, seed).cuda()


# 256 and 496 rows split K, the latter beside packed activations; 12288 and
# 16384 columns: packed rows at most counts; 24576 rows: prefill tiles.
@pytest.mark.parametrize("N,K", [(256, 4096), (496, 16896), (1024, 4096), (4096, 12288), (6144, 4096), (5008, 2560),
                                 (24576, 4096)])
@pytest.mark.parametrize("M", [1, 2, 8, 16, 17, 24, 33, 64, 65, 128])
@pytest.mark.parametrize("matmul", [fp8_matmul, fp8_matmul_w8a16])
def test_one_row_for_every_token(N, K, M, matmul):
    print(f"broadcast rows {matmul.__name__} N={N} K={K} M={M}", flush=True)
    wq, sw = quantize_rows(synthetic.weight(N, K, 40).cuda())
    x = row(K, 41).expand(M, K) if M > 1 else row(K, 41).expand(8, K)[:1]
    assert x.stride(0) == 0
    want = matmul(x.clone(memory_format=torch.contiguous_format).reshape(M, K), wq, sw)
    assert torch.equal(matmul(x, wq, sw), want)
    assert torch.equal(matmul(x, tile_weight(wq), sw, tiled=True), want)


@pytest.mark.parametrize("activations", ["fp8", "bf16"])
@pytest.mark.parametrize("B,T", [(1, 3), (2, 8), (3, 8), (4, 32)])
def test_modules_take_one_row_for_every_token(B, T, activations):
    hidden, inter = 2560, 1152
    gate_up, down = FP8Linear(hidden, 2 * inter, device="cuda"), FP8Linear(inter, hidden, device="cuda")
    gate_up.load_weight(synthetic.weight(2 * inter, hidden, 42).cuda())
    down.load_weight(synthetic.weight(hidden, inter, 43).cuda())
    mlp = FP8SwiGLU(gate_up, down)
    mlp.set_activations(activations)
    x = row(hidden, 44).expand(B, T, hidden)
    for m in (gate_up, mlp):
        assert torch.equal(m(x), m(x.contiguous()))


@pytest.mark.parametrize("M", [1, 8, 33, 200])
def test_broadcast_codes(M):
    """Codes of one row, and weight codes of one row, broadcast over the rows."""
    N, K = 1040, 2560
    wq, sw = quantize_rows(synthetic.weight(N, K, 45).cuda())
    xq, sx = quantize_rows(row(K, 46))
    x = xq.expand(M, K) if M > 1 else xq.expand(8, K)[:1]
    want = fp8_matmul_quantized(xq.repeat(M, 1), sx.repeat(M), wq, sw)
    assert torch.equal(fp8_matmul_quantized(x, sx.repeat(M), wq, sw), want)
    one = wq[5:6].expand(N, K)
    assert torch.equal(fp8_matmul_quantized(x, sx.repeat(M), one, sw), fp8_matmul_quantized(x, sx.repeat(M), one.contiguous(), sw))
    assert torch.equal(fp8_matmul(row(K, 46).expand(M, K), one, sw), fp8_matmul(row(K, 46).expand(M, K), one.contiguous(), sw))
