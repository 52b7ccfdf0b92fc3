"""The LoRA quantizer with two rows per workgroup (from 1024 rows, 512 above
K = 4096): codes, scales and x A^T bitwise those of the one-row form that
shorter batches of the same rows take, odd row counts and short rows included."""

from __future__ import annotations

import math

import pytest
import torch

from jeeves_amd import synthetic
from jeeves_amd.fp8 import quantize_swiglu_output

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K", [(1024, 128), (1025, 2048), (1039, 4096), (513, 4224), (515, 8192), (527, 12288), (512, 16384)])
def test_two_rows_equal_one_row(M, K):
    print(f"LoRA quantizer M={M} K={K}", flush=True)
    x = synthetic.activations_heavy_tail(M, K, 90 + K)
    x[1, 3], x[2, K - 1], x[M - 1, 0] = float("inf"), float("nan"), -500.0
    x[4] = 0.0
    x = x.cuda()
    a = synthetic.lora_factors(1024, K, 91)[0].cuda()
    codes, scales, t = quantize_swiglu_output(x, lora_a=a, packed=False)
    packed, pscales, pt = quantize_swiglu_output(x, lora_a=a, packed=True)
    same = lambda p, q: torch.equal(torch.nan_to_num(p), torch.nan_to_num(q)) and torch.equal(p.isnan(), q.isnan())  # noqa: E731
    assert same(pscales, scales) and same(pt, t)
    assert torch.equal(packed, quantize_swiglu_output(x, packed=True)[0])
    for lo, hi in ((0, 300), (M - 131, M)):
        c1, s1, t1 = quantize_swiglu_output(x[lo:hi].contiguous(), lora_a=a, packed=False)
        assert torch.equal(codes[lo:hi].view(torch.uint8), c1.view(torch.uint8))
        assert same(scales[lo:hi], s1) and same(t[lo:hi], t1)


@pytest.mark.parametrize("M,K", [(16, 4096), (512, 4096), (2048, 4096), (16, 12288), (300, 12288), (2048, 12288)])
def test_low_rank_product_against_64_bits(M, K):
    """x A^T in fp32 against 64 bits: relative 2-norm within 0.5 u sqrt(levels),
    u = 2^-24. Products are exact; a sum tree over terms of random sign whose
    levels each round once has a relative rms error of 0.41 u per level (a
    rounding's rms over a mantissa's range), adding in quadrature: 9 levels
    across lanes and waves, and a chain of c dot products of pairs, whose
    partial sums grow like sqrt(i), counts as (c + 1) / 2."""
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(92)).to(torch.bfloat16).cuda()
    a = synthetic.lora_factors(1024, K, 93)[0].cuda()
    t = quantize_swiglu_output(x, lora_a=a, packed=False)[2].double()
    want = x.double() @ a.double().t().contiguous()
    err = ((t - want).norm() / want.norm()).item()
    chain = 4 * -(-K // (8 * 256))
    bound = 0.5 * 2.0 ** -24 * math.sqrt(9 + (chain + 1) / 2)
    print(f"t M={M} K={K}: {err:.3g} from 64 bits, bound {bound:.3g}", flush=True)
    assert err <= bound
