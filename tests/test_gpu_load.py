"""FP8Linear.load_weight through the one-pass intake kernel: codes and scales
bitwise those of the numpy oracle's quantize_rows, the tiled copy bitwise the
layout formula's, at the edges of the kernel's unit counts and for rows that
hold zeros of both signs, infinities and NaNs; what the kernel does not take
goes the general way to the same result."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from jeeves_amd import _lib, synthetic
from jeeves_amd.fp8 import FP8Linear, tile_weight

pytestmark = pytest.mark.gpu


def special_rows(N: int, K: int, seed: int) -> torch.Tensor:
    """fp32 [N,K] ~ N(0, 0.02) whose first rows hold the values where a
    quantizer can go wrong."""
    g = torch.Generator().manual_seed(seed)
    w = torch.randn(N, K, generator=g) * 0.02
    w[0] = 0.0
    w[1, ::2] = -0.0
    w[2] *= 1e-14  # below the scale's clamp
    w[3, K - 1] = float("inf")
    w[4, 5] = float("nan")
    w[5, K // 2] = -3e38
    w[6, :] = 3.0
    w[7, 1] = 1e-40
    return w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K", [(16, 128), (32, 1024), (48, 2048), (16, 2176), (32, 4096), (16, 4224), (32, 8192),
                                 (16, 8320), (32, 12288), (16, 16384), (21, 4096), (9, 272), (16, 16512)])
def test_load_weight_equals_oracle(N, K, dtype):
    w = special_rows(N, K, 7 * N + K).to(dtype)
    m = FP8Linear(K, N, device="cuda")
    m.load_weight(w.cuda())
    codes, scale = oracle.quantize_rows(w.float().numpy())
    # a NaN row's codes are NaN codes of either sign; its scale is a NaN
    got, gs = m.weight.view(torch.uint8).cpu().numpy(), m.scale.cpu().numpy()
    nan = np.isnan(scale)
    assert np.array_equal(nan, np.isnan(gs)) and nan.sum() == 1
    assert np.array_equal(gs[~nan], scale[~nan])
    assert np.array_equal(got[~nan], codes[~nan])
    assert ((got[nan] & 0x7F) == 0x7F).all()
    assert m.tiled == (N % 16 == 0 and K % 128 == 0)
    if m.tiled:
        assert torch.equal(m.kernel_weight()[0].cpu(), tile_weight(m.weight.view(torch.uint8).cpu()))


@pytest.mark.parametrize("form", ["strided", "transposed", "fp16", "broadcast", "cpu"])
def test_load_weight_forms(form):
    """Weights that the kernel does not take as they are, against the same values in the form that it takes."""
    N, K = 64, 1024
    w = (synthetic.weight(N, K, 11).float() * 8).half().float()
    if form == "broadcast":
        w = w[:1].expand(N, K)
    given = {"strided": torch.nn.functional.pad(w, (0, 12)).cuda()[:, :K], "transposed": w.t().contiguous().cuda().t(),
             "fp16": w.half().cuda(), "broadcast": w[:1].cuda(), "cpu": w}[form]
    a, b = (FP8Linear(K, N, device="cuda") for _ in range(2))
    a.load_weight(given)
    b.load_weight(w.contiguous().cuda())
    assert torch.equal(a.weight.view(torch.uint8), b.weight.view(torch.uint8)) and torch.equal(a.scale, b.scale)
    assert torch.equal(a.kernel_weight()[0], b.kernel_weight()[0])


def test_load_weight_into_a_part_reaches_the_merged_module():
    parts = [FP8Linear(256, n, device="cuda") for n in (32, 48)]
    for i, p in enumerate(parts):
        p.load_weight(synthetic.weight(p.out_features, 256, 20 + i).cuda())
    merged = FP8Linear.concatenated(parts)
    new = synthetic.weight(48, 256, 30).cuda()
    parts[1].load_weight(new)
    alone = FP8Linear(256, 48, device="cuda")
    alone.load_weight(new)
    assert torch.equal(merged.kernel_weight()[0][32:], alone.kernel_weight()[0])
    assert torch.equal(merged.weight.view(torch.uint8)[32:], alone.weight.view(torch.uint8))
    x = synthetic.activations_outliers(4, 256, 31).cuda()
    assert torch.equal(merged(x)[:, 32:], alone(x))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("where", ["weight", "scale", "tiled_codes"])
def test_load_weight_from_memory_of_its_own_buffers(where, dtype):
    """The checkpoint's weight may lie where the module keeps its codes: it is
    read before anything is written."""
    N, K = 512, 4096
    w = synthetic.weight(N, K, 32).to(dtype).cuda()
    want = FP8Linear(K, N, device="cuda")
    want.load_weight(w)
    pool = torch.zeros(N * K * 8, dtype=torch.uint8, device="cuda")
    m = FP8Linear(K, N, device="cuda")
    own = getattr(m, where)
    n = own.numel() * own.element_size()
    m._buffers[where] = pool[1024:1024 + n].view(own.dtype).view(own.shape)
    given = pool[:N * K * w.element_size()].view(dtype).view(N, K)
    given.copy_(w)
    m.load_weight(given)
    assert torch.equal(m.weight.view(torch.uint8), want.weight.view(torch.uint8)) and torch.equal(m.scale, want.scale)
    assert torch.equal(m.kernel_weight()[0], want.kernel_weight()[0])


def test_load_weight_leaves_other_tensors_to_load_codes():
    """Calls that load_codes alone may answer: its override on an instance, a
    parametrized weight, inference tensors outside inference mode (refused),
    a weight that torch negates on reading."""
    N, K = 64, 1024
    w = synthetic.weight(N, K, 33).cuda()
    want = FP8Linear(K, N, device="cuda")
    want.load_weight(w)

    m = FP8Linear(K, N, device="cuda")
    seen = []
    m.load_codes = lambda codes, scale: seen.append((codes, scale))
    m.load_weight(w)
    assert torch.equal(seen[0][0].view(torch.uint8), want.weight.view(torch.uint8)) and torch.equal(seen[0][1], want.scale)

    class Flip(torch.nn.Module):
        def forward(self, codes):
            return (codes.view(torch.uint8) ^ 0x80).view(codes.dtype)

    m = FP8Linear(K, N, device="cuda")
    m.load_weight(w)
    torch.nn.utils.parametrize.register_parametrization(m, "weight", Flip(), unsafe=True)
    m.load_weight(w * 2)  # written to the parametrization's result, which nothing keeps
    assert torch.equal(m.kernel_weight()[0], tile_weight(want.weight.view(torch.uint8) ^ 0x80))

    with torch.inference_mode():
        m = FP8Linear(K, N, device="cuda")
        m.load_weight(w)
        assert torch.equal(m.weight.view(torch.uint8), want.weight.view(torch.uint8))
    with pytest.raises(RuntimeError, match="[Ii]nference"):
        m.load_weight(w)

    m = FP8Linear(K, N, device="cuda")
    m.load_weight(torch._neg_view(w.float()))
    assert torch.equal(m.weight.view(torch.uint8) ^ 0x80, want.weight.view(torch.uint8))


def test_load_weight_refuses_what_it_cannot_take():
    L, buf = _lib.lib(), torch.zeros(64 * 256, dtype=torch.uint8, device="cuda")
    p = buf.data_ptr()
    for args in ((p, 256, 3, 16, 256, p, 256), (p, 256, 2, 16, 250, p, 256), (p + 2, 256, 2, 16, 256, p, 256),
                 (p, 128, 2, 16, 256, p, 256), (p, 20000, 2, 16, 20000, p, 20000)):
        assert L.jv_fp8_load_weight(*args, p, None, None) == _lib.JV_ERR_VALUE
    assert L.jv_fp8_load_weight(p, 256, 2, 24, 256, p, 256, p, p, None) == _lib.JV_ERR_VALUE
