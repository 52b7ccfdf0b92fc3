"""Outputs over the activations (C ABI): jv_fp8_linear and the fused SwiGLU
read all of x before they store, at the token counts whose GEMM quantizes for
itself (1-4) and above; bitwise the call with an output of its own, with y on
x's rows, between them and on part of them. (The no-allocation form is in
test_zz_no_alloc.py, whose first test needs its first call.)"""

from __future__ import annotations

import pytest
import torch

from jeeves_amd import _lib, synthetic
from jeeves_amd.fp8 import fp8_matmul, gate_up_swiglu, tile_weight
from jeeves_amd.fp8_weights import quantize_rows

pytestmark = pytest.mark.gpu


def scratch(M, N, K):
    L = _lib.lib()
    n = L.jv_fp8_linear_workspace_bytes(M, N, K, 0)
    return torch.empty(n, dtype=torch.uint8, device="cuda"), torch.zeros(65536, dtype=torch.int32, device="cuda")


def stream() -> int:
    return torch.cuda.current_stream().cuda_stream


# (row stride of the shared buffer, first element of y in it)
@pytest.mark.parametrize("ld,offset", [(4096, 0), (8192, 4096), (4096, 2048), (4352, 256)])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 16])
def test_linear_over_its_activations(M, ld, offset):
    print(f"in-place linear M={M} ld={ld} offset={offset}", flush=True)
    N = K = 4096
    wq, sw = quantize_rows(synthetic.weight(N, K, 20).cuda())
    w = tile_weight(wq)
    x = synthetic.activations_outliers(M, K, 21 + M).cuda()
    want = fp8_matmul(x, w, sw, tiled=True)
    buf = torch.zeros(M + 2, ld, dtype=torch.bfloat16, device="cuda")
    buf[:M, :K] = x
    y = buf.view(-1)[offset:].as_strided((M, N), (ld, 1))
    ws, counters = scratch(M, N, K)
    _lib.check(_lib.lib().jv_fp8_linear(buf.data_ptr(), ld, w.data_ptr(), 0, sw.data_ptr(), None, None, None, 0, 0.0,
                                        y.data_ptr(), ld, M, N, K, ws.data_ptr(), ws.numel(), _lib.counters_ptr(counters),
                                        counters.numel(), stream()))
    assert torch.equal(y, want)


@pytest.mark.parametrize("part", ["h", "amax"])
@pytest.mark.parametrize("M", [1, 2, 4, 5])
def test_swiglu_over_its_activations(M, part):
    print(f"in-place SwiGLU M={M} {part}", flush=True)
    I, K = 2048, 4096
    wq, sw = quantize_rows(synthetic.weight(2 * I, K, 30).cuda())
    w = tile_weight(wq)
    x = synthetic.activations_outliers(M, K, 31 + M).cuda()
    want, amax = gate_up_swiglu(x, w, sw, tiled=True, amax=True)
    buf = x.clone()
    h = buf.view(-1)[:M * I].view(M, I) if part == "h" else torch.empty(M, I, dtype=torch.bfloat16, device="cuda")
    maxima = buf.view(torch.int16).view(-1)[-M * I // 16:].view(M, I // 16) if part == "amax" else torch.empty_like(amax)
    ws, counters = scratch(M, 2 * I, K)
    _lib.check(_lib.lib().jv_fp8_linear_swiglu(buf.data_ptr(), K, w.data_ptr(), 0, sw.data_ptr(), None, None, None, 0, 0.0,
                                               h.data_ptr(), I, maxima.data_ptr(), M, I, K, ws.data_ptr(), ws.numel(),
                                               _lib.counters_ptr(counters), counters.numel(), stream()))
    assert torch.equal(h, want) and torch.equal(maxima, amax)
