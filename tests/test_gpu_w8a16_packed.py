"""The W8A16 decode kernel on activations packed in fragment order: bitwise the
same call on the rows as they are (a workspace without room for the packing),
at the edges of the token tiles and of the rule that packs."""

from __future__ import annotations

import pytest
import torch

from jeeves_amd import _lib, synthetic
from jeeves_amd.fp8 import fp8_matmul_w8a16, tile_weight
from jeeves_amd.fp8_weights import quantize_rows

pytestmark = pytest.mark.gpu


# 4096 x 12288: packed from 17 tokens; 6144 x 4096 and 5008 x 2560: from 33;
# 24576 x 4096 (a wide weight) and 1024 x 4096 (the batch-decode kernel): never.
@pytest.mark.parametrize("N,K", [(24576, 4096), (4096, 12288), (6144, 4096), (5008, 2560), (1024, 4096)])
@pytest.mark.parametrize("M", [16, 17, 31, 32, 33, 48, 64, 128])
@pytest.mark.parametrize("tiled", [True, False])
def test_packed_rows_equal_rows(N, K, M, tiled):
    print(f"W8A16 packed N={N} K={K} M={M} tiled={tiled}", flush=True)
    wq, sw = quantize_rows(synthetic.weight(N, K, 50).cuda())
    w = tile_weight(wq) if tiled else wq
    x = synthetic.activations_outliers(M, K + 8, 51 + M).cuda()[:, :K]
    y = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    L = _lib.lib()
    need = L.jv_w8a16_workspace_bytes(M, N, K)
    pack = (M + 15) // 16 * 16 * K * 2
    decode = M <= 64 and N not in (24576, 1024)
    packs = decode and M > 16 and N * K >= (8 << 20 if M > 32 else 48 << 20)
    if packs:
        assert need == pack  # these sizes do not split K on the decode kernels
        ws = torch.zeros(256, dtype=torch.uint8, device="cuda")
        _lib.check(L.jv_w8a16_linear(x.data_ptr(), x.stride(0), w.data_ptr(), 0 if tiled else K, sw.data_ptr(), None,
                                     y.data_ptr(), N, M, N, K, ws.data_ptr(), 256, None, 0,
                                     torch.cuda.current_stream().cuda_stream))
        assert torch.equal(fp8_matmul_w8a16(x, w, sw, tiled=tiled), y)
    else:
        assert decode is False or need < pack
        want = (x.float() @ wq.float().t()) * sw
        got = fp8_matmul_w8a16(x, w, sw, tiled=tiled).float()
        # one rounding to bf16 (2^-9 relative) and fp32 sums in another order
        assert ((got - want).norm() / want.norm()).item() < 4e-3
