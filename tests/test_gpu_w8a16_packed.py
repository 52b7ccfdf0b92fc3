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


# Token counts at which each weight's activations are packed; 24576 x 4096 (a
# wide weight) and 1024 x 4096 (the batch-decode kernel): never. 496 x 16896 splits K.
PACKED = {(24576, 4096): (), (4096, 12288): (31, 32, 33, 48, 64), (6144, 4096): (48, 64), (5008, 2560): (64,),
          (1024, 4096): (), (10240, 3072): (31, 32, 33, 48, 64), (496, 16896): (31, 32, 33, 48, 64)}


@pytest.mark.parametrize("N,K", list(PACKED))
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
    splits = L.jv_fp8_split_for(1, N, K, torch.cuda.get_device_properties(0).multi_processor_count)
    partials = (splits * M * N * 4 + 255) // 256 * 256 if splits > 1 else 0
    if M in PACKED[N, K]:
        assert need == (pack + 255) // 256 * 256 + partials
        ws = torch.zeros(max(partials, 256), dtype=torch.uint8, device="cuda")
        counters = torch.zeros(4096, dtype=torch.int32, device="cuda")
        _lib.check(L.jv_w8a16_linear(x.data_ptr(), x.stride(0), w.data_ptr(), 0 if tiled else K, sw.data_ptr(), None,
                                     y.data_ptr(), N, M, N, K, ws.data_ptr(), ws.numel(), _lib.counters_ptr(counters),
                                     counters.numel(), torch.cuda.current_stream().cuda_stream))
        assert torch.equal(fp8_matmul_w8a16(x, w, sw, tiled=tiled), y)
    else:
        assert need < pack
        want = (x.float() @ wq.float().t()) * sw
        got = fp8_matmul_w8a16(x, w, sw, tiled=tiled).float()
        # one rounding to bf16 (2^-9 relative) and fp32 sums in another order
        assert ((got - want).norm() / want.norm()).item() < 4e-3


# (tokens, N, K, us on rows as they are, us packed) on both sides of the lines
# of the packing rule; graphs over 1 GiB of rotated weights.
ROWS_OR_PACKED = [
    (17, 10240, 8192, 33.2, 34.4), (24, 10240, 8192, 40.3, 34.4), (24, 12288, 2048, 12.5, 12.9), (28, 12288, 2048, 13.6, 12.9),
    (20, 16384, 4096, 19.7, 20.4), (24, 16384, 4096, 20.9, 20.5), (32, 16384, 1024, 8.2, 9.1), (28, 4096, 12288, 24.2, 21.8),
    (32, 4096, 12288, 26.4, 21.9), (17, 4096, 12288, 18.3, 21.7), (32, 8192, 8192, 22.4, 23.8), (33, 4096, 8192, 20.4, 19.3),
    (33, 4096, 3072, 9.5, 10.6), (44, 4096, 3072, 11.0, 10.6), (48, 4096, 1024, 5.7, 6.1), (33, 12288, 1024, 10.5, 9.9),
    (33, 6144, 12288, 32.6, 33.2), (36, 6144, 12288, 34.2, 33.2), (36, 6144, 4096, 13.7, 14.2), (44, 6144, 4096, 15.3, 14.3),
    (33, 16384, 4096, 25.2, 25.6), (36, 16384, 4096, 26.6, 25.6), (36, 16384, 1024, 9.3, 10.2), (64, 4096, 2048, 10.3, 8.4),
    (64, 16384, 2048, 22.9, 19.8), (49, 6144, 2560, 12.8, 12.2), (49, 8192, 2048, 11.0, 12.3),
]


def test_packs_where_that_is_faster():
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the timings are of 256 CUs")
    for M, N, K, rows, packed in ROWS_OR_PACKED:
        packs = _lib.lib().jv_w8a16_workspace_bytes(M, N, K) >= (M + 15) // 16 * 16 * K * 2
        assert packs == (packed < rows), (M, N, K)
