"""Edges of the tile that the two-copy quantizers load: rows and columns that end inside a thread's share, rows that divide
plainly next to rows that do not."""
import pytest
import torch

import mdy_triton_amd as m
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("M,K", [(1, 8), (2, 120), (3, 128), (5, 136), (127, 264), (129, 248), (255, 8), (2561, 4096)])
def test_edges(M, K, dtype):
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M * 1000 + K))
    x[M // 2, K - 1] = 2e4                    # beyond the clamp: this row, its column and its block divide and saturate
    x[0, :8] = 0.0
    x = x.to(dtype)
    for got, ref in ((m.quant_input(x.cuda(), False), O.quant_input(x, False)), (m.quant_grad_output(x.cuda()), O.quant_grad_output(x)),
                     (m.quant_weight(x.cuda(), False), O.quant_weight(x, False))):
        for g, r in zip(got, ref):
            assert g.shape == r.shape and torch.equal(g.cpu().contiguous().view(torch.uint8), r.contiguous().view(torch.uint8))
