"""Narrow weights with 8 columns per workgroup, and the reduction of K slabs in its widths and slab counts."""
import pytest
import torch

import mdy_triton_amd as m

pytestmark = pytest.mark.gpu


def _operands(M, N, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, s = m.act_quant(torch.randn(M, K, generator=g, device="cuda").bfloat16())
    NB = -(-N // 128)
    wq, ws = m.weight_quant_block((torch.randn(NB * 128, K, generator=g, device="cuda") * 0.05).bfloat16(), dtype=torch.float8_e4m3fn)
    return q, s, wq[:N], ws


@pytest.mark.parametrize("M", [2, 9, 16])
@pytest.mark.parametrize("N,K", [(1592, 1024), (1600, 7168), (2041, 2048), (2048, 7168), (2048, 128), (2056, 1024)])
def test_columns_of_a_narrow_weight(M, N, K):
    """The K blocks are shared out among the waves whatever the columns: the same bits as inside a wider weight."""
    q, s, w, ws = _operands(M, 4096, K)
    whole = m.fp8_gemm(q, s, w, ws, out_dtype=torch.bfloat16)
    part = m.fp8_gemm(q, s, w[:N].contiguous(), ws[:-(-N // 128)].contiguous(), out_dtype=torch.bfloat16)
    assert torch.equal(part, whole[:, :N])


@pytest.mark.parametrize("M,N,K", [(777, 2112, 7168), (777, 2116, 7168), (777, 2110, 7168), (777, 2113, 7168), (100, 1024, 7168), (48, 2048, 7168),
                                   (200, 4096, 7168), (300, 1028, 4096), (256, 7168, 18432)])
@pytest.mark.parametrize("biased", [False, True])
def test_reduction(M, N, K, biased):
    """bf16 results are the fp32 ones rounded once, whatever width the reduction has."""
    q, s, w, ws = _operands(M, N, K)
    bias = torch.randn(N, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda").bfloat16() if biased else None
    out = [m.fp8_gemm(q, s, w.contiguous(), ws, out_dtype=dt, bias=bias) for dt in (torch.bfloat16, torch.float32)]
    assert torch.equal(out[0], out[1].bfloat16())
