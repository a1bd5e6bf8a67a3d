"""Narrow weights with 8 columns per workgroup, and the reduction of K slabs in its widths and slab counts."""
import pytest
import torch

import mdy_triton_amd as m
from mdy_triton_amd import _lib

pytestmark = pytest.mark.gpu


def slabs_are(form, slabs):
    """The plan cuts K into as many slabs as a case is meant to have, so that a later rule cannot change that unnoticed."""
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert form >> 8 == slabs, form


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


# one launch; slabs whose reduction takes eight, four and one columns per thread
@pytest.mark.parametrize("M,N,K,slabs", [(777, 2112, 7168, 0), (777, 2116, 7168, 0), (777, 2110, 7168, 0), (777, 2113, 7168, 0),
                                         (245, 3664, 5120, 2), (628, 1712, 9728, 3), (598, 1384, 12160, 4), (200, 4096, 7168, 4), (256, 7168, 18432, 3),
                                         (637, 1252, 7552, 2), (793, 592, 3840, 3), (238, 3788, 11648, 4), (300, 1028, 4096, 4), (48, 2048, 7168, 4),
                                         (100, 1024, 7168, 8), (189, 852, 9216, 9), (243, 564, 15104, 14),
                                         (548, 1767, 6528, 2), (662, 833, 9984, 3), (842, 451, 13056, 4), (202, 721, 9472, 9), (194, 405, 15104, 14)])
@pytest.mark.parametrize("biased", [False, True])
def test_reduction(M, N, K, slabs, biased):
    """bf16 results are the fp32 ones rounded once, whatever width the reduction has."""
    slabs_are(_lib.load().mdy_fp8_gemm_form(M, N, K, 1), slabs)
    q, s, w, ws = _operands(M, N, K)
    bias = torch.randn(N, generator=torch.Generator(device="cuda").manual_seed(1), device="cuda").bfloat16() if biased else None
    out = [m.fp8_gemm(q, s, w.contiguous(), ws, out_dtype=dt, bias=bias) for dt in (torch.bfloat16, torch.float32)]
    assert torch.equal(out[0], out[1].bfloat16())


@pytest.mark.parametrize("M,N,K,slabs", [(161, 1536, 3712, 5), (441, 1472, 17408, 5), (82, 2432, 6016, 6), (97, 1536, 3968, 7), (441, 1470, 17408, 5), (213, 576, 8832, 8),
                                         (123, 574, 7040, 8)])
def test_counts_of_slabs(M, N, K, slabs):
    """Whole numbers: exact in any order, over however many slabs (5 to 8 all in flight at once)."""
    slabs_are(_lib.load().mdy_fp8_gemm_form(M, N, K, 1), slabs)
    g = torch.Generator(device="cuda").manual_seed(slabs)
    a, b = (torch.randint(-2, 3, (r, K), generator=g, device="cuda").float() for r in (M, N))
    s, ws = torch.ones(M, K // 128, device="cuda"), torch.ones(-(-N // 128), K // 128, device="cuda")
    bias = torch.randint(-9, 10, (N,), generator=g, device="cuda").bfloat16()
    ref = a @ b.t() + bias.float()
    for dtype in (torch.float32, torch.bfloat16):
        assert torch.equal(m.fp8_gemm(a.to(torch.float8_e4m3fn), s, b.to(torch.float8_e4m3fn), ws, out_dtype=dtype, bias=bias), ref.to(dtype))


@pytest.mark.parametrize("M,N,K,slabs", [(128, 2432, 2688, 5), (384, 3584, 9344, 6), (128, 1536, 3968, 7), (256, 3456, 15104, 8), (256, 1920, 5760, 9), (384, 832, 9216, 12),
                                         (256, 960, 14208, 16)])
def test_counts_of_row_scaled_slabs(M, N, K, slabs):
    from mdy_triton_amd import fp8_kernel
    slabs_are(_lib.load().mdy_fp8_gemm_rowscaled_form(M, N, K, 1), slabs)
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.randint(-2, 3, (r, K), generator=g, device="cuda").float() for r in (M, N))
    sa, sb = (torch.ones(r, K // 128, device="cuda") for r in (M, N))
    got = fp8_kernel.fp8_matmul(a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn), sa, sb, have_w=False)
    assert torch.equal(got, (a @ b.t()).to(got.dtype))
