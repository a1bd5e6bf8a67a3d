"""The row-scaled GEMM on every kernel its dispatch picks, bit for bit: integer operands and power-of-two scales make every
product and partial sum exact in fp32, so any order of summation gives the float64 result."""
import pytest
import torch

from mdy_triton_amd import fp8_kernel as FK

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def exact_case(M, N, K, fmt, transposed_scales):
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)
    KB = K // 128
    dtype = (torch.float8_e4m3fn, torch.float8_e5m2)[fmt]
    ai, bi = (torch.randint(-2, 3, (r, K), generator=g) for r in (M, N))
    ea, eb = (torch.randint(-2, 3, (r, KB), generator=g) for r in (M, N))
    a, b = (v.double().to(DEV).view(-1, KB, 128) * torch.exp2(e.double()).to(DEV)[:, :, None] for v, e in ((ai, ea), (bi, eb)))
    ref = a.view(M, K) @ b.view(N, K).t()
    sa, sb = (torch.exp2(e.float()).to(DEV) for e in (ea, eb))
    if transposed_scales:
        sa, sb = (s.t().contiguous().t() for s in (sa, sb))
    got = FK._matmul_rowscaled(ai.float().to(dtype).to(DEV), sa, bi.float().to(dtype).to(DEV), sb, M, N, K, torch.device(DEV), fmt)
    assert torch.equal(got, ref.float().bfloat16())


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("M,N,K", [(4090, 3336, 384),      # 256x256 tiles, one round, ragged rows and columns
                                   (4352, 4360, 128),      # 256x256 tiles, more than one per CU, one K block
                                   (130, 1032, 640),       # 128x256 tiles
                                   (250, 1036, 512)])      # the plain loop
def test_exact_integer(M, N, K, fmt):
    exact_case(M, N, K, fmt, transposed_scales=bool(fmt))


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("transposed_scales", [False, True])      # row-major (what Fp8Linear passes) and column-major
@pytest.mark.parametrize("M,N,K", [(512, 512, 4096), (1000, 1020, 4224), (130, 257, 9600), (1536, 1536, 5120)])
def test_exact_integer_cut_along_k(M, N, K, transposed_scales, fmt):
    from mdy_triton_amd import _lib
    assert _lib.load().mdy_fp8_gemm_rowscaled_workspace_bytes(M, N, K) >= 2 * M * N * 4
    exact_case(M, N, K, fmt, transposed_scales)
