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
@pytest.mark.parametrize("M,N,K", [(512, 512, 4096), (1000, 1020, 4224), (130, 257, 9600), (1536, 1536, 5120),
                                   (1530, 640, 4736), (2176, 638, 8576)])      # counts that 8 does not divide, short and long slabs
def test_exact_integer_cut_along_k(M, N, K, transposed_scales, fmt):
    from mdy_triton_amd import _lib
    assert _lib.load().mdy_fp8_gemm_rowscaled_workspace_bytes(M, N, K) >= 2 * M * N * 4
    exact_case(M, N, K, fmt, transposed_scales)


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("M,N,K", [(890, 3712, 3072), (250, 1036, 1664), (1000, 2301, 896),      # 128x128 tiles, ring of 3: one tile per CU at most
                                   (2550, 3190, 1024), (7290, 2170, 640), (770, 260, 384), (512, 640, 512)])      # two workgroups per CU
def test_exact_integer_128x128_tiles(M, N, K, fmt):
    exact_case(M, N, K, fmt, transposed_scales=bool(fmt))


@pytest.mark.parametrize("M,N,K", [(890, 1028, 3072), (300, 700, 512), (2550, 3190, 1024)])
def test_exact_integer_128x128_tiles_fp32(M, N, K):
    from mdy_triton_amd import _lib
    lib = _lib.load()
    g = torch.Generator().manual_seed(M + N)
    ai, bi = (torch.randint(-2, 3, (r, K), generator=g) for r in (M, N))
    a, b = (v.float().to(torch.float8_e4m3fn).to(DEV) for v in (ai, bi))
    sa, sb = (torch.full((r, K // 128), 2.0, device=DEV) for r in (M, N))
    c = torch.full((M, N), float("nan"), device=DEV)
    rc = lib.mdy_fp8_gemm_nt_rowscaled_ws(a.data_ptr(), sa.data_ptr(), K // 128, 1, b.data_ptr(), sb.data_ptr(), K // 128, 1, c.data_ptr(), M, N, K, 0, 1,
                                          0, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(c.double(), 4 * (ai.double().to(DEV) @ bi.double().to(DEV).t()))
