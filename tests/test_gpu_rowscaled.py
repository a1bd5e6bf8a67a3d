"""The row-scaled GEMM on every kernel its dispatch picks, bit for bit: integer operands and power-of-two scales make every
product and partial sum exact in fp32, so any order of summation gives the float64 result."""
import pytest
import torch

from mdy_triton_amd import _lib
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


# MDY_FORM_...: 128x128 tiles alone on a CU and two per CU, 128x256, 256x256, the plain loop
RING3, TWO, T128X256, T256X256, PLAIN = 7, 8, 10, 12, 14


def runs(M, N, K, form, workspace=1):
    """The kernel that a case means, so that a later rule cannot send it elsewhere unnoticed; (form, slabs of K)."""
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        got = _lib.load().mdy_fp8_gemm_rowscaled_form(M, N, K, workspace)
        assert got & 255 == form, (M, N, K, got)
        return got >> 8


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("M,N,K,form", [(4090, 3336, 384, T256X256),      # one round, ragged rows and columns
                                        (4358, 5519, 256, T256X256),      # more than one per CU: LDS handed from tile to tile; odd N
                                        (644, 5433, 640, T128X256), (3074, 4879, 640, T128X256),      # less than a round, more than one
                                        (250, 1036, 256, PLAIN), (1990, 3300, 384, PLAIN),
                                        (4352, 4360, 128, PLAIN), (5504, 4735, 128, T256X256),       # one K block, several rounds
                                        (130, 1032, 640, TWO), (250, 1036, 512, TWO)])
def test_exact_integer(M, N, K, form, fmt):
    assert not runs(M, N, K, form)
    exact_case(M, N, K, fmt, transposed_scales=bool(fmt))


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("transposed_scales", [False, True])      # row-major (what Fp8Linear passes) and column-major
@pytest.mark.parametrize("M,N,K", [(512, 512, 4096), (1000, 1020, 4224), (130, 257, 9600), (1536, 1536, 5120),
                                   (1530, 640, 4736), (2176, 638, 8576)])      # counts that 8 does not divide, short and long slabs
def test_exact_integer_cut_along_k(M, N, K, transposed_scales, fmt):
    slabs = runs(M, N, K, T128X256)
    assert slabs is None or slabs >= 2
    exact_case(M, N, K, fmt, transposed_scales)


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("M,N,K,form", [(890, 3712, 3072, RING3), (250, 1036, 1664, RING3), (1000, 2301, 896, RING3),
                                        (2550, 3190, 1024, TWO), (7290, 2170, 640, TWO), (770, 260, 384, TWO), (512, 640, 512, TWO)])
def test_exact_integer_128x128_tiles(M, N, K, form, fmt):
    assert not runs(M, N, K, form)
    exact_case(M, N, K, fmt, transposed_scales=bool(fmt))


@pytest.mark.parametrize("M,N,K,form", [(890, 1028, 3072, RING3), (300, 700, 512, TWO), (2550, 3190, 1024, TWO),
                                        (644, 5433, 640, T128X256), (4090, 3336, 384, T256X256), (250, 1036, 256, PLAIN)])
def test_exact_integer_fp32(M, N, K, form):
    lib = _lib.load()
    runs(M, N, K, form, workspace=0)
    g = torch.Generator().manual_seed(M + N)
    ai, bi = (torch.randint(-2, 3, (r, K), generator=g) for r in (M, N))
    a, b = (v.float().to(torch.float8_e4m3fn).to(DEV) for v in (ai, bi))
    sa, sb = (torch.full((r, K // 128), 2.0, device=DEV) for r in (M, N))
    c = torch.full((M, N), float("nan"), device=DEV)
    rc = lib.mdy_fp8_gemm_nt_rowscaled_ws(a.data_ptr(), sa.data_ptr(), K // 128, 1, b.data_ptr(), sb.data_ptr(), K // 128, 1, c.data_ptr(), M, N, K, 0, 1,
                                          0, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(c.double(), 4 * (ai.double().to(DEV) @ bi.double().to(DEV).t()))


@pytest.mark.parametrize("M,N,K,form", [(890, 1028, 3072, RING3), (300, 700, 512, TWO), (644, 5433, 640, T128X256), (4090, 3336, 384, T256X256)])
def test_scale_products_are_rounded_once_and_keep_special_values(M, N, K, form):
    """One product per result, 1 * 1, in the second of the K blocks: the result is the fp32 product of the two scales to the bit, among them
    denormal products, zeros, infinities and NaN (the matrix instruction that multiplies scales rounds and propagates as v_mul_f32)."""
    lib = _lib.load()
    runs(M, N, K, form, workspace=0)
    g = torch.Generator().manual_seed(K)
    a, b = (torch.zeros(r, K) for r in (M, N))
    a[:, 200] = b[:, 200] = 1.0
    a, b = (v.to(torch.float8_e4m3fn).to(DEV) for v in (a, b))

    def scales(r):
        s = torch.ones(r, K // 128)
        v = torch.rand(r, generator=g) + 0.5
        v[: r // 2] *= torch.exp2(torch.randint(-75, -60, (r // 2,), generator=g).float())      # products from 2^-152 to 2^-118
        v[r - 40:r - 32], v[r - 20], v[r - 10], v[r - 5] = 0.0, float("inf"), float("nan"), 2.0 ** -140
        s[:, 1] = v
        return s, v

    (sa, va), (sb, vb) = scales(M), scales(N)
    c = torch.full((M, N), 7.0, device=DEV)
    sa, sb = sa.to(DEV), sb.to(DEV)
    rc = lib.mdy_fp8_gemm_nt_rowscaled_ws(a.data_ptr(), sa.data_ptr(), K // 128, 1, b.data_ptr(), sb.data_ptr(), K // 128, 1, c.data_ptr(), M, N, K, 0, 1,
                                          0, 0, torch.cuda.current_stream().cuda_stream)
    ref = va[:, None] * vb[None, :]
    assert rc == 0 and torch.equal(c.cpu().nan_to_num(nan=-1.0), ref.nan_to_num(nan=-1.0))
