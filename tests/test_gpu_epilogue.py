"""The tile kernels write bf16 results through LDS in whole rows when the row length allows it and fp32 results straight from
registers: the two must agree to the bit (the fp32 result rounded once) wherever a tile ends inside the matrix."""
import pytest
import torch

from mdy_triton_amd import _lib
from tests import problems as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _gemm(a, a_s, b, b_s, bias, dtype):
    (M, K), N = a.shape, b.size(0)
    out = torch.full((M + 1, N), float("nan"), device=DEV, dtype=dtype)      # the row behind the result must stay untouched
    _lib.check(_lib.load().mdy_fp8_gemm_nt(a.data_ptr(), a_s.data_ptr(), K // 128, 1, b.data_ptr(), b_s.data_ptr(), out.data_ptr(),
                                           bias.data_ptr() if bias is not None else None, M, N, K, 0 if dtype == torch.bfloat16 else 1,
                                           None), "gemm")
    torch.cuda.synchronize()
    assert torch.isnan(out[M].float()).all()
    return out[:M]


# ragged rows and columns that are and are not a multiple of 8
SIZES = [(4100, 5000, 256), (3590, 4612, 128), (1100, 6008, 1024), (12700, 392, 1024), (4090, 1544, 1024), (2040, 2056, 256), (2040, 1036, 384), (1000, 1096, 256),
         (65, 136, 128), (300, 520, 384), (200, 7168, 256), (33000, 120, 1024), (33000, 100, 1024), (1348, 3564, 1280), (1348, 3560, 1280), (1055, 424, 1408),
         (1055, 420, 1408), (680, 2712, 1024), (822, 2380, 1024)]


def test_sizes_take_every_tile():
    """64x64, 64x128, 128x64, 128x128 one and two per CU, 128x192, 128x256, 256x128 and 256x256 tiles with a 128x256 remainder."""
    got = {_lib.load().mdy_fp8_gemm_form(*size, 0) for size in SIZES}
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert got == {4, 5, 6, 7, 8, 9, 10, 11, 13}


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("with_bias", [False, True])
def test_bf16_rows_equal_rounded_fp32(M, N, K, with_bias):
    g = torch.Generator().manual_seed(M + N + K)
    a, a_s = O.act_quant(P.activations("normal", M, K, M))
    b = (torch.randn(N, K, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn).to(DEV)
    b_s = (torch.rand((N + 127) // 128, K // 128, generator=g) * 1e-3 + 1e-4).to(DEV)
    bias = torch.randn(N, generator=g).bfloat16().to(DEV) if with_bias else None
    a, a_s = a.to(DEV), a_s.to(DEV)
    assert torch.equal(_gemm(a, a_s, b, b_s, bias, torch.bfloat16), _gemm(a, a_s, b, b_s, bias, torch.float32).bfloat16())


@pytest.mark.parametrize("M,N,K", [(130, 200, 384), (250, 1036, 128), (4090, 3336, 256)])      # plain loop twice, scheduled tiles
def test_row_scaled_bf16_rows_equal_rounded_fp32(M, N, K):
    g = torch.Generator().manual_seed(M + N)
    a, b = [(torch.randn(r, K, generator=g) * 100).clamp(-448, 448).to(torch.float8_e4m3fn).to(DEV) for r in (M, N)]
    a_s, b_s = [(torch.rand(r, K // 128, generator=g) * 1e-3 + 1e-4).to(DEV) for r in (M, N)]
    out = {}
    for dtype in (torch.bfloat16, torch.float32):
        out[dtype] = torch.full((M, N), float("nan"), device=DEV, dtype=dtype)
        _lib.check(_lib.load().mdy_fp8_gemm_nt_rowscaled(a.data_ptr(), a_s.data_ptr(), K // 128, 1, b.data_ptr(), b_s.data_ptr(), K // 128, 1,
                                                         out[dtype].data_ptr(), M, N, K, 0, 0 if dtype == torch.bfloat16 else 1, None), "rowscaled")
    torch.cuda.synchronize()
    assert torch.equal(out[torch.bfloat16], out[torch.float32].bfloat16())
