"""The general GEMM entry point: a bias added after rounding gives the bits of add_bias on the product on every kernel the
dispatch picks, and e5m2 operands take the K split and the transposed-scale copy like e4m3fn ones."""
import pytest
import torch

from mdy_triton_amd import _lib
from mdy_triton_amd.fp8 import add_bias

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _operands(M, N, K, fmt):
    g = torch.Generator().manual_seed(M + N + K + fmt)
    KB = K // 128
    dtype = (torch.float8_e4m3fn, torch.float8_e5m2)[fmt]
    ai, bi = (torch.randint(-2, 3, (r, K), generator=g) for r in (M, N))
    ea = torch.randint(-2, 3, (M, KB), generator=g)
    eb = torch.randint(-2, 3, ((N + 127) // 128, KB), generator=g)
    a = ai.double().to(DEV).view(M, KB, 128) * torch.exp2(ea.double()).to(DEV)[:, :, None]
    b = bi.double().to(DEV).view(N, KB, 128) * torch.exp2(eb.double()).to(DEV)[torch.arange(N) // 128][:, :, None]
    ref = (a.view(M, K) @ b.view(N, K).t()).float()
    return (ai.float().to(dtype).to(DEV), torch.exp2(ea.float()).to(DEV), bi.float().to(dtype).to(DEV), torch.exp2(eb.float()).to(DEV),
            torch.randn(N, generator=g).bfloat16().to(DEV), ref)


def _call(a, a_s, b, b_s, bias, mode, fmt):
    (M, K), N = a.shape, b.size(0)
    L = _lib.load()
    ws = torch.empty(max(16, L.mdy_fp8_gemm_workspace_bytes(M, N, K)), dtype=torch.uint8, device=DEV)
    c = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    _lib.check(L.mdy_fp8_gemm_nt_ex(a.data_ptr(), a_s.data_ptr(), K // 128, 1, b.data_ptr(), b_s.data_ptr(), c.data_ptr(),
                                    bias.data_ptr() if bias is not None else None, mode, M, N, K, fmt, 0, ws.data_ptr(), ws.numel(), None), "ex")
    torch.cuda.synchronize()
    return c


CUT = [(64, 1024, 4224), (128, 1030, 4224), (70, 600, 8320), (637, 1252, 7552), (662, 833, 9984)]      # split along K


@pytest.mark.parametrize("fmt", [0, 1])
@pytest.mark.parametrize("M,N,K", [(1, 1000, 4224), (16, 2050, 1024), (20, 26000, 256), (48, 16640, 256), (40, 6500, 384),      # up to 64 rows
                                   *CUT, (777, 2112, 4096), (100, 264, 384), (2050, 1032, 384), (4100, 4620, 256), (5300, 18440, 2176)])                 # tiles
def test_bias_after_rounding_and_formats(M, N, K, fmt):
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert (_lib.load().mdy_fp8_gemm_form(M, N, K, 1) >> 8 > 1) == ((M, N, K) in CUT)
    a, a_s, b, b_s, bias, ref = _operands(M, N, K, fmt)
    plain = _call(a, a_s, b, b_s, None, 0, fmt)
    assert torch.equal(plain, ref.bfloat16())
    assert torch.equal(_call(a, a_s, b, b_s, bias, 1, fmt), add_bias(plain.clone(), bias))
    assert torch.equal(_call(a, a_s, b, b_s, bias, 0, fmt), (ref + bias.float()).bfloat16())
