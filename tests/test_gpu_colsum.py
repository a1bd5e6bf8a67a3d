"""The output-gradient quantizers with column sums: bytes and scales of the quantizer without them, sums in fp32 rounded once."""
import pytest
import torch

from mdy_triton_amd import fp8, fp8_kernel as FK

pytestmark = pytest.mark.gpu


def _check_sum(got, x):
    # fp32 sums in any order: at most M rounding errors of the running absolute sum, then one rounding to bf16
    ref = x.double().sum(0)
    bound = x.size(0) * 2.0 ** -24 * x.double().abs().sum(0) + 2.0 ** -8 * ref.abs()
    assert ((got.double() - ref).abs() <= bound).all()


@pytest.mark.parametrize("M,N,transposed", [(1, 128, False), (130, 384, False), (4096, 1536, False), (5000, 5120, False), (300, 256, True)])
def test_column_sums(M, N, transposed):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, N, generator=g).bfloat16().cuda()
    if transposed:
        x = x.t().contiguous().t()
    out = torch.empty(N, device="cuda", dtype=torch.bfloat16)
    for quantize in (lambda o: fp8._quant_transpose(x, 0, "t", o), lambda o: FK._act_quant_transposed(x, True, "t", torch.float8_e5m2, o),
                     lambda o: FK._act_quant_transposed(x, False, "t", torch.float8_e4m3fn, o)):
        out.fill_(float("nan"))
        for a, b in zip(quantize(out), quantize(None)):
            assert (a is None and b is None) or torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))
        _check_sum(out, x)


def test_ragged_columns():
    x = torch.randn(1000, 200, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    out = torch.full((201,), float("nan"), device="cuda", dtype=torch.bfloat16)
    fp8._quant_transpose(x, 0, "t", out[:200])
    _check_sum(out[:200], x)
    assert torch.isnan(out[200])


@pytest.mark.parametrize("M,K,PM,PK", [(0, 200, 0, 256), (0, 128, 128, 128), (0, 0, 128, 128), (5, 0, 128, 128), (0, 0, 0, 128), (0, 0, 0, 0)])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_empty_sums_are_zero(M, K, PM, PK, mode):
    from mdy_triton_amd import _lib
    x, y, yt = (torch.empty(128 * 256, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    s, st, part = (torch.empty(512, device="cuda") for _ in range(3))
    out = torch.full((K + 1,), float("nan"), device="cuda", dtype=torch.bfloat16)
    rc = _lib.load().mdy_quant_transpose_colsum(x.data_ptr(), y.data_ptr(), s.data_ptr(), yt.data_ptr(), st.data_ptr(), M, K, max(K, 1), 1, PM, PK,
                                                PM, mode, part.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert not out[:K].any() and torch.isnan(out[K])
