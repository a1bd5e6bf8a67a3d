"""e5m2 quantizers on groups of every magnitude: the reciprocal quotient's range, its lower edge and what lies below it."""
import numpy as np
import pytest
import torch

from mdy_triton_amd import fp8_kernel as FK
from oracle import oracle as O

pytestmark = pytest.mark.gpu
E5M2 = torch.float8_e5m2


def _same(got, ref):
    (y, s), (ry, rs) = got, ref
    b, rb = y.cpu().view(torch.uint8).numpy(), ry.view(torch.uint8).numpy()
    nan = (rb & 0x7F) > 0x7C                       # an all-zero group divides 0 by 0: the NaN's sign is not compared
    assert np.array_equal(b[~nan], rb[~nan]) and np.array_equal((b & 0x7F) > 0x7C, nan)
    assert torch.equal(s.cpu(), rs)


@pytest.mark.parametrize("M,K", [(254, 1024), (3, 128), (8232, 8192)])      # the last: large enough for every launch shape
def test_e5m2_bit_exact_over_all_exponents(M, K):
    g = torch.Generator().manual_seed(M)
    # bf16 patterns whose group maximum sits in exponent 1..254, with values down to 2^-24 of it
    e = torch.arange(M * (K // 128)).reshape(M, K // 128) % 254 + 1
    drop = torch.randint(0, 24, (M, K), generator=g)
    exp = (e.repeat_interleave(128, 1) - drop).clamp(min=0)
    bits = (exp << 7) | torch.randint(0, 128, (M, K), generator=g) | (torch.randint(0, 2, (M, K), generator=g) << 15)
    x = bits.to(torch.int32).to(torch.int16).view(torch.bfloat16)
    _same(FK.act_quant_block(x.cuda(), dtype=E5M2), O.act_quant_block(x, dtype=E5M2))
    if M < 1000:
        _same(FK.act_quant_block(x.cuda(), transpose=True, dtype=E5M2), O.act_quant_block(x, transpose=True, dtype=E5M2))
        w = x.repeat(-(-128 // M), 1)[:128]
        _same(FK.weight_quant_block(w.cuda(), dtype=E5M2), O.weight_quant_block(w, dtype=E5M2))
