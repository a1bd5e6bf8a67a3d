"""Every tile of a launch is computed once, whatever the tile count leaves over 8 (the tiles are dealt out to 8 XCDs in runs)."""
import pytest
import torch

import mdy_triton_amd as m

pytestmark = pytest.mark.gpu


# integer operands and power-of-two scales: every order of summation is exact, so any tile left out or computed twice elsewhere shows
@pytest.mark.parametrize("M,N,K", [(70, 64, 256), (130, 200, 256), (300, 264, 256), (321, 449, 256), (513, 1000, 128), (650, 1410, 128),      # 64x64
                                   (1030, 3001, 256), (1153, 3840, 256), (1270, 2112, 256),      # 128x64 and 128x128
                                   (777, 7168, 1024), (1100, 6000, 1024),                        # 128x256
                                   (4097, 4400, 128), (3752, 15224, 256), (5000, 5000, 128),     # 256x256, walked
                                   (777, 2112, 4096), (200, 1100, 4096), (100, 1000, 7168),      # cut along K
                                   # (slab, tile) counts that 8 does not divide: slabs of 9 and 10 K blocks, of 12 against a long K, of 16, of 9 against a long K
                                   (771, 896, 5632), (631, 760, 7808), (219, 704, 13568), (314, 1150, 13824), (130, 2624, 12160), (164, 1280, 11264)])
def test_exact_integer(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    KB, NB = K // 128, -(-N // 128)
    a, b = (torch.randint(-2, 3, (r, K), generator=g, device="cuda").float() for r in (M, N))
    sa, sb = (torch.exp2(torch.randint(-2, 3, s, generator=g, device="cuda").float()) for s in ((M, KB), (NB, KB)))
    got = m.fp8_gemm(a.to(torch.float8_e4m3fn), sa, b.to(torch.float8_e4m3fn), sb, out_dtype=torch.float32)
    ref = (a * sa.repeat_interleave(128, 1)) @ (b * sb.repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)).t()
    assert torch.equal(got, ref)
