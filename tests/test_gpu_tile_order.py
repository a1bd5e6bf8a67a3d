"""Every tile of a launch is computed once, whatever the tile count leaves over 8 (the tiles are dealt out to 8 XCDs in runs)."""
import pytest
import torch

import mdy_triton_amd as m
from mdy_triton_amd import _lib

pytestmark = pytest.mark.gpu

# MDY_FORM_...
T64, T64X128, T128X64, T128, TWO, T128X192, T128X256, T256X128, BIG, REST = 4, 5, 6, 7, 8, 9, 10, 11, 12, 13
EDGES = {T64: (64, 64), T64X128: (64, 128), T128X64: (128, 64), T128: (128, 128), TWO: (128, 128), T128X192: (128, 192), T128X256: (128, 256), T256X128: (256, 128)}
ONE_LAUNCH = [((128, 3433, 1280), T64), ((1055, 422, 1408), T64), ((151, 3614, 1408), T64), ((680, 2712, 1024), T64X128), ((822, 2383, 1024), T64X128),
              ((70, 64, 256), T128X64), ((300, 264, 256), T128X64), ((321, 449, 256), T128X64), ((650, 1410, 128), T128X64), ((343, 2087, 1152), T128X64),
              ((777, 2112, 4096), T128X64), ((863, 3096, 256), T128), ((1246, 1881, 1024), T128), ((1030, 3001, 256), T128), ((1270, 2112, 256), T128),
              ((1153, 3840, 256), TWO), ((1076, 3680, 384), TWO), ((1348, 3563, 1280), T128X192), ((777, 7168, 1024), T128X256), ((1100, 6000, 1024), T128X256),
              ((33000, 128, 1024), T256X128), ((4097, 4400, 128), REST), ((3752, 15224, 256), BIG), ((5000, 5000, 128), BIG)]
# (M, N, K), form, slabs of K, K blocks per slab: in runs from 13 K blocks on, and with tiles of at least 128x128 against K > 8192 from 10 on; else in plain order
CUT = [((183, 838, 5632), T64, 5, 9), ((68, 895, 14080), T64, 9, 13), ((132, 2095, 5632), T64X128, 5, 9), ((170, 1413, 9600), T64X128, 7, 11),
       ((529, 888, 7680), T64X128, 4, 15), ((314, 1150, 13824), T64X128, 5, 22), ((469, 560, 5632), T128X64, 5, 9), ((148, 857, 11520), T128X64, 9, 10),
       ((219, 704, 13568), T128X64, 11, 10), ((884, 264, 14080), T128X64, 7, 16), ((771, 896, 5632), T128X64, 2, 22), ((67, 3561, 7680), T128, 7, 9),
       ((86, 2368, 11520), T128, 10, 9), ((80, 3430, 11520), T128, 9, 10), ((195, 2153, 9600), T128, 7, 11), ((532, 1216, 7680), T128, 5, 12),
       ((300, 1398, 14080), T128, 7, 16), ((130, 2624, 12160), T128, 6, 16), ((66, 6592, 16640), T128X192, 7, 19), ((287, 3598, 8832), T128X192, 4, 18)]
# counts that 8 divides
EVEN = [((130, 200, 256), T128X64, 0, 2), ((513, 1000, 128), T128X64, 0, 1), ((200, 1100, 4096), T128X64, 4, 8), ((100, 1000, 7168), T128X64, 8, 7),
        ((631, 760, 7808), T128X64, 4, 16), ((164, 1280, 11264), T64X128, 8, 11)]


def runs(size, form, slabs, per):
    """The kernel, the slabs and their length that a case means, so that a later rule cannot send it elsewhere unnoticed; how many (slab, tile) pairs."""
    M, N, K = size
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert _lib.load().mdy_fp8_gemm_form(M, N, K, 1) == form | slabs << 8, size
    assert -(-(K // 128) // max(slabs, 1)) == per
    bm, bn = EDGES.get(form, (256, 256))
    return -(-M // bm) * -(-N // bn) * max(slabs, 1)


# integer operands and power-of-two scales: every order of summation is exact, so any tile left out or computed twice elsewhere shows
@pytest.mark.parametrize("size,form,slabs,per", [(s, f, 0, s[2] // 128) for s, f in ONE_LAUNCH] + CUT + EVEN)
def test_exact_integer(size, form, slabs, per):
    M, N, K = size
    count = runs(size, form, slabs, per)
    if (size, form, slabs, per) in CUT:
        assert count % 8 != 0
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    KB, NB = K // 128, -(-N // 128)
    a, b = (torch.randint(-2, 3, (r, K), generator=g, device="cuda").float() for r in (M, N))
    sa, sb = (torch.exp2(torch.randint(-2, 3, s, generator=g, device="cuda").float()) for s in ((M, KB), (NB, KB)))
    got = m.fp8_gemm(a.to(torch.float8_e4m3fn), sa, b.to(torch.float8_e4m3fn), sb, out_dtype=torch.float32)
    ref = (a * sa.repeat_interleave(128, 1)) @ (b * sb.repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)).t()
    assert torch.equal(got, ref)
