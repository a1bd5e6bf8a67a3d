"""17 to 64 rows: the form a call takes (whole-line kernel, 64x64 or 64x128 tiles, either over slabs of K) is chosen by estimated
times; here every form with ragged rows and columns, one K block to more than a ring holds."""
import random

import pytest
import torch

from mdy_triton_amd import _lib
from test_gpu_gemm import test_gemm_exact_integer_cases_all_kernels as exact_integer

WHOLE_LINES, T64X64, T64X128 = 1, 4, 5      # MDY_FORM_...
# (M, N, K), form, slabs of K (0: one launch)
FORMS = [((17, 5001, 512), WHOLE_LINES, 0), ((64, 7168, 2048), WHOLE_LINES, 0), ((17, 2050, 7168), WHOLE_LINES, 0),
         ((17, 14802, 256), T64X64, 0), ((64, 16384, 128), T64X64, 0), ((33, 10945, 1280), T64X64, 0), ((64, 18181, 2816), T64X128, 0),
         ((63, 18180, 640), T64X128, 0), ((63, 3001, 6528), T64X64, 5), ((64, 8900, 7168), T64X128, 3), ((17, 1537, 16384), T64X64, 8),
         ((40, 1025, 9088), WHOLE_LINES, 7), ((18, 9665, 6912), T64X128, 3), ((64, 9000, 7168), T64X128, 3), ((20, 4998, 11520), T64X128, 6),
         # where the lines between sizes and an estimate disagree by less than the estimate's error: the lines' form
         ((34, 4096, 8192), T64X64, 4), ((50, 512, 4992), WHOLE_LINES, 4), ((60, 1792, 6272), WHOLE_LINES, 4),
         ((34, 832, 4864), WHOLE_LINES, 4), ((64, 1536, 4096), WHOLE_LINES, 4), ((64, 1536, 3968), WHOLE_LINES, 0),
         # what one launch finishes before the host has enqueued a second
         ((19, 576, 7424), WHOLE_LINES, 0), ((20, 768, 10112), WHOLE_LINES, 5)]


@pytest.mark.parametrize("shape,form,slabs", FORMS)
def test_forms(shape, form, slabs):
    """On a full-size part, which is also what the query assumes without a GPU."""
    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the form of a call depends on the number of CUs")
    got = _lib.load().mdy_fp8_gemm_form(*shape, 1)
    assert (got & 255, got >> 8) == (form, slabs)


def test_every_plan_fits_the_static_scratch():
    """A call that the entry point without allocation took is not refused because its slabs grew."""
    lib, r = _lib.load(), random.Random(5)
    limit = lib.mdy_fp8_gemm_static_workspace_bytes()
    for _ in range(10000):
        M, N, K = r.choice([r.randrange(17, 65), r.randrange(65, 2500)]), r.choice([r.randrange(1, 3000), r.randrange(1, 30000)]), 128 * r.randrange(1, 513)
        if lib.mdy_fp8_gemm_form(M, N, K, 1) >> 8:
            assert lib.mdy_fp8_gemm_workspace_bytes(M, N, K) <= limit, (M, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [f[0] for f in FORMS])
def test_exact_integer(shape):
    exact_integer(*shape)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(33, 10944, 1280), (64, 9000, 7168), (17, 14801, 256)])
def test_e5m2_and_bias(M, N, K):
    """The same routes with e5m2 bytes and a bias (in the epilogue of one launch, in the reduction of slabs)."""
    g = torch.Generator().manual_seed(M + N)
    ai, bi = torch.randint(-2, 3, (M, K), generator=g), torch.randint(-2, 3, (N, K), generator=g)
    bias = torch.randint(-8, 9, (N,), generator=g).float()
    from mdy_triton_amd import fp8_kernel
    fmt = torch.float8_e5m2
    ones_a, ones_b = torch.ones(M, K // 128, device="cuda"), torch.ones((N + 127) // 128, K // 128, device="cuda")
    got = fp8_kernel.fp8_matmul(ai.float().to(fmt).cuda(), bi.float().to(fmt).cuda(), ones_a, ones_b, bias=bias.bfloat16().cuda())
    want = (ai.double() @ bi.double().t() + bias.double()).float().bfloat16()
    assert torch.equal(got.cpu(), want)


# more than 64 rows where the estimates of one fit or another override the line between sizes: among them 64x128 tiles in one launch and over slabs, 128x192 over slabs
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(113, 11451, 8576), (354, 3968, 12032), (123, 17920, 1152), (65, 961, 3584), (163, 1725, 3584), (294, 960, 12928),
                                   (150, 8897, 2304), (256, 4096, 4096), (255, 4090, 4224), (142, 8960, 896), (129, 3000, 4608), (900, 960, 6400)])
def test_exact_integer_where_an_estimate_decides(M, N, K):
    exact_integer(M, N, K)


# barely more than a full round of 256x256 tiles: all of it on 128x256 tiles; one round of 128x192 / 128x256 tiles with few K blocks
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2383, 6656, 256), (2303, 6651, 640), (65900, 250, 128), (1508, 3072, 896), (1503, 3065, 384), (511, 8450, 512), (1860, 2750, 768),
                                   (320, 19100, 768)])
def test_exact_integer_tiles_of_a_round(M, N, K):
    exact_integer(M, N, K)


# K blocks per wave that no depth of a pass divides (5 with 32 rows, 9, 11, 13, 17): the last pass is filled up
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 4608, 3968), (8, 4224, 8448), (9, 17472, 8576), (16, 1537, 11264), (13, 6401, 8960), (2, 7170, 13312), (16, 1000, 17408),
                                   (28, 7168, 5120), (17, 8190, 4736)])
def test_exact_integer_filled_passes(M, N, K):
    exact_integer(M, N, K)
