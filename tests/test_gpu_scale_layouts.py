"""Activation and weight-row scales in every layout that the kernels read them in (K blocks ahead, four at a time, one at a time): a scale of its own for
every row and K block, NaN around them, K blocks in every remainder of four and up to more than a tile holds ahead.  Powers of two: exact."""
import pytest
import torch

from mdy_triton_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _operand(R, K, g):
    v = torch.randint(-2, 3, (R, K), generator=g, device=DEV)
    e = torch.randint(-2, 3, (R, K // 128), generator=g, device=DEV).float()
    return v.float(), torch.exp2(e)


def _laid_out(s, layout):
    """(first element, row stride, column stride, the buffer that holds it)"""
    R, KB = s.shape
    if layout == "rows":                                # the official dialect's
        return s.contiguous(), KB, 1
    if layout == "columns":                             # DeepLinear's
        return s.t().contiguous(), 1, R
    room = torch.full((R + 3, KB + 5), float("nan"), device=DEV)      # rows of a larger array, NaN around them
    room[1:R + 1, 3:KB + 3] = s
    return room[1:, 3:], KB + 5, 1


# forms (one launch or slabs of K): 128x128, 128x64, 64x128, 64x64, 128x192, 128x256, 256x256, and K blocks from 1 to 66
DENSE = [(777, 2112, 7168), (1024, 2048, 8192), (1000, 2048, 8448), (771, 3000, 128), (700, 2111, 640), (300, 7168, 4224), (520, 4096, 1408), (640, 512, 7296),
         (200, 4096, 7040), (130, 5000, 384), (64, 8900, 7168), (63, 18180, 640), (129, 320, 1152), (4096, 1536, 896), (1500, 4096, 3200), (1400, 4100, 3072),
         (3840, 3840, 384)]


@pytest.mark.parametrize("layout", ["rows", "columns", "inside"])
@pytest.mark.parametrize("M,N,K", DENSE)
def test_block_scaled(M, N, K, layout):
    lib, g = _lib.load(), torch.Generator(device=DEV).manual_seed(M + N + K)
    KB, NB = K // 128, -(-N // 128)
    a, sa = _operand(M, K, g)
    b = torch.randint(-2, 3, (N, K), generator=g, device=DEV).float()
    sb = torch.exp2(torch.randint(-2, 3, (NB, KB), generator=g, device=DEV).float())
    s, rs, cs = _laid_out(sa, layout)
    qa, qb = a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn)
    c = torch.full((M, N), float("nan"), device=DEV)
    nbytes = lib.mdy_fp8_gemm_workspace_bytes(M, N, K)
    ws = torch.empty(max(nbytes, 16), device=DEV, dtype=torch.uint8)
    rc = lib.mdy_fp8_gemm_nt_ws(qa.data_ptr(), s.data_ptr(), rs, cs, qb.data_ptr(), sb.data_ptr(), c.data_ptr(), None, M, N, K, 1, ws.data_ptr(), max(nbytes, 0),
                                torch.cuda.current_stream().cuda_stream)
    ref = (a * sa.repeat_interleave(128, 1)) @ (b * sb.repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)).t()
    assert rc == 0 and torch.equal(c, ref)


# the producer / consumer tiles in one launch: K blocks in every remainder of the four that their loop takes at a time, and on either side of the
# twelve whose scales come with a tile's start
@pytest.mark.parametrize("KB", [*range(1, 10), 11, 12, 13, 15, 16, 17, 18, 33])
@pytest.mark.parametrize("M,N,form", [(900, 2100, 5), (2000, 1000, 6), (2030, 1900, 7), (3000, 1500, 9)])
def test_chunks_of_scales(M, N, form, KB):
    lib, K = _lib.load(), KB * 128
    if form == 9 and KB < 3 or lib.mdy_fp8_gemm_form(M, N, K, 0) != form:
        pytest.skip("another form")
    g = torch.Generator(device=DEV).manual_seed(M + KB)
    a, sa = _operand(M, K, g)
    b = torch.randint(-2, 3, (N, K), generator=g, device=DEV).float()
    sb = torch.exp2(torch.randint(-2, 3, (-(-N // 128), KB), generator=g, device=DEV).float())
    qa, qb = a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn)
    ref = (a * sa.repeat_interleave(128, 1)) @ (b * sb.repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)).t()
    for layout in ("rows", "columns", "inside"):
        s, rs, cs = _laid_out(sa, layout)
        c = torch.full((M, N), float("nan"), device=DEV)
        rc = lib.mdy_fp8_gemm_nt_ws(qa.data_ptr(), s.data_ptr(), rs, cs, qb.data_ptr(), sb.data_ptr(), c.data_ptr(), None, M, N, K, 1, None, 0,
                                    torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and torch.equal(c, ref)


# plain loop, 128x128 tiles alone and two per CU, 128x256 (also slabs), 256x256 (also walked), K blocks 1 to 37
ROWS = [(250, 1036, 256), (890, 1028, 3072), (250, 1036, 1664), (1000, 2301, 896), (300, 700, 512), (2550, 3190, 1024), (770, 260, 384), (7290, 2170, 640), (644, 5433, 640),
        (3074, 4879, 640), (512, 512, 4096), (1530, 640, 4736), (4090, 3336, 384), (4352, 4104, 640), (4352, 4104, 256), (4097, 4160, 1152), (5504, 4735, 128),
        # on either side of the 12 K blocks from which row-major scales come in chunks
        (4000, 7100, 1408), (4000, 7096, 1536), (4000, 4090, 1920), (4352, 4104, 1664), (3074, 4879, 1920), (1790, 4097, 1792), (2305, 512, 3712)]


@pytest.mark.parametrize("layout", [("rows", "rows"), ("columns", "columns"), ("inside", "columns"), ("columns", "inside")])
@pytest.mark.parametrize("M,N,K", ROWS)
def test_row_scaled(M, N, K, layout):
    lib, g = _lib.load(), torch.Generator(device=DEV).manual_seed(M + N + K)
    (a, sa), (b, sb) = _operand(M, K, g), _operand(N, K, g)
    (s, rs, cs), (t, rt, ct) = _laid_out(sa, layout[0]), _laid_out(sb, layout[1])
    qa, qb = a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn)
    ref = (a * sa.repeat_interleave(128, 1)) @ (b * sb.repeat_interleave(128, 1)).t()
    for dtype, code in ((torch.bfloat16, 0), (torch.float32, 1)):
        c = torch.full((M, N), float("nan"), device=DEV, dtype=dtype)
        nbytes = lib.mdy_fp8_gemm_rowscaled_workspace_bytes(M, N, K)
        ws = torch.empty(max(nbytes, 16), device=DEV, dtype=torch.uint8)
        rc = lib.mdy_fp8_gemm_nt_rowscaled_ws(qa.data_ptr(), s.data_ptr(), rs, cs, qb.data_ptr(), t.data_ptr(), rt, ct, c.data_ptr(), M, N, K, 0, code, ws.data_ptr(),
                                              max(nbytes, 0), torch.cuda.current_stream().cuda_stream)
        assert rc == 0 and torch.equal(c, ref.to(dtype))
