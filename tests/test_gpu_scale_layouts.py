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
         (3840, 3840, 384), (1055, 422, 1408), (183, 838, 5632), (822, 2383, 1024), (529, 888, 7680), (287, 3598, 8832)]
DENSE_FORMS = {4, 5, 6, 7, 9, 10, 12}, {4, 5, 6, 7, 9}      # MDY_FORM_... in one launch, over slabs


def on_256_cus():
    return torch.cuda.get_device_properties(0).multi_processor_count == 256


def test_sizes_take_these_forms():
    """The kernels that the sizes above mean, so that a later rule cannot send them elsewhere unnoticed."""
    got = [_lib.load().mdy_fp8_gemm_form(*size, 1) for size in DENSE]
    if on_256_cus():
        assert DENSE_FORMS == ({v for v in got if v < 256}, {v & 255 for v in got if v >= 256})


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
KBS = [*range(1, 10), 11, 12, 13, 15, 16, 17, 18, 33]


@pytest.mark.parametrize("M,N,form,KB", [(*tile, KB) for tile in ((900, 2100, 5), (2000, 1000, 6), (2030, 1900, 7), (3000, 1500, 9)) for KB in KBS
                                         if tile[2] != 9 or KB >= 3])      # 128x192 tiles do not run with less
def test_chunks_of_scales(M, N, form, KB):
    lib, K = _lib.load(), KB * 128
    if on_256_cus():
        assert lib.mdy_fp8_gemm_form(M, N, K, 0) == form
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


# MDY_FORM_..., and slabs of K above it: plain loop, 128x128 tiles alone and two per CU, 128x256 (also slabs), 256x256 (also walked), K blocks 1 to 37
PLAIN, RING3, TWO, WIDE, BIG = 14, 7, 8, 10, 12
ROWS = [((250, 1036, 256), PLAIN), ((250, 1036, 1664), RING3), ((1000, 2301, 896), RING3), ((300, 700, 512), TWO), ((2550, 3190, 1024), TWO), ((770, 260, 384), TWO),
        ((7290, 2170, 640), TWO), ((4352, 4104, 256), TWO), ((4097, 4160, 1152), TWO), ((4352, 4104, 1664), TWO), ((644, 5433, 640), WIDE), ((3074, 4879, 640), WIDE),
        ((4352, 4104, 640), TWO), ((4090, 3336, 384), BIG),
        # walked, in results that go out in whole lines and otherwise
        ((4352, 5000, 640), BIG), ((4000, 7104, 640), BIG), ((4358, 5519, 256), BIG), ((5504, 4735, 128), BIG),
        # on either side of the 12 K blocks from which row-major scales come in chunks, every remainder of 4; the first two in one round, the others walked
        ((4000, 4090, 1920), BIG), ((4090, 4096, 1408), BIG), ((4000, 7100, 1408), BIG), ((4000, 7096, 1536), BIG), ((4000, 7104, 1536), BIG), ((4000, 7104, 1664), BIG),
        ((4000, 7104, 1792), BIG), ((4000, 7104, 1920), BIG), ((3074, 4879, 1920), WIDE), ((1790, 4097, 1792), WIDE),
        # slabs, in rows of whole lines and, where 4 does not divide N, a result at a time
        ((512, 512, 4096), WIDE | 8 << 8), ((890, 1028, 3072), WIDE | 4 << 8), ((1530, 640, 4736), WIDE | 5 << 8), ((2305, 512, 3712), WIDE | 5 << 8),
        ((1000, 1030, 4224), WIDE | 5 << 8), ((1530, 638, 4736), WIDE | 5 << 8)]


@pytest.mark.parametrize("layout", [("rows", "rows"), ("columns", "columns"), ("inside", "columns"), ("columns", "inside")])
@pytest.mark.parametrize("size,form", ROWS)
def test_row_scaled(size, form, layout):
    M, N, K = size
    lib, g = _lib.load(), torch.Generator(device=DEV).manual_seed(M + N + K)
    if on_256_cus():
        assert lib.mdy_fp8_gemm_rowscaled_form(M, N, K, 1) == form
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
