"""256x256 tile kernels whose workgroups have a second tile: its copies are issued in front of the first one's results."""
import pytest
import torch

import mdy_triton_amd as m
from mdy_triton_amd import fp8, fp8_kernel as FK

pytestmark = pytest.mark.gpu


def _sides(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * 0.1).bfloat16()
    return x, w


def _same_in_pieces(got, piece, rows=512, cols=2048):
    """Every tile kernel adds the K blocks in their order: pieces that smaller tiles compute have the same bits (whole pieces only:
    the kernels for a few rows share the K blocks out among waves)."""
    for r in range(0, got.size(0), rows):
        r = min(r, got.size(0) - rows)
        for c in range(0, got.size(1), cols):
            assert torch.equal(got[r:r + rows, c:c + cols], piece(slice(r, r + rows), slice(c, c + cols))), (r, c)


# 272 and 273 tiles (16 or 17 workgroups with two), ragged rows and columns, one to three K blocks and more
@pytest.mark.parametrize("M,N,K", [(4352, 4096, 128), (4352, 4096, 256), (4300, 4104, 384), (4097, 4160, 128), (5377, 3080, 640), (8192, 8192, 256)])
def test_row_scales(M, N, K):
    x, w = _sides(M, N, K)
    qx, sx = FK.act_quant_block(x, dtype=torch.float8_e4m3fn)
    qw, sw = FK.act_quant_block(w, dtype=torch.float8_e4m3fn)
    M -= M % 128      # the operator takes whole groups of 128 rows
    qx, sx = qx[:M], sx[:M]
    got = FK.fp8_matmul(qx, qw, sx, sw, have_w=False)
    _same_in_pieces(got, lambda r, c: FK.fp8_matmul(qx[r], qw[c], sx[r], sw[c], have_w=False))


@pytest.mark.parametrize("M,N,K", [(8192, 8192, 128), (8449, 8192, 256), (8200, 8200, 384), (16384, 4104, 512)])
@pytest.mark.parametrize("mode", [None, fp8.BIAS_IN_SUM, fp8.BIAS_AFTER_ROUNDING])
def test_block_scales_and_nothing_beyond(M, N, K, mode):
    x, w = _sides(M, N, K)
    qx, sx = m.act_quant(x)
    qw, sw, _, _ = fp8.quant_weight(torch.nn.functional.pad(w, (0, 0, 0, -N % 128)))
    qw = qw[:N, :K].contiguous()
    sw = sw[:, :K // 128].contiguous()
    bias = torch.randn(N, device="cuda").bfloat16() if mode is not None else None
    room = torch.full((M * N + 512,), float("nan"), device="cuda", dtype=torch.bfloat16)      # 256 elements before and behind
    out = room[256:-256].view(M, N)
    fp8._matmul(qx, sx, qw, sw, out, bias, mode or 0)
    assert torch.isnan(room[:256]).all() and torch.isnan(room[-256:]).all()
    _same_in_pieces(out, lambda r, c: fp8._matmul(qx[r], sx[r], qw[c], sw[c.start // 128:(min(c.stop, N) + 127) // 128], None,
                                                  bias[c] if bias is not None else None, mode or 0))
