"""Grouped GEMM: the tile rows that whole rounds of 256x256 tiles do not reach, in pieces of 128 rows and 128 or 192 columns.  Integer
operands and power-of-two scales: exact whatever the tile."""
import ctypes

import pytest
import torch

import mdy_triton_amd as m
from mdy_triton_amd import _lib
from tests.test_gpu_grouped import PIECES128, PIECES192, QUARTERS, REST128, REST192, REST256, TILES, runs

pytestmark = pytest.mark.gpu
DEV = "cuda"


# rows per group, N, K, kernel: pieces of 128 columns (less than a quarter round), of 192 (up to 3/8), behind a whole round, ragged rows
# and columns, empty groups, a group that ends within the first half of a tile row, rows that start inside lines
CASES = [([256, 300, 0, 1], 520, 384, REST128), ([100, 70, 513], 1032, 640, REST128), ([129] * 7, 264, 256, REST128),
         ([700, 1, 0, 900, 411], 1536, 384, REST128), ([256] * 11, 1800, 256, REST192), ([2000, 130, 640], 1544, 128, REST192),
         ([640] * 7, 4096, 256, REST192), ([1000, 3000, 129, 1], 4104, 384, REST128), ([512, 700] * 4, 3848, 128, REST128),
         ([2500, 2500, 388], 4100, 256, REST256),      # too many pieces for 192 columns: halves of tiles
         # a round and a quarter whose left tile rows are more than a round of 128-column pieces: quarters of tiles, on whole lines, with
         # an empty column piece, odd N; empty, short and full second rows; 33 K blocks
         ([256] * 12 + [300, 70, 200], 5056, 256, QUARTERS), ([256] * 13 + [0, 450, 129], 4900, 128, QUARTERS),
         ([256] * 12 + [300, 70, 256], 5111, 384, QUARTERS), ([256] * 15 + [200], 5000, 4224, QUARTERS),
         # 128-column pieces from 32 K blocks on, of full tile rows and of half empty ones
         ([256, 100, 300], 1300, 4224, REST128),
         # counted by pieces of 128 rows, of 128 columns and of 192: groups of one piece, two and three, empty and of one row
         ([300] * 9, 1100, 384, PIECES128), ([70, 128, 1, 0, 129, 300, 90, 65] * 2, 2050, 256, PIECES192), ([100] * 16, 2044, 384, PIECES128),
         ([66] * 32, 900, 640, PIECES128), ([128, 70] * 8, 3070, 256, PIECES192), ([257, 0, 385, 90] * 3, 1905, 128, PIECES192),
         ([257, 0, 385, 90] * 3, 2305, 128, TILES)]


@pytest.mark.parametrize("rows,N,K,form", CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_exact_integer(rows, N, K, form, dtype):
    runs(rows, N, K, form)
    g = torch.Generator(device=DEV).manual_seed(sum(rows) + N + K)
    M, G, KB, NB = sum(rows), len(rows), K // 128, (N + 127) // 128
    ai, bi = torch.randint(-3, 4, (M, K), generator=g, device=DEV), torch.randint(-3, 4, (G, N, K), generator=g, device=DEV)
    ea, eb = torch.randint(-2, 3, (M, KB), generator=g, device=DEV), torch.randint(-2, 3, (G, NB, KB), generator=g, device=DEV)
    fp8 = torch.float8_e4m3fn
    qa, sa, qb, sb = ai.float().to(fp8), torch.exp2(ea.float()), bi.float().to(fp8), torch.exp2(eb.float())
    if dtype == torch.bfloat16:
        got = m.fp8_grouped_matmul(qa, sa, qb, sb, rows)
    else:
        got = torch.full((M, N), float("nan"), device=DEV)
        splits = (ctypes.c_int64 * G)(*rows)
        assert _lib.load().mdy_fp8_grouped_gemm_nt(qa.data_ptr(), sa.data_ptr(), KB, 1, qb.data_ptr(), sb.data_ptr(), got.data_ptr(), None,
                                                   ctypes.cast(splits, ctypes.c_void_p), G, N, K, 1, torch.cuda.current_stream().cuda_stream) == 0
    a = (ai.double().view(M, KB, 128) * torch.exp2(ea.double())[:, :, None]).view(M, K)
    row = 0
    for i, r in enumerate(rows):
        b = (bi[i].double().view(N, KB, 128) * torch.exp2(eb[i].double())[torch.arange(N, device=DEV) // 128][:, :, None]).view(N, K)
        assert torch.equal(got[row:row + r], (a[row:row + r] @ b.t()).to(dtype)), i
        row += r
