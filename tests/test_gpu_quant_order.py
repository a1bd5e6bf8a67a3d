"""Quantizers with a transposed copy deal their tiles out to the XCDs in patches beyond 1280 tiles: every tile once, the same bytes and scales as
slabs of the rows, which stay below that and run in plain order."""
import ctypes

import pytest
import torch

from mdy_triton_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# tiles: 22 x 59 (the last 6 rows are no patch), 8 x 161, 9 x 143, 160 x 8 = 1280 (in plain order), 161 x 8, 1 x 1300 (no patch at all), 80 x 16 = 1280, 1264
SIZES = [(2816, 7552), (1024, 20608), (1152, 18304), (20480, 1024), (20608, 1024), (128, 166400), (10240, 2048), (10112, 2048)]


def _x(M, K, seed=0):
    g = torch.Generator(device=DEV).manual_seed(M + K + seed)
    return torch.randn(M, K, generator=g, device=DEV).bfloat16()


def _bytes(*size):
    return torch.full(size, 0x55, device=DEV, dtype=torch.uint8)


def _floats(*size):
    return torch.full(size, float("nan"), device=DEV)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _slabs(M, K, rows=None):
    rows = rows or max(128, 1279 // (K // 128) * 128)
    return [(r, min(rows, M - r)) for r in range(0, M, rows)]


def _same(whole, parts):
    """parts: per slab (y, s, y_t, s_t [, sums]) with s as [rows, K/128], s_t as [K, rows/128]."""
    y, s, yt, st = (torch.cat(p, d) for p, d in zip(zip(*[p[:4] for p in parts]), (0, 0, 1, 1)))
    assert torch.equal(whole[0], y) and torch.equal(whole[1], s) and torch.equal(whole[2], yt) and torch.equal(whole[3], st)


@pytest.mark.parametrize("M,K", SIZES)
@pytest.mark.parametrize("mode", [0, 2])
def test_official_copies(M, K, mode):
    x, lib = _x(M, K), _lib.load()

    def run(x, col_sum):
        M = x.size(0)
        y, s, yt, st, part, sums = _bytes(M, K), _floats(M, K // 128), _bytes(K, M), _floats(K, M // 128), _floats(M // 128, K), torch.empty(K, device=DEV).bfloat16()
        if col_sum:
            rc = lib.mdy_quant_transpose_colsum(x.data_ptr(), y.data_ptr(), s.data_ptr(), yt.data_ptr(), st.data_ptr(), M, K, K, 1, M, K, 0, mode,
                                                part.data_ptr(), sums.data_ptr(), _stream())
        else:
            rc = lib.mdy_act_quant_transpose(x.data_ptr(), 0, y.data_ptr(), s.data_ptr(), yt.data_ptr(), st.data_ptr(), M, K, K, 1, M, K, mode, _stream())
        assert rc == 0
        return y, s, yt, st, part

    for col_sum in (False, True):
        whole, parts = run(x, col_sum), [run(x[r:r + n], col_sum) for r, n in _slabs(M, K)]
        _same(whole, parts)
        if col_sum:
            assert torch.equal(whole[4], torch.cat([p[4] for p in parts]))


@pytest.mark.parametrize("M,K", SIZES)
@pytest.mark.parametrize("t_mode", [0, 1])
def test_deep_copies_and_groups(M, K, t_mode):
    x, lib = _x(M, K), _lib.load()

    def run(x):
        M = x.size(0)
        y, s, yt, st = _bytes(M, K), _floats(K // 128, M), _bytes(K, M), _floats(M // 128, K) if t_mode == 0 else _floats(K // 128, M // 128)
        rc = lib.mdy_quant_transpose_typed(x.data_ptr(), 0, y.data_ptr(), s.data_ptr(), yt.data_ptr(), st.data_ptr(), M, K, K, 1, M, K, M, t_mode, _stream())
        assert rc == 0
        return y, s.t(), yt, st.t() if t_mode == 0 else st

    whole, slabs = run(x), _slabs(M, K)
    _same(whole, [run(x[r:r + n]) for r, n in slabs])
    if t_mode == 0:      # groups: the transposed copies are arrays of their own
        y, s = _bytes(M, K), _floats(K // 128, M)
        yt, st = [_bytes(K, n) for _, n in slabs], [_floats(n // 128, K) for _, n in slabs]
        G = len(slabs)
        rc = lib.mdy_quant_transpose_grouped(x.data_ptr(), 0, y.data_ptr(), s.data_ptr(), (ctypes.c_void_p * G)(*[t.data_ptr() for t in yt]),
                                             (ctypes.c_void_p * G)(*[t.data_ptr() for t in st]), (ctypes.c_int64 * G)(*[n for _, n in slabs]), G, K, K, 1, _stream())
        assert rc == 0
        _same(whole, [(y[r:r + n], s.t()[r:r + n], a, b.t()) for (r, n), a, b in zip(slabs, yt, st)])


@pytest.mark.parametrize("N,K", SIZES)
@pytest.mark.parametrize("G", [1, 3])
def test_weights(N, K, G):
    if G == 3:
        N = N // 128 // 3 * 128
        if N == 0:
            pytest.skip("one row of tiles")
    ws, lib = [_x(N, K, i) for i in range(G)], _lib.load()

    def run(ws):
        G, N = len(ws), ws[0].size(0)
        y, s, yt, st = _bytes(G, N, K), _floats(G, N // 128, K // 128), _bytes(G, K, N), _floats(G, K // 128, N // 128)
        if G == 1:
            rc = lib.mdy_weight_quant(ws[0].data_ptr(), y.data_ptr(), s.data_ptr(), yt.data_ptr(), st.data_ptr(), N, K, K, 1, N, K, 1, _stream())
        else:
            rc = lib.mdy_weight_quant_group((ctypes.c_void_p * G)(*[w.data_ptr() for w in ws]), G, 0, y.data_ptr(), s.data_ptr(), yt.data_ptr(), st.data_ptr(),
                                            N, K, K, 1, N, K, 1, _stream())
        assert rc == 0
        return y, s, yt, st

    whole = run(ws)
    for g, w in enumerate(ws):
        _same([t[g] for t in whole], [[t[0] for t in run([w[r:r + n]])] for r, n in _slabs(N, K)])


@pytest.mark.parametrize("M,I", [(2816, 7552), (1152, 18304), (10240, 2048)])
def test_swiglu_backward(M, I):
    x, d, lib = _x(M, 2 * I), _x(M, I, 1), _lib.load()

    def run(x, d):
        M = x.size(0)
        at, ats, y, s, yt, st = _bytes(I, M), _floats(I, M // 128), _bytes(M, 2 * I), _floats(M, I // 64), _bytes(2 * I, M), _floats(2 * I, M // 128)
        rc = lib.mdy_swiglu_bwd_quant(x.data_ptr(), d.data_ptr(), at.data_ptr(), ats.data_ptr(), y.data_ptr(), s.data_ptr(), yt.data_ptr(), st.data_ptr(),
                                      M, I, 0, M, I, 0, _stream())
        assert rc == 0
        return y, s, yt, st, at, ats

    whole, parts = run(x, d), [run(x[r:r + n], d[r:r + n]) for r, n in _slabs(M, I)]
    _same(whole[:4], parts)
    assert torch.equal(whole[4], torch.cat([p[4] for p in parts], 1)) and torch.equal(whole[5], torch.cat([p[5] for p in parts], 1))
