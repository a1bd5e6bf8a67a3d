"""The C-ABI library loads, exports every symbol include/mdy_fp8.h declares, and
rejects bad arguments before touching a device (no compute calls here)."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "mdy_fp8.h")


@pytest.fixture(scope="module")
def lib():
    from mdy_triton_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        from mdy_triton_amd.csrc.build import build
        build()
    return _lib.load()


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mdy_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_are_exported(lib):
    names = declared_functions()
    assert "mdy_act_quant" in names and "mdy_fp8_gemm_nt" in names and len(names) >= 9
    for n in names:
        assert hasattr(lib, n), "missing export %s" % n
    from mdy_triton_amd._lib import SIGNATURES
    assert sorted(SIGNATURES) == names


def test_abi_version(lib):
    text = open(HEADER).read()
    v = int(re.search(r"#define MDY_FP8_ABI_VERSION (\d+)", text).group(1))
    assert lib.mdy_fp8_abi_version() == v


def test_older_library_is_named_as_such(lib, tmp_path, monkeypatch):
    """A library of another version is refused for its version, whatever else it lacks."""
    import subprocess
    from mdy_triton_amd import _lib
    src, old = tmp_path / "old.c", tmp_path / "libmdyfp8.so"
    src.write_text("int mdy_fp8_abi_version(void) { return %d; }\n" % (_lib.ABI_VERSION - 1))
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(old)], check=True)
    monkeypatch.setattr(_lib, "LIB_PATH", str(old))
    monkeypatch.setattr(_lib, "_lib", None)
    with pytest.raises(_lib.MdyFp8Error, match="rebuild"):
        _lib.load()


def test_argument_validation_without_device(lib):
    buf = ctypes.create_string_buffer(4096)
    p = ctypes.addressof(buf)
    # PK not a multiple of 128
    assert lib.mdy_act_quant(p, p, p, 4, 100, 100, 4, 100, 1, 1, 0, None) == -2
    assert b"128" in lib.mdy_fp8_last_error()
    # unknown dialect / dtype
    assert lib.mdy_act_quant(p, p, p, 4, 128, 128, 4, 128, 1, 1, 7, None) == -4
    assert lib.mdy_weight_dequant(p, p, p, 128, 128, 9, None) == -4
    # null pointers
    assert lib.mdy_act_quant(None, p, p, 4, 128, 128, 4, 128, 1, 1, 0, None) == -1
    assert lib.mdy_fp8_gemm_nt(p, p, 1, 1, p, None, p, None, 4, 4, 128, 0, None) == -1
    # misaligned output
    assert lib.mdy_act_quant(p, p + 4, p, 4, 128, 128, 4, 128, 1, 1, 0, None) == -3
    # y_t without s_t
    assert lib.mdy_weight_quant(p, p, p, p, None, 128, 128, 128, 1, 128, 128, 1, None) == -1
    # negative / inconsistent sizes
    assert lib.mdy_fp8_gemm_nt(p, p, 1, 1, p, p, p, None, -1, 4, 128, 0, None) == -2
    assert lib.mdy_act_quant(p, p, p, 8, 128, 128, 4, 128, 1, 1, 0, None) == -2
    # empty problems are no-ops that never reach a device
    assert lib.mdy_act_quant(None, None, None, 0, 0, 0, 0, 0, 1, 1, 0, None) == 0
    assert lib.mdy_fp8_gemm_nt(p, p, 1, 1, p, p, p, None, 0, 4, 128, 0, None) == 0
    assert lib.mdy_add_bias(p, p, 0, 16, None) == 0


def test_argument_validation_of_the_later_entry_points(lib):
    buf = ctypes.create_string_buffer(8192)
    p = (ctypes.addressof(buf) + 255) // 256 * 256
    # GEMM with a workspace: negative size, misaligned buffer, empty problem, workspace query of a bad shape
    assert lib.mdy_fp8_gemm_nt_ws(p, p, 1, 1, p, p, p, None, 4, 4, 128, 0, p, -1, None) == -2
    assert lib.mdy_fp8_gemm_nt_ws(p, p, 1, 1, p, p, p, None, 4, 4, 128, 0, p + 4, 64, None) == -3
    assert lib.mdy_fp8_gemm_nt_ws(p, p, 1, 1, p, p, p, None, 0, 4, 128, 0, None, 0, None) == 0
    assert lib.mdy_fp8_gemm_nt_ws(p, p, 1, 1, p, p, p, None, 4, 4, 128, 5, None, 0, None) == -4
    assert lib.mdy_fp8_gemm_workspace_bytes(-1, 4, 128) == 0 and lib.mdy_fp8_gemm_workspace_bytes(4, 4, 0) == 0
    assert lib.mdy_fp8_gemm_workspace_bytes(128, 1536, 4096) >= 2 * 128 * 1536 * 4      # split along K
    assert lib.mdy_fp8_gemm_workspace_bytes(1, 7168, 2048) == 0                          # decode: never
    # grouped GEMM: no group table, a negative group, too many groups, nothing to do
    splits = (ctypes.c_int64 * 3)(4, -1, 4)
    assert lib.mdy_fp8_grouped_gemm_nt(p, p, 1, 1, p, p, p, None, None, 3, 4, 128, 0, None) == -1
    assert lib.mdy_fp8_grouped_gemm_nt(p, p, 1, 1, p, p, p, None, splits, 3, 4, 128, 0, None) == -2
    assert lib.mdy_fp8_grouped_gemm_nt(p, p, 1, 1, p, p, p, None, splits, (1 << 20) + 1, 4, 128, 0, None) == -2
    zero = (ctypes.c_int64 * 2)(0, 0)
    assert lib.mdy_fp8_grouped_gemm_nt(p, p, 1, 1, p, p, p, None, zero, 2, 4, 128, 0, None) == 0
    assert lib.mdy_fp8_grouped_gemm_nt(None, None, 1, 1, None, None, None, None, None, 0, 4, 128, 0, None) == 0
    # training quantizer: unknown transposed-scale mode, unpadded sizes, scale stride shorter than the rows
    assert lib.mdy_quant_transpose(p, p, p, p, p, 128, 128, 128, 1, 128, 128, 128, 7, None) == -4
    assert lib.mdy_quant_transpose(p, p, p, p, p, 100, 128, 128, 1, 100, 128, 128, 0, None) == -2
    assert lib.mdy_quant_transpose(p, p, p, p, p, 128, 128, 128, 1, 128, 128, 64, 0, None) == -2
    assert lib.mdy_quant_transpose(p, p, p, None, p, 128, 128, 128, 1, 128, 128, 128, 0, None) == -1
    # SwiGLU: nothing to write, quantized output without scales, row stride shorter than the row
    assert lib.mdy_swiglu(p, None, None, None, 4, 128, 256, 0, 4, 128, 1, 1, 0, None) == -1
    assert lib.mdy_swiglu(p, None, p, None, 4, 128, 256, 0, 4, 128, 1, 1, 0, None) == -1
    assert lib.mdy_swiglu(p, p, None, None, 4, 128, 200, 0, 0, 0, 1, 1, 0, None) == -2
    assert lib.mdy_swiglu(p, None, p, p, 4, 128, 256, 0, 4, 100, 1, 1, 0, None) == -2
    assert lib.mdy_swiglu(p, p, None, None, 0, 128, 256, 0, 0, 0, 1, 1, 0, None) == 0
    # diagnostics
    assert lib.mdy_quotient_selfcheck(None, 0, 16, 0, None) == -1
    assert lib.mdy_quotient_selfcheck(p, 16, 8, 0, None) == -2
    assert lib.mdy_cast_f32_to_e4m3(p, p, -1, 0, None) == -2 and lib.mdy_cast_f32_to_e4m3(None, None, 0, 0, None) == 0
    assert lib.mdy_fp8_last_error()            # the last message is kept


def test_python_wrappers_keep_reference_preconditions():
    import mdy_triton_amd as m
    x = torch.zeros(4, 130, dtype=torch.bfloat16)
    with pytest.raises(AssertionError):
        m.act_quant(x)                      # last dim % 128 (offical_kernel.py:23)
    with pytest.raises(AssertionError):
        m.act_quant(torch.zeros(4, 256, dtype=torch.bfloat16)[:, ::2])  # contiguity (:22)
    with pytest.raises(AssertionError):
        m.weight_dequant(torch.zeros(2, 128, 128).to(torch.float8_e4m3fn), torch.zeros(1, 1))  # 2-D (:48)
    with pytest.raises(RuntimeError, match="no CPU path"):
        m.act_quant(torch.zeros(4, 128, dtype=torch.bfloat16))
    with pytest.raises(RuntimeError, match="no CPU path"):
        m.DeepLinear(256, 128, dtype=torch.bfloat16)(torch.zeros(4, 256, dtype=torch.bfloat16))


def test_product_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "mdy_triton_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h", ".cpp")):
                text = open(os.path.join(dirpath, f)).read()
                assert not re.search(r"^\s*(from|import)\s+oracle\b", text, flags=re.M), f


def test_gemm_path_query_needs_no_gpu(lib):
    """mdy_fp8_gemm_path only inspects sizes, strides and pointer alignment."""
    q = lib.mdy_fp8_gemm_path
    assert q(None, None, 56, 1, 4096, 18432, 7168, 1) == 3          # MFMA tiles
    assert q(None, None, 56, 1, 4096, 18432, 7168, 0) == 3
    assert q(None, None, 16, 1, 16, 7168, 2048, 1) == 1             # weight streaming
    assert q(None, None, 2, 1, 300, 200, 200, 1) == 0               # K % 128 != 0: scalar
    assert q(None, None, 1025, 1, 100, 256, 131200, 1) == 0         # K > 65536 and M > 64: scalar
    assert q(8, None, 56, 1, 4096, 1536, 7168, 1) == 0              # misaligned operand: scalar
    assert q(None, None, 32, 1, 128, 1536, 4096, 1) == 4            # split along K with a workspace ...
    assert q(None, None, 32, 1, 128, 1536, 4096, 0) == 3            # ... plain tiles without
    assert q(None, None, 56, 1, 0, 5, 128, 0) == -2


def test_workspace_query_is_what_the_chosen_kernel_uses(lib):
    """Room for slabs of K only where the call is cut along K; otherwise that of a transposed copy of the scales, or none."""
    import random
    r, cut = random.Random(7), 0
    shapes = [(256, 4096, 4096)] + [(r.randrange(1, 1600), r.randrange(1, 9000), 128 * r.randrange(1, 130)) for _ in range(4000)]
    for M, N, K in shapes:
        need, path = lib.mdy_fp8_gemm_workspace_bytes(M, N, K), lib.mdy_fp8_gemm_path(None, None, K // 128, 1, M, N, K, 1)
        scales = (M * (K // 128) * 4 + 255) // 256 * 256
        cut += path == 4
        assert need % (4 * M * N) == 0 and need >= 8 * M * N if path == 4 else need in (0, scales), (M, N, K)
    assert cut > 100


def test_swiglu_workspace_holds_slabs_or_a_product(lib):
    """The slabs alone where they go to the activation quantizer, else the product behind what its GEMM needs."""
    q, gemm = lib.mdy_fp8_gemm_swiglu_workspace_bytes, lib.mdy_fp8_gemm_workspace_bytes
    for M, N, K in ((200, 4096, 7168), (197, 2048, 7168), (61, 1536, 7168)):
        assert q(M, N, K) == gemm(M, N, K) > 4 * M * N
    assert q(250, 1034, 4096) == -(-gemm(250, 1034, 4096) // 256) * 256 + 2 * 250 * 1034 and gemm(250, 1034, 4096) > 0      # halves of odd columns
    assert q(5, 1536, 2048) == 2 * 5 * 1536


def test_form_queries(lib):
    """The kernel that a call runs: within the family that the path query names, with the slabs that the workspace query makes room for."""
    import random
    r = random.Random(11)
    path_of = {0: 0, 1: 1, 2: 2, 3: 1}
    for _ in range(3000):
        M, N, K, ws = r.choice([r.randrange(1, 65), r.randrange(65, 6000)]), r.randrange(1, 30000), 128 * r.randrange(1, 600), r.randrange(2)
        v = lib.mdy_fp8_gemm_form(M, N, K, ws)
        form, slabs = v & 255, v >> 8
        assert lib.mdy_fp8_gemm_path(None, None, K // 128, 1, M, N, K, ws) == (4 if slabs else path_of.get(form, 3)), (M, N, K)
        assert slabs == 0 or (ws == 1 and lib.mdy_fp8_gemm_workspace_bytes(M, N, K) == 4 * slabs * M * N), (M, N, K)
        slabs = lib.mdy_fp8_gemm_rowscaled_form(M, N, K, 1) >> 8
        assert lib.mdy_fp8_gemm_rowscaled_workspace_bytes(M, N, K) == 4 * slabs * M * N and lib.mdy_fp8_gemm_rowscaled_form(M, N, K, 0) >> 8 == 0
    assert lib.mdy_fp8_gemm_form(4, 4, 100, 1) == 0 and lib.mdy_fp8_gemm_form(0, 4, 128, 1) == -2
    assert lib.mdy_fp8_gemm_rowscaled_form(4, 4, 100, 1) == -2
    form = lambda rows, N, K: lib.mdy_fp8_grouped_gemm_form((ctypes.c_int64 * len(rows))(*rows), len(rows), N, K)
    assert form([1, 0, 7], 512, 1024) == 1 and form([24] * 9, 3000, 2560) == 2 and form([4, 4], 512, 100) == 15 and form([2] * 300, 48, 128) == 15
    assert form([0, 0], 512, 128) == -2 and form([-1, 4], 512, 128) == -2 and lib.mdy_fp8_grouped_gemm_form(None, 2, 512, 128) == -1


@pytest.mark.parametrize("M,N,K,tiles", [(59, 6464, 2176, False), (47, 6837, 2432, False), (22, 10112, 1280, False), (28, 8704, 640, False),
                                         (48, 4352, 640, False), (30, 15552, 2176, True), (25, 15040, 4608, True), (33, 8256, 2688, True),
                                         (64, 4928, 1792, False), (62, 6208, 3200, True)])
def test_small_rows_leave_the_whole_line_kernel_where_its_rounds_cost(lib, M, N, K, tiles):
    """17 to 64 rows: tiles in one launch only where the whole-line kernel needs another round or pass (256 CUs)."""
    assert (lib.mdy_fp8_gemm_form(M, N, K, 1) == 1) != tiles


def grouped_form(lib, rows, N, K):
    return lib.mdy_fp8_grouped_gemm_form((ctypes.c_int64 * len(rows))(*rows), len(rows), N, K)


def test_grouped_form_of_33_to_64_rows(lib):
    """Fewer than 144 strips: the whole-line kernel, which reads weights from HBM faster than pieces of 128 rows do."""
    assert grouped_form(lib, [45] * 8, 1344, 1792) == grouped_form(lib, [58] * 4, 2880, 2048) == grouped_form(lib, [40] * 4, 2688, 1024) == 1
    assert grouped_form(lib, [33] * 8, 2752, 1408) == 19 and grouped_form(lib, [64] * 8, 2304, 2048) == 19 and grouped_form(lib, [33] * 8, 2752, 2304) == 2


def test_grouped_form_of_a_quarter_round(lib):
    """Up to a quarter of a round behind whole ones, in whole tile rows more than a round of 128-column pieces: quarters of tiles."""
    assert grouped_form(lib, [104] * 32, 4608, 896) == grouped_form(lib, [256] * 12 + [300, 70, 200], 5056, 256) == 21
    assert grouped_form(lib, [256] * 16 + [130, 1, 257], 3848, 640) == 16 and grouped_form(lib, [256] * 17 + [130, 1, 257], 3848, 640) == 17


def test_rowscaled_slab_counts(lib):
    """Slabs of K of the row-scaled GEMM (kernel 10, 128x256 tiles): the counts in use before its times were estimated."""
    for shape, slabs in (((768, 640, 8192), 11), ((1536, 768, 4480), 5), ((512, 1152, 5248), 7), ((1152, 640, 7680), 9), ((1024, 1024, 8192), 8)):
        assert lib.mdy_fp8_gemm_rowscaled_form(*shape, 1) == 10 | slabs << 8, shape


def test_short_calls_are_not_cut_by_an_estimate(lib):
    """What one launch finishes in less than the host takes for a second one stays in one launch (256 CUs)."""
    for shape in ((19, 576, 7424), (30, 576, 7552), (68, 384, 2048), (163, 384, 2176)):
        assert lib.mdy_fp8_gemm_form(*shape, 1) >> 8 == 0, shape
    for shape in ((20, 768, 10112), (109, 1280, 2560), (64, 832, 4096)):
        assert lib.mdy_fp8_gemm_form(*shape, 1) >> 8 > 1, shape


def test_large_tiles_that_just_miss_a_round(lib):
    """128x256 tiles in place of 256x256: at any K where they need no more rounds, from 16 K blocks on where they need one more (256 CUs)."""
    assert lib.mdy_fp8_gemm_form(2383, 6656, 2176, 0) == lib.mdy_fp8_gemm_form(2841, 5632, 128, 0) == 10
    assert lib.mdy_fp8_gemm_form(7172, 3264, 128, 0) == lib.mdy_fp8_gemm_form(1854, 12480, 1920, 0) != 10
    assert lib.mdy_fp8_gemm_form(1854, 12480, 2048, 0) == 10


def test_one_tile_row_keeps_the_slabs_of_a_weight_from_memory(lib):
    """65 to 128 rows: 128x64 tiles in one launch, or in fewer slabs, are faster with the operands in the caches and up to 15 % slower without (256 CUs)."""
    for shape, form in (((107, 8576, 4736), 7 | 3 << 8), ((66, 12032, 6784), 9 | 4 << 8), ((115, 6208, 6912), 7 | 5 << 8), ((104, 6080, 5248), 7 | 5 << 8)):
        assert lib.mdy_fp8_gemm_form(*shape, 1) == form, shape
    assert lib.mdy_fp8_gemm_form(123, 1088, 1152, 1) == lib.mdy_fp8_gemm_form(120, 2112, 1280, 1) == 4
    assert lib.mdy_fp8_gemm_form(777, 2112, 7168, 1) == 6      # seven tile rows: as before
