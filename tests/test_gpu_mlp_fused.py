"""The up/gate projection that goes from its K slabs straight to the activation quantizer: the bits of the separate operators."""
import pytest
import torch

import mdy_triton_amd as m
from mdy_triton_amd import fp8 as L, fp8_kernel as FK
from mdy_triton_amd._torch_glue import host, lib

pytestmark = pytest.mark.gpu
E4M3 = torch.float8_e4m3fn


# slabs of the up/gate projection (0: one launch) with the sizes of either dialect; tiles and the whole-line kernel's; ragged rows; halves of 8 k and of odd columns
@pytest.mark.parametrize("M,H,I,slabs", [(200, 7168, 2048, (4, 4)), (300, 7168, 2048, (2, 2)), (197, 7168, 1024, (4, 4)), (100, 16384, 256, (16, 16)),
                                         (61, 7168, 768, (5, 5)), (40, 4096, 512, (4, 4)), (777, 7168, 1056, (0, 0)), (333, 7168, 1000, (5, 3)),
                                         (250, 4096, 517, (4, 4)), (5, 2048, 768, (0, 0)), (2048, 2048, 512, (0, 0)), (130, 6528, 352, (8, 8)),
                                         (211, 4224, 320, (7, 7)), (110, 11136, 2240, (7, 7)), (185, 7552, 2312, (3, 3)), (326, 7040, 400, (6, 6)),
                                         (83, 3840, 568, (6, 6)), (104, 9344, 336, (9, 9)), (169, 12544, 280, (11, 11))])
@pytest.mark.parametrize("order", ["up-gate", "gate-up"])
@pytest.mark.parametrize("dialect", ["deeplinear", "official"])
def test_same_bits_as_the_operators_in_turn(M, H, I, slabs, order, dialect):
    if dialect == "official" and I % 128:
        I = I // 128 * 128
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        assert lib().mdy_fp8_gemm_form(M, 2 * I, H, 1) >> 8 == slabs[dialect == "official"]
    g = torch.Generator(device="cuda").manual_seed(M + H + I)
    x = torch.randn(M, H, generator=g, device="cuda").bfloat16()
    wu, wd = ((torch.randn(*s, generator=g, device="cuda") * 0.02).bfloat16() for s in ((2 * I, H), (H, I)))
    deep = dialect == "deeplinear"
    if deep:
        (qu, su), (qd, sd) = (L.quant_weight(w)[:2] for w in (wu, wd))
        qx, sx = L.quant_input(x)[:2]
        up_gate = L.fp8_matmul(qx[:M], sx[:M], qu[:2 * I], su[:-(-2 * I // 128)])
        qa, sa = FK.silu_act_quant(up_gate, order, dialect=dialect)
        ref = L.fp8_matmul(qa[:M], sa[:M], qd[:H], sd[:-(-H // 128)])
    else:
        (qu, su), (qd, sd) = (FK.weight_quant_block(w, dtype=E4M3) for w in (wu, wd))
        up_gate = FK.fp8_matmul(*[t for p in zip(FK.act_quant_block(x, dtype=E4M3), (qu, su)) for t in p])
        qa, sa = FK.silu_act_quant(up_gate, order, dialect=dialect)
        ref = FK.fp8_matmul(qa, qd, sa, sd)
    got = host().mlp(x, qu, su, 2 * I, qd, sd, H, int(order == "gate-up"), int(deep))
    assert got is not None and torch.equal(got, ref)
    assert host().mlp(x[:, :-256], qu, su, 2 * I, qd, sd, H, 0, int(deep)) is None      # operands that do not fit together


def test_order_is_looked_at():
    mlp = m.Fp8MLP(256, 256, device="cuda", dialect="deeplinear", fp8_dtype=E4M3)
    x = torch.randn(4, 256, device="cuda", dtype=torch.bfloat16)
    for dialect in ("official", "deeplinear"):
        with pytest.raises(Exception), torch.no_grad():
            FK.fp8_ckpt_mlp(x, mlp.up_gate_proj.weight, mlp.down_proj.weight, E4M3, "down-up", dialect)


def test_slabs_are_what_these_shapes_take():
    q = lib().mdy_fp8_gemm_workspace_bytes
    assert q(200, 4096, 7168) == 4 * 200 * 4096 * 4 and q(197, 2048, 7168) > 0 and q(61, 1536, 7168) > 0 and q(5, 1536, 2048) == 0


# split along K, and not: the quantized input, the projection and the down projection's result are not all held at once
@pytest.mark.parametrize("M,H,I", [(500, 16384, 2048), (2048, 8192, 512)])
def test_forward_peak_memory(M, H, I):
    g = torch.Generator(device="cuda").manual_seed(I)
    x = torch.randn(M, H, generator=g, device="cuda").bfloat16()
    (qu, su), (qd, sd) = (L.quant_weight((torch.randn(*s, generator=g, device="cuda") * 0.02).bfloat16())[:2] for s in ((2 * I, H), (H, I)))
    scales = lambda k: M * k // 128 * 4
    up = lib().mdy_fp8_gemm_swiglu_workspace_bytes(M, 2 * I, H)
    act = M * I + scales(I)
    bound = act + max(M * H + scales(H) + up, 2 * M * H + lib().mdy_fp8_gemm_workspace_bytes(M, H, I))
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    y = host().mlp(x, qu, su, 2 * I, qd, sd, H, 0, 1)
    assert y is not None and torch.cuda.max_memory_allocated() - before <= bound + (2 << 20)      # what the allocator rounds up


def test_operands_that_the_slabs_do_not_take():
    """A weight on 8 bytes runs the scalar kernel: the product lies where the slabs would."""
    M, I, K = 70, 256, 4096
    g = torch.Generator(device="cuda").manual_seed(3)
    qa, sa = FK.act_quant_block(torch.randn(M, K, generator=g, device="cuda").bfloat16(), dtype=E4M3)
    qb, sb = FK.weight_quant_block((torch.randn(2 * I, K, generator=g, device="cuda") * 0.05).bfloat16(), dtype=E4M3)
    odd = torch.empty(qb.numel() + 8, dtype=torch.uint8, device="cuda")[8:]
    odd.copy_(qb.view(torch.uint8).flatten())
    C, need = lib(), lib().mdy_fp8_gemm_swiglu_workspace_bytes(M, 2 * I, K)
    assert C.mdy_fp8_gemm_path(None, None, K // 128, 1, M, 2 * I, K, 1) == 4 and C.mdy_fp8_gemm_path(None, 8, K // 128, 1, M, 2 * I, K, 1) == 0
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")
    y, s = torch.empty(M, I, dtype=E4M3, device="cuda"), torch.empty(M, I // 128, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert C.mdy_fp8_gemm_swiglu(qa.data_ptr(), sa.data_ptr(), K // 128, 1, odd.data_ptr(), sb.data_ptr(), M, 2 * I, K, 0, y.data_ptr(), s.data_ptr(), M, I,
                                 I // 128, 1, 0, ws.data_ptr(), need, stream) == 0
    c = torch.empty(M, 2 * I, dtype=torch.bfloat16, device="cuda")
    assert C.mdy_fp8_gemm_nt(qa.data_ptr(), sa.data_ptr(), K // 128, 1, odd.data_ptr(), sb.data_ptr(), c.data_ptr(), None, M, 2 * I, K, 0, stream) == 0
    ry, rs = FK.silu_act_quant(c, "up-gate")
    assert torch.equal(y.view(torch.uint8), ry.view(torch.uint8)) and torch.equal(s, rs)


class _Without:
    """The native host side with one function that takes no call."""

    def __init__(self, module, name):
        self._module, self._name = module, name

    def __getattr__(self, name):
        return (lambda *args: None) if name == self._name else getattr(self._module, name)


# one to many row tiles with ragged last ones, 128-column halves whose padding to 256 is a tile of its own, an outlier beyond the clamp
@pytest.mark.parametrize("M,H,I", [(1, 256, 128), (129, 384, 384), (300, 512, 256), (1000, 1280, 640), (640, 256, 2048)])
@pytest.mark.parametrize("order", ["up-gate", "gate-up"])
@pytest.mark.parametrize("dialect,fmt", [("official", E4M3), ("official", torch.float8_e5m2), ("deeplinear", E4M3)])
def test_backward_same_bits_as_the_operators_in_turn(monkeypatch, M, H, I, order, dialect, fmt):
    g = torch.Generator(device="cuda").manual_seed(M + H + I)
    x = torch.randn(M, H, generator=g, device="cuda").bfloat16().requires_grad_(True)
    wu, wd = ((torch.randn(*s, generator=g, device="cuda") * 0.1).bfloat16().requires_grad_(True) for s in ((2 * I, H), (H, I)))
    dy = torch.randn(M, H, generator=g, device="cuda").bfloat16()
    dy[M // 2, 3] = 3e4
    if dialect == "deeplinear" and M > 1:      # (a scale of zero makes NaN in the official dialect)
        dy[-1] = 0
    got, ref = [], []
    for out in (got, ref):
        y = FK.fp8_ckpt_mlp(x, wu, wd, fmt, order, dialect)
        if out is ref:
            module = host()
            assert module.mlp_backward(dy, x, wu, wd, int(order == "gate-up"), 0 if fmt == E4M3 else 1, int(dialect == "deeplinear")) is not None
            monkeypatch.setattr(FK, "host", lambda: _Without(module, "mlp_backward"))
        out += torch.autograd.grad(y, (x, wu, wd), dy)
    for a, b in zip(got, ref):
        assert a.shape == b.shape and torch.equal(a, b)
    assert all(t.abs().sum() > 0 for t in got)


def test_arguments_without_device():
    import ctypes
    L_ = lib()
    p = ctypes.addressof(ctypes.create_string_buffer(8192)) // 256 * 256 + 256
    a = (p,) * 8
    assert L_.mdy_swiglu_bwd_quant(*a, 100, 64, 0, 128, 128, 0, None) == -2 and L_.mdy_swiglu_bwd_quant(*a, 100, 128, 0, 100, 128, 0, None) == -2
    assert L_.mdy_swiglu_bwd_quant(*a, 0, 128, 0, 128, 128, 0, None) == -2 and L_.mdy_swiglu_bwd_quant(*a, 0, 128, 0, 0, 128, 0, None) == 0
    assert L_.mdy_swiglu_bwd_quant(p + 8, *a[1:], 100, 128, 0, 128, 128, 0, None) == -3 and L_.mdy_swiglu_bwd_quant(*a, 100, 128, 0, 128, 128, 7, None) == -4
    g = (p, p, 1, 1, p, p)
    assert L_.mdy_fp8_gemm_swiglu(*g, 4, 255, 128, 0, p, p, 4, 128, 1, 4, 1, p, 1 << 20, None) == -2      # an odd number of columns
    assert L_.mdy_fp8_gemm_swiglu(*g, 4, 256, 128, 0, p, p, 4, 128, 1, 4, 1, p, 64, None) == -2           # workspace too small
    assert L_.mdy_fp8_gemm_swiglu(*g, 4, 256, 128, 0, p, p, 4, 128, 1, 4, 1, None, 1 << 20, None) == -1
