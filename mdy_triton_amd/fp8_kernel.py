"""SwiGLU and block quantizers of the FP8 MLP on MI355X.

Drop-in for the parts of /root/reference/triton_kernels/deepseekv3/fp8_kernel.py that sit
directly before the FP8 linear path: silu_fwd / silu_bwd / triton_silu (fp8_kernel.py:384-434),
weight_quant_block (:124-138), plus silu_act_quant, which fuses the `silu_fwd -> act_quant`
pair of the FP8 MLP (fp8_kernel.py:447-450, 500-515) into one pass over the up/gate tensor; and for
that file's own linear layer in the official dialect (s = amax / finfo.max, no clamp, no eps):
act_quant_block (:62-87), fp8_matmul (:214-252), fp8_matmul_bwd (:254-257), Fp8Linear (:259-313).
Both float8_e4m3fn and float8_e5m2 (the reference's default dtype, fp8_kernel.py:62, 124, 303) are implemented for the
official-dialect functions, on the same kernels with the byte format as a template parameter (an e5m2 product beyond what
those take, K > 65536, unaligned operands or scales spanning 2^31 bytes, runs the GEMM with row scales on both operands, the
weight's 128x128 block scales expanded to one per row).  The DeepLinear dialect and the fused silu_act_quant are e4m3fn only.
"""
from typing import Optional, Tuple

import torch

from ._torch_glue import FP8, check, gemm_workspace, host, lib, on_device, parameter_of, ptr, require_gpu, rowscaled_workspace, stream_ptr, xt_code

_ORDERS = ("up-gate", "gate-up")


E5M2 = torch.float8_e5m2


def _require_e4m3(fp8_dtype, who: str):
    if fp8_dtype != FP8:
        raise TypeError("%s: only torch.float8_e4m3fn is implemented here, got %s" % (who, fp8_dtype))


def _fp8_mode(fp8_dtype, who: str):
    """(quantizer mode, GEMM operand format) of an fp8 dtype: official dialect with e4m3fn bytes, or with e5m2 bytes."""
    if fp8_dtype == FP8:
        return 0, 0
    if fp8_dtype == E5M2:
        return 2, 1
    raise TypeError("%s: fp8 dtype must be torch.float8_e4m3fn or torch.float8_e5m2, got %s" % (who, fp8_dtype))


def _flatten_up_gate(x: torch.Tensor, order: str, who: str):
    assert order in _ORDERS, "please indicate the order of input, up-gate or gate-up"
    if x.dtype != torch.bfloat16:
        raise TypeError("%s expects a bfloat16 tensor, got %s" % (who, x.dtype))
    if x.size(-1) % 2 != 0:
        raise ValueError("%s: the last dimension holds up and gate and must be even" % who)
    x2 = x.reshape(-1, x.size(-1))
    if x2.numel() > 0 and x2.stride(1) != 1:
        x2 = x2.contiguous()
    return x2, x2.size(0), x2.size(1) // 2


def silu_fwd(x: torch.Tensor, order: str = "up-gate") -> torch.Tensor:
    """act = silu(gate) * up as bf16 [..., N] from x [..., 2N] (fp8_kernel.py:384-402)."""
    if order in _ORDERS:
        done = host().silu_fwd(x, int(order == "gate-up"))
        if done is not None:
            return done
    x2, M, N = _flatten_up_gate(x, order, "silu_fwd")
    dev = require_gpu(x)
    y = torch.empty(*x.shape[:-1], N, device=dev, dtype=x.dtype)
    if M * N == 0:
        return y
    with on_device(dev):
        check(lib().mdy_swiglu(ptr(x2), ptr(y), None, None, M, N, x2.stride(0) if M else 2 * N, int(order == "gate-up"),
                               0, 0, 0, 0, 0, stream_ptr(dev)), "silu_fwd")
    return y


def silu_bwd(dy: torch.Tensor, x: torch.Tensor, order: str = "up-gate") -> torch.Tensor:
    """Gradient of silu_fwd with respect to x (fp8_kernel.py:404-421); dx has x's shape."""
    if order in _ORDERS:
        done = host().silu_bwd(dy, x, int(order == "gate-up"))
        if done is not None:
            return done
    x2, M, N = _flatten_up_gate(x, order, "silu_bwd")
    dev = require_gpu(x, dy)
    if dy.dtype != torch.bfloat16 or dy.numel() != M * N:
        raise ValueError("silu_bwd: dy must be bfloat16 with %d elements" % (M * N))
    dy2 = dy.reshape(M, N).contiguous()
    dx = torch.empty(x.shape, device=dev, dtype=x.dtype)
    if M * N == 0:
        return dx
    with on_device(dev):
        check(lib().mdy_swiglu_bwd(ptr(x2), ptr(dy2), ptr(dx), M, N, x2.stride(0) if M else 2 * N,
                                   int(order == "gate-up"), stream_ptr(dev)), "silu_bwd")
    return dx


class _SiluOps(torch.autograd.Function):
    """fp8_kernel.py:423-433."""

    @staticmethod
    def forward(ctx, x, order="up-gate"):
        ctx.x = x
        ctx.order = order
        return silu_fwd(x, order)

    @staticmethod
    def backward(ctx, dy):
        return silu_bwd(dy, ctx.x, ctx.order), None


triton_silu = _SiluOps.apply


def silu_act_quant(x: torch.Tensor, order: str = "up-gate", return_act: bool = False, dialect: str = "official"):
    """One pass: act = silu_fwd(x, order) and its 1x128 quantization.

    dialect "official": (y, s) as offical_kernel.act_quant(act) returns them (N % 128 == 0);
    dialect "deeplinear": (y, s) as fp8.quant_input(act, only_forward=True) returns them (padded,
    column-major scales).  With return_act=True the bf16 act comes back as a third value (the
    backward pass needs it); otherwise it is never written to memory.
    """
    if not return_act and order in _ORDERS and dialect in ("official", "deeplinear"):
        done = host().silu_act_quant(x, int(order == "gate-up"), int(dialect == "deeplinear"))
        if done is not None:
            return done
    x2, M, N = _flatten_up_gate(x, order, "silu_act_quant")
    dev = require_gpu(x)
    act = torch.empty(*x.shape[:-1], N, device=dev, dtype=x.dtype) if return_act else None
    gate_first = int(order == "gate-up")
    xs = x2.stride(0) if M else 2 * N
    if dialect == "official":
        assert N % 128 == 0
        y = torch.empty(*x.shape[:-1], N, device=dev, dtype=FP8)
        s = torch.empty(*x.shape[:-1], N // 128, device=dev, dtype=torch.float32)
        if M * N > 0:
            with on_device(dev):
                check(lib().mdy_swiglu(ptr(x2), ptr(act), ptr(y), ptr(s), M, N, xs, gate_first, M, N, N // 128, 1, 0,
                                       stream_ptr(dev)), "silu_act_quant")
    elif dialect == "deeplinear":
        PN = (N + 255) // 256 * 256
        PM = (M + 3) // 4 * 4
        y = torch.empty(PM, PN, device=dev, dtype=FP8)
        sbuf = torch.empty(PN // 128, PM, device=dev, dtype=torch.float32)
        if PM * PN > 0:
            with on_device(dev):
                check(lib().mdy_swiglu(ptr(x2), ptr(act), ptr(y), ptr(sbuf), M, N, xs, gate_first, PM, PN, 1, PM, 1,
                                       stream_ptr(dev)), "silu_act_quant")
        s = sbuf.transpose(0, 1)
    else:
        raise ValueError("dialect must be 'official' or 'deeplinear'")
    return (y, s, act) if return_act else (y, s)


def weight_quant_block(x: torch.Tensor, BLOCK_M: int = 128, BLOCK_N: int = 128,
                       dtype: torch.dtype = E5M2) -> Tuple[torch.Tensor, torch.Tensor]:
    """128x128 block quantizer with s = amax / finfo(dtype).max (fp8_kernel.py:124-138, kernel :88-122); dtype
    defaults to float8_e5m2 as in the reference.

    x [M, N] (any strides, N % 128 == 0); returns y [M, N] of `dtype` and s [M//128, N//128].
    """
    assert x.size(-1) % BLOCK_N == 0
    if BLOCK_M != 128 or BLOCK_N != 128:
        raise ValueError("only 128x128 blocks are implemented (the reference default)")
    mode, fmt = _fp8_mode(dtype, "weight_quant_block")
    done = host().block_copies(x, True, False, fmt)
    if done is not None:
        return done[:2]
    if x.dim() != 2:
        raise TypeError("weight_quant_block expects a 2-D tensor")
    xt = xt_code(x, "weight_quant_block")
    dev = require_gpu(x)
    M, N = x.shape
    if M % 128 != 0:
        raise ValueError("weight_quant_block: M must be a multiple of 128 (the reference drops the ragged rows)")
    y = torch.empty(M, N, device=dev, dtype=dtype)
    s = torch.empty(M // 128, N // 128, device=dev, dtype=torch.float32)
    with on_device(dev):
        check(lib().mdy_weight_quant_typed(ptr(x), xt, ptr(y), ptr(s), None, None, M, N, x.stride(0), x.stride(1), M, N, mode,
                                           stream_ptr(dev)), "weight_quant_block")
    return y, s


def _weight_quant_both(w: torch.Tensor, rows: bool, transposed: bool, dtype: torch.dtype, who: str):
    """One pass over w [N, K] (multiples of 128, any strides): (y, s) as weight_quant_block(w) gives them and (y_t, s_t) as
    weight_quant_block(w.t()) gives them (a block's scale does not depend on its orientation); None for what is not asked for.
    Reading w once, in rows, instead of once in rows and once in columns: [4096, 4096] e5m2 14 + 40 -> 19 us."""
    mode, fmt = _fp8_mode(dtype, who)
    done = host().block_copies(w, rows, transposed, fmt)
    if done is not None:
        return done
    xt = xt_code(w, who)
    dev = require_gpu(w)
    N, K = w.shape
    if N % 128 != 0:
        raise ValueError("%s: the weight's rows must be a multiple of 128 (the reference drops the ragged rows)" % who)
    assert K % 128 == 0
    y = torch.empty(N, K, device=dev, dtype=dtype) if rows else None
    s = torch.empty(N // 128, K // 128, device=dev, dtype=torch.float32) if rows else None
    y_t = torch.empty(K, N, device=dev, dtype=dtype) if transposed else None
    s_t = torch.empty(K // 128, N // 128, device=dev, dtype=torch.float32) if transposed else None
    with on_device(dev):
        check(lib().mdy_weight_quant_typed(ptr(w), xt, ptr(y), ptr(s), ptr(y_t), ptr(s_t), N, K, w.stride(0), w.stride(1), N, K, mode,
                                           stream_ptr(dev)), who)
    return y, s, y_t, s_t


def _act_quant_transposed(x2: torch.Tensor, with_rows: bool, who: str, dtype: torch.dtype = FP8, col_sum: Optional[torch.Tensor] = None):
    """x2 [M, N] (any strides) -> (y, s, y_t_padded, s_t): the official-dialect row-wise quantization (None, None
    unless with_rows) and the quantized transpose y_t [N, PM] with s_t [N, PM/128], PM = cdiv(M, 128) * 128.  col_sum (bf16
    x2): a bf16 [N] tensor that receives the sums of x2's columns from the same pass."""
    mode, fmt = _fp8_mode(dtype, who)
    if col_sum is None:
        done = host().act_copies(x2, with_rows, fmt)
        if done is not None:
            return done
    xt = xt_code(x2, who)
    dev = require_gpu(x2)
    M, N = x2.shape
    PM = (M + 127) // 128 * 128
    y = torch.empty(PM, N, device=dev, dtype=dtype) if with_rows else None
    s = torch.empty(PM, N // 128, device=dev, dtype=torch.float32) if with_rows else None
    y_t = torch.empty(N, PM, device=dev, dtype=dtype)
    s_t = torch.empty(N, PM // 128, device=dev, dtype=torch.float32)
    if PM * N > 0:
        with on_device(dev):
            if col_sum is not None:
                part = torch.empty(PM // 128, N, device=dev, dtype=torch.float32)
                check(lib().mdy_quant_transpose_colsum(ptr(x2), ptr(y), ptr(s), ptr(y_t), ptr(s_t), M, N, x2.stride(0), x2.stride(1), PM, N, 0,
                                                       mode, ptr(part), ptr(col_sum), stream_ptr(dev)), who)
                return y, s, y_t, s_t
            check(lib().mdy_act_quant_transpose(ptr(x2), xt, ptr(y), ptr(s), ptr(y_t), ptr(s_t), M, N, x2.stride(0), x2.stride(1),
                                                PM, N, mode, stream_ptr(dev)), who)
    return y, s, y_t, s_t


def act_quant_block(x: torch.Tensor, transpose: bool = False, dtype: torch.dtype = E5M2,
                    BLOCK_N: int = 128) -> Tuple[torch.Tensor, torch.Tensor]:
    """1x128 quantizer with s = amax / finfo(dtype).max (fp8_kernel.py:62-87); dtype defaults to float8_e5m2 as in the
    reference.

    transpose=False: (y like x, s [..., N/128]); with float8_e4m3fn the same as offical_kernel.act_quant.
    transpose=True: the flattened [M, N] input is quantized along M: y [N, M], s [N, cdiv(M, 128)] (a last group
    shorter than 128 is completed with zeros, as the reference's masked loads do).
    """
    assert x.size(-1) % BLOCK_N == 0
    if BLOCK_N != 128:
        raise ValueError("only BLOCK_N=128 is implemented (the reference default)")
    mode, fmt = _fp8_mode(dtype, "act_quant_block")
    if not transpose:
        done = host().act_quant(x, 128, fmt)
        if done is not None:
            return done
        xc = x if x.is_contiguous() else x.contiguous()
        if mode == 0:
            from .offical_kernel import act_quant
            return act_quant(xc)
        xt = xt_code(xc, "act_quant_block")
        dev = require_gpu(xc)
        K = xc.size(-1)
        M = xc.numel() // K if K else 0
        y = torch.empty_like(xc, dtype=dtype)
        s = xc.new_empty(*xc.size()[:-1], K // 128, dtype=torch.float32)
        with on_device(dev):
            check(lib().mdy_act_quant_typed(ptr(xc), xt, 128, ptr(y), ptr(s), M, K, K, M, K, K // 128, 1, mode, stream_ptr(dev)),
                  "act_quant_block")
        return y, s
    x2 = x.reshape(-1, x.size(-1))
    M = x2.size(0)
    _, _, y_t, s_t = _act_quant_transposed(x2, False, "act_quant_block", dtype)
    return (y_t if y_t.size(1) == M else y_t[:, :M].contiguous()), s_t


def fp8_matmul(x: torch.Tensor, w: torch.Tensor, scale_x: torch.Tensor, scale_w: torch.Tensor,
               bias: Optional[torch.Tensor] = None, have_w: bool = True) -> torch.Tensor:
    """bf16 y = x . w^T on block-scaled FP8 operands, both float8_e4m3fn or both float8_e5m2 (fp8_kernel.py:214-252).

    have_w=True (forward, input gradient): x [..., K] with scale_x [..., K/128], w [N, K] with 128x128 block scales
    scale_w [N/128, K/128], optional bias [N] added in fp32.  have_w=False (weight gradient): x [M, K] and w [N, K]
    both carry one scale per row and 128 columns, scale_x [M, cdiv(K,128)], scale_w [N, cdiv(K,128)]; a K that is not a
    multiple of 128 is completed with zeros.
    """
    if x.dtype != w.dtype:
        raise TypeError("fp8_matmul expects operands of one fp8 dtype, got %s and %s" % (x.dtype, w.dtype))
    _, fmt = _fp8_mode(x.dtype, "fp8_matmul")
    if have_w:
        done = host().fp8_gemm(x, scale_x, w, scale_w, torch.bfloat16, bias, fmt)
        if done is not None:
            return done
        assert x.size(-1) % 128 == 0, 'in forward x @ w.T'
        x2 = x.reshape(-1, x.size(-1))
        sx2 = scale_x.reshape(-1, scale_x.size(-1))
        if fmt == 0:
            from .offical_kernel import fp8_gemm
            fused = bias is not None and bias.dtype == torch.bfloat16        # the GEMM epilogue takes a bf16 bias
            y = fp8_gemm(x2 if x2.is_contiguous() else x2.contiguous(), sx2.contiguous(),
                         w if w.is_contiguous() else w.contiguous(), scale_w.contiguous(), out_dtype=torch.bfloat16,
                         bias=bias.contiguous() if fused else None)
        else:
            dev = require_gpu(x, w, scale_x, scale_w)
            M, K = x2.shape
            N = w.size(0)
            x2c, wc = (x2 if x2.is_contiguous() else x2.contiguous()), (w if w.is_contiguous() else w.contiguous())
            sxc, swc = sx2.contiguous(), scale_w.contiguous()
            scales_ok = M == 0 or ((M - 1) * sxc.stride(0) + K // 128) * 4 < (1 << 31)
            if K <= 65536 and scales_ok and x2c.data_ptr() % 16 == 0 and wc.data_ptr() % 16 == 0:
                # e5m2 on the MFMA kernels (operand format bf8): tile kernels, split along K where e4m3fn is, or the
                # weight-streaming / strip kernels for up to 64 rows
                fused = bias is not None and bias.dtype == torch.bfloat16
                y = torch.empty(M, N, device=dev, dtype=torch.bfloat16)
                with on_device(dev):
                    ws = gemm_workspace(dev, M, N, K)
                    check(lib().mdy_fp8_gemm_nt_ex(ptr(x2c), ptr(sxc), sxc.stride(0), 1, ptr(wc), ptr(swc), ptr(y),
                                                   ptr(bias.contiguous()) if fused else None, 0, M, N, K, fmt, 0, ptr(ws),
                                                   ws.numel() if ws is not None else 0, stream_ptr(dev)), "fp8_matmul")
            else:
                # K beyond 65536, unaligned operands or scales spanning 2^31 bytes: the GEMM with row scales on both
                # operands, the weight's block scales expanded to one per row
                fused = False
                sw_rows = scale_w.repeat_interleave(128, dim=0)[:N].contiguous()
                y = _matmul_rowscaled(x2, sx2, w, sw_rows, M, N, K, dev, fmt)
        if bias is not None and not fused:                               # added in fp32 afterwards
            from .fp8 import add_bias
            add_bias(y, bias.contiguous())
        return y.view(*x.shape[:-1], w.size(0))
    assert x.size(0) % 128 == 0, 'in backward dy.T @ x or dy @ w'
    assert bias is None
    done = host().row_scaled_product(x, w, scale_x, scale_w, fmt)
    if done is not None:
        return done
    dev = require_gpu(x, w, scale_x, scale_w)
    x2 = x.reshape(-1, x.size(-1))
    M, K = x2.shape
    N = w.size(0)
    if w.size(1) != K or tuple(scale_x.shape[-2:]) != (M, (K + 127) // 128) or tuple(scale_w.shape) != (N, (K + 127) // 128):
        raise ValueError("shape mismatch: x %s scale_x %s w %s scale_w %s" % (tuple(x.shape), tuple(scale_x.shape), tuple(w.shape),
                                                                                tuple(scale_w.shape)))
    return _matmul_rowscaled(x2, scale_x.reshape(M, -1), w, scale_w, M, N, K, dev, fmt)


def _matmul_rowscaled(x2, sx, w, sw, M, N, K, dev, fmt=0):
    """[M, K] . [N, K]^T with per-row scales on both sides; operands may be column slices of K-padded buffers."""
    PK = (K + 127) // 128 * 128

    def k_padded(t):      # a [rows, K] view whose storage already runs to a multiple of 128 columns, zero filled
        if K == PK and t.stride(1) == 1 and t.stride(0) == K and t.data_ptr() % 16 == 0:
            return t
        full = torch.zeros(t.size(0), PK, device=dev, dtype=torch.uint8)
        full[:, :K] = t.view(torch.uint8)
        return full
    a, b = k_padded(x2), k_padded(w)
    out = torch.empty(M, N, device=dev, dtype=torch.bfloat16)
    if M * N == 0:
        return out
    _rowscaled_into(out, a, sx, b, sw, M, N, PK, fmt, dev, "fp8_matmul")
    return out


def _rowscaled_into(out, a, sa, b, sb, M, N, K, fmt, dev, who):
    with on_device(dev):
        ws = rowscaled_workspace(dev, M, N, K)      # scratch for outputs that are cut along K, else None
        check(lib().mdy_fp8_gemm_nt_rowscaled_ws(ptr(a), ptr(sa), sa.stride(0), sa.stride(1), ptr(b), ptr(sb), sb.stride(0), sb.stride(1),
                                                 ptr(out), M, N, K, fmt, 0, ptr(ws), ws.numel() if ws is not None else 0,
                                                 stream_ptr(dev)), who)


def fp8_matmul_bwd(xt, w, dy, dyt, scale_xt, scale_w, scale_dy, scale_dyt):
    """Input and weight gradient of y = x . w^T from the quantized copies (fp8_kernel.py:254-257)."""
    dx = fp8_matmul(dy, w, scale_dy, scale_w, have_w=True)
    dw = fp8_matmul(dyt, xt, scale_dyt, scale_xt, have_w=False)
    return dx, dw


def _saved_copy(copy, fp8_dtype, cols, scale_shape, dev, who):
    """(bytes [rows, cols], scales) as the kernels read them, from what autograd's saved tensors gave back: a hook of the user's
    may have moved them, changed their strides or returned something else."""
    y, s = copy
    require_gpu(y, s)
    if y.device != dev or s.device != dev:
        raise RuntimeError("%s: a saved copy came back on %s and %s, the gradient is on %s" % (who, y.device, s.device, dev))
    if y.dtype != fp8_dtype or s.dtype != torch.float32:
        raise TypeError("%s: a saved %s copy with float32 scales came back as %s and %s" % (who, fp8_dtype, y.dtype, s.dtype))
    if y.dim() != 2 or y.size(1) != cols or tuple(s.shape) != scale_shape(y.size(0)):
        raise ValueError("%s: a saved copy of %d columns came back as %s with scales %s" % (who, cols, tuple(y.shape), tuple(s.shape)))
    y = y.contiguous()
    return (y if y.data_ptr() % 16 == 0 else y.clone()), s.contiguous()


def _official_linear_backward(dy2, w_t, x_t, need_dx, need_dw, fp8_dtype=FP8, need_dbias=False, w=None):
    """Gradients of y = x . w^T in the official dialect (fp8_kernel.py:274-301): dx = dy . w on the row-wise copy of dy
    and the block-quantized w^T, dw = dy^T . x on the transposed copies of dy and x (row scales on both operands).
    w_t = (bytes, scales) of w^T, or (None, None) for them to be taken from w; x_t = (bytes, scales) of the transposed x; either
    may be None when its gradient is not needed.  One kernel pass over dy gives both of its copies and, for the bias gradient, its
    column sums; the transposed copies keep their zero padding to a multiple of 128 tokens."""
    _, fmt = _fp8_mode(fp8_dtype, "Fp8Linear.backward")
    done = host().official_backward(dy2, *x_t, *w_t, fmt, need_dx, need_dw, need_dbias, w)
    if done is not None:
        return done
    dy2 = dy2.reshape(-1, dy2.size(-1))
    if dy2.dtype != torch.bfloat16:
        dy2 = dy2.to(torch.bfloat16)
    M, N = dy2.shape
    dev = dy2.device
    dx = dw = None
    if not need_dx and not need_dw:
        return None, None, dy2.sum(0) if need_dbias else None
    dbias = torch.empty(N, device=dev, dtype=torch.bfloat16) if need_dbias and dy2.numel() > 0 else None
    qdy, sdy, qdyt, sdyt = _act_quant_transposed(dy2, need_dx, "Fp8Linear.backward", fp8_dtype, dbias)
    if need_dx:
        if w_t[0] is None:
            w_t = _weight_quant_both(w, False, True, fp8_dtype, "Fp8Linear.backward")[2:]
        qwt, swt = _saved_copy(w_t, fp8_dtype, N, lambda rows: ((rows + 127) // 128, N // 128), dev, "Fp8Linear.backward")
        dx = fp8_matmul(qdy[:M], qwt, sdy[:M], swt, have_w=True)
    if need_dw:
        PM = qdyt.size(1)
        qxt, sxt = _saved_copy(x_t, fp8_dtype, PM, lambda rows: (rows, PM // 128), dev, "Fp8Linear.backward")
        K = qxt.size(0)
        dw = torch.empty(N, K, device=dev, dtype=torch.bfloat16)
        if qdyt.size(1) == 0:
            dw.zero_()                                   # no tokens: an empty sum
        elif N * K > 0:
            _rowscaled_into(dw, qdyt, sdyt, qxt, sxt, N, K, qdyt.size(1), fmt, dev, "Fp8Linear.backward")
    if need_dbias and dbias is None:
        dbias = dy2.sum(0)
    return dx, dw, dbias


def _versions(*tensors):
    """What save_for_backward keeps of tensors that only their version is needed of; an inference tensor itself, which it refuses."""
    return [t if t.is_inference() else host().version_guard(t) for t in tensors]


class _Fp8LinearFunction(torch.autograd.Function):
    """fp8_kernel.py:259-301.  Forward: act_quant_block(x), weight_quant_block(w), GEMM with the bias in its epilogue.
    Backward: x and dy quantized along the tokens (transposed copies, one kernel pass over dy for both of its copies),
    w^T block-quantized; dx = dy . w through the tile kernels, dw = dy^T . x through the GEMM with row scales on both
    operands.  The transposed copies keep their zero padding to a multiple of 128 tokens, so any token count works.
    What the backward pass will need of x is quantized by the forward's own pass over it (x is read once per step instead of
    twice) and kept in place of x: one byte per element of x, also where x stays alive for another reason.  The same is done with
    w, one byte per element of it, as long as both copies take no more memory than x itself (N <= M for a bf16 x): every forward pass
    whose backward pass is still to come holds its own.  Beyond that w is kept, which costs nothing, and quantized again
    by the backward pass.  The version counters of x and w are kept too, so that a backward pass after an in-place change of either is
    refused as for any saved tensor.  (A change through `.data` bumps none: a backward pass behind it takes w as the forward pass
    saw it where the copy was kept, and as it is then where w was.)"""

    @staticmethod
    def forward(ctx, x, w, bias, fp8_dtype, grad_enabled=True):
        _, fmt = _fp8_mode(fp8_dtype, "Fp8Linear")
        input_shape = x.shape
        need_dx, need_dw = [bool(grad_enabled and n) for n in ctx.needs_input_grad[:2]]
        ctx.has_bias = bias is not None
        ctx.fp8_dtype = fp8_dtype
        ctx.input_shape = input_shape
        # both copies within x's memory (their scales, one 64th on top, apart).  Quantizing w again costs a pass over it: 256x8192x8192 170 -> 195 us
        # a step, 1024x4096x4096 116 -> 121, 2048x7168x2048 148 -> 153 (351, 200 and 247 with x quantized again as well)
        keep_wt = need_dx and w.numel() + (x.numel() if need_dw else 0) <= x.numel() * x.element_size()
        done = host().official_forward(x, w, bias, fmt, need_dw, keep_wt, need_dx or need_dw)
        if done is not None:
            ctx.save_for_backward(*(done[1:] if keep_wt or not need_dx else done[1:6] + (w,)))
            return done[0]
        x2 = x.reshape(-1, input_shape[-1])
        if need_dw:
            assert x2.size(-1) % 128 == 0
            qx, sx, qxt, sxt = _act_quant_transposed(x2, True, "Fp8Linear", fp8_dtype)
            qx, sx = qx[:x2.size(0)], sx[:x2.size(0)]
        else:
            qx, sx = act_quant_block(x2, dtype=fp8_dtype)
            qxt = sxt = None
        qw, sw, qwt, swt = _weight_quant_both(w, True, keep_wt, fp8_dtype, "Fp8Linear")
        y = fp8_matmul(qx, qw, sx, sw, bias, have_w=True)
        versions = _versions(x2, w) if need_dx or need_dw else (None, None)
        ctx.save_for_backward(qxt, sxt, qwt, swt, versions[0], versions[1] if keep_wt or not need_dx else w)
        return y.view(*input_shape[:-1], w.size(0))

    @staticmethod
    def backward(ctx, dy):
        qxt, sxt, qwt, swt, _, w = ctx.saved_tensors
        need = ctx.needs_input_grad
        dx, dw, dbias = _official_linear_backward(dy, (qwt, swt), (qxt, sxt), need[0], need[1], ctx.fp8_dtype, ctx.has_bias and need[2],
                                                  w)
        if dx is not None and len(ctx.input_shape) != 2:
            dx = dx.view(ctx.input_shape)
        return dx, dw, dbias, None, None


def fp8_linear_with_quant_ops(x, w, bias, fp8_dtype):
    return _Fp8LinearFunction.apply(x, w, bias, fp8_dtype, torch.is_grad_enabled())


class Fp8Linear(torch.nn.Linear):
    """nn.Linear on the official-dialect FP8 path (fp8_kernel.py:303-313); fp8_dtype float8_e5m2 (the reference's
    default) or float8_e4m3fn (what its notebook passes, and the faster one here)."""

    def __init__(self, in_features, out_features, bias=True, device=None, dtype=None, fp8_dtype=E5M2):
        super().__init__(in_features, out_features, bias, device, dtype)
        _fp8_mode(fp8_dtype, "Fp8Linear")
        self.fp8_dtype = fp8_dtype

    def forward(self, x):
        return fp8_linear_with_quant_ops(x, self.weight, self.bias, self.fp8_dtype)


def _deep_mlp(x, w_up_gate, w_down, order, up_gate_cache=None, down_cache=None):
    """The MLP's forward pass on DeepLinear quantizers: up/gate projection, fused SwiGLU quantizer (the activation itself is
    never written), down projection."""
    from . import fp8 as L
    shape = x.shape
    N2, out_f = w_up_gate.size(0), w_down.size(0)
    q_wu, s_wu = (up_gate_cache or L.quant_weight(w_up_gate, only_forward=True))[:2]
    q_wd, s_wd = (down_cache or L.quant_weight(w_down, only_forward=True))[:2]
    y = host().mlp(x, q_wu, s_wu, N2, q_wd, s_wd, out_f, int(order == "gate-up"), 1) if order in _ORDERS else None
    if y is not None:
        return y
    up_gate = host().deep_linear(x, q_wu, s_wu, N2, None, 0)
    if up_gate is None:
        x2 = x.reshape(-1, shape[-1])
        q_x, s_x, _, _ = L.quant_input(x2, only_forward=True)
        up_gate = L.fp8_matmul(q_x[:x2.size(0)], s_x[:x2.size(0)], q_wu[:N2], s_wu[:L._cdiv(N2, 128)])
    M = up_gate.numel() // N2
    q_act, s_act = silu_act_quant(up_gate, order, dialect="deeplinear")
    y = host().matmul(q_act, s_act, q_wd, s_wd, None, 0, M, out_f)
    if y is None:
        y = L.fp8_matmul(q_act[:M], s_act[:M], q_wd[:out_f], s_wd[:L._cdiv(out_f, 128)])
    return y if len(shape) == 2 else y.view(*shape[:-1], out_f)


class _Fp8MlpCkptOps(torch.autograd.Function):
    """Memory-saving MLP step (fp8_kernel.py:436-494): the forward keeps only x and the two weights; the
    backward recomputes the up/gate projection and the activation, then runs the two weight-gradient and
    the two input-gradient GEMMs on the quantizers' transposed copies."""

    @staticmethod
    def forward(ctx, x, w_up_gate, w_down, fp8_dtype=FP8, order="up-gate", up_gate_cache=None, down_cache=None):
        _require_e4m3(fp8_dtype, "fp8_ckpt_mlp")
        y = _deep_mlp(x, w_up_gate, w_down, order, up_gate_cache, down_cache)
        x2 = x.reshape(-1, x.size(-1))
        ctx.save_for_backward(x2, w_up_gate, w_down)
        ctx.order, ctx.shape, ctx.dims = order, x.shape, (x2.size(0), x2.size(1), w_up_gate.size(0), w_down.size(1))
        return y

    @staticmethod
    def backward(ctx, dy):
        from . import fp8 as L
        x2, w_up_gate, w_down = ctx.saved_tensors
        M, H, N2, inter = ctx.dims
        out_f = w_down.size(0)
        dy2 = dy.reshape(-1, out_f)
        if dy2.dtype != torch.bfloat16:
            dy2 = dy2.to(torch.bfloat16)
        done = host().mlp_backward(dy2, x2, w_up_gate, w_down, int(ctx.order == "gate-up"), 0, 1) if ctx.order in _ORDERS else None
        if done is not None:
            return (done[0].view(ctx.shape),) + done[1:] + (None, None, None, None)
        cd = L._cdiv
        # recompute up_gate and act; the transposed copies feed the weight gradients
        q_x, s_x, q_xt, s_xt = L.quant_input(x2, only_forward=False)
        q_wu, s_wu, q_wut, s_wut = L.quant_weight(w_up_gate, only_forward=False)
        up_gate = L.fp8_matmul(q_x[:M], s_x[:M], q_wu[:N2], s_wu[:cd(N2, 128)])
        act = silu_fwd(up_gate, ctx.order)
        _, _, q_actt, s_actt = L.quant_input(act, only_forward=False)
        _, _, q_wdt, s_wdt = L.quant_weight(w_down, only_forward=False)
        q_dy, s_dy, q_dyt, s_dyt = L.quant_grad_output(dy2)
        dact = L.fp8_matmul(q_dy[:M], s_dy[:M], q_wdt[:inter], s_wdt[:cd(inter, 128)])
        dw_down = L.fp8_matmul(q_dyt[:out_f], s_dyt[:out_f], q_actt[:inter], s_actt[:cd(inter, 128)])
        dup_gate = silu_bwd(dact, up_gate, ctx.order)
        q_du, s_du, q_dut, s_dut = L.quant_grad_output(dup_gate)
        dx = L.fp8_matmul(q_du[:M], s_du[:M], q_wut[:H], s_wut[:cd(H, 128)]).view(ctx.shape)
        dw_up_gate = L.fp8_matmul(q_dut[:N2], s_dut[:N2], q_xt[:H], s_xt[:cd(H, 128)])
        return dx, dw_up_gate, dw_down, None, None, None, None


def _official_mlp(x2, w_up_gate, w_down, fp8_dtype, order):
    """The MLP's forward pass in the official dialect; in e4m3fn the activation is quantized by the fused SwiGLU kernel (the
    bytes of silu_fwd + act_quant_block)."""
    mode, _ = _fp8_mode(fp8_dtype, "fp8_ckpt_mlp")
    qwu, swu = weight_quant_block(w_up_gate, dtype=fp8_dtype)
    qwd, swd = weight_quant_block(w_down, dtype=fp8_dtype)
    if mode == 0 and order in _ORDERS:
        y = host().mlp(x2, qwu, swu, qwu.size(0), qwd, swd, qwd.size(0), int(order == "gate-up"), 0)
        if y is not None:
            return y
    qx, sx = act_quant_block(x2, dtype=fp8_dtype)
    up_gate = fp8_matmul(qx, qwu, sx, swu)
    if mode == 0:
        qact, sact = silu_act_quant(up_gate, order, dialect="official")       # one pass, e4m3fn
    else:
        qact, sact = act_quant_block(silu_fwd(up_gate, order), dtype=fp8_dtype)
    return fp8_matmul(qact, qwd, sact, swd)


class _Fp8MlpCkptOfficial(torch.autograd.Function):
    """The same memory-saving step in the official dialect, as the reference runs it (fp8_kernel.py:436-494):
    act_quant_block / weight_quant_block / fp8_matmul, the activation quantized by the fused SwiGLU kernel in the
    forward (same bytes as silu_fwd + act_quant_block), x the only activation kept."""

    @staticmethod
    def forward(ctx, x, w_up_gate, w_down, fp8_dtype=E5M2, order="up-gate"):
        shape = x.shape
        x2 = x.reshape(-1, shape[-1])
        y = _official_mlp(x2, w_up_gate, w_down, fp8_dtype, order)
        ctx.save_for_backward(x2, w_up_gate, w_down)
        ctx.order, ctx.shape, ctx.fp8_dtype = order, shape, fp8_dtype
        return y.view(*shape[:-1], w_down.size(0))

    @staticmethod
    def backward(ctx, dy):
        x2, w_up_gate, w_down = ctx.saved_tensors
        dy2 = dy.reshape(-1, dy.size(-1))
        if dy2.dtype != torch.bfloat16:
            dy2 = dy2.to(torch.bfloat16)
        done = host().mlp_backward(dy2, x2, w_up_gate, w_down, int(ctx.order == "gate-up"), _fp8_mode(ctx.fp8_dtype, "fp8_ckpt_mlp")[1], 0) if ctx.order in _ORDERS else None
        if done is not None:
            return (done[0].view(ctx.shape),) + done[1:] + (None, None)
        M = x2.size(0)
        # one pass over x and over each weight for the copies of the recomputation and of the gradients
        qx, sx, qxt, sxt = _act_quant_transposed(x2, True, "fp8_ckpt_mlp", ctx.fp8_dtype)
        qwu, swu, qwut, swut = _weight_quant_both(w_up_gate, True, True, ctx.fp8_dtype, "fp8_ckpt_mlp")
        up_gate = fp8_matmul(qx[:M], qwu, sx[:M], swu)
        del qx, sx, qwu, swu
        act = silu_fwd(up_gate, ctx.order)
        _, _, qwdt, swdt = _weight_quant_both(w_down, False, True, ctx.fp8_dtype, "fp8_ckpt_mlp")
        _, _, qactt, sactt = _act_quant_transposed(act, False, "fp8_ckpt_mlp", ctx.fp8_dtype)
        dact, dw_down, _ = _official_linear_backward(dy2, (qwdt, swdt), (qactt, sactt), True, True, ctx.fp8_dtype)
        dup_gate = silu_bwd(dact, up_gate, ctx.order)
        dx, dw_up_gate, _ = _official_linear_backward(dup_gate, (qwut, swut), (qxt, sxt), True, True, ctx.fp8_dtype)
        return dx.view(ctx.shape), dw_up_gate, dw_down, None, None


def fp8_ckpt_mlp(x, w_up_gate, w_down, fp8_dtype=E5M2, order="up-gate", dialect="official"):
    """Memory-saving FP8 MLP step with the reference's positional order and default dtype (fp8_kernel.py:436-494:
    `fp8_ckpt_mlp(h, w1, w2, self.fp8_dtype, self.order)`).  dialect "official" (the reference's: s = amax /
    finfo(fp8_dtype).max, float8_e5m2 or float8_e4m3fn) or "deeplinear" (clamp 1e4 + eps 1e-8, the quantizers of
    dpsk_fp8linear/fp8.py; float8_e4m3fn only)."""
    if dialect == "official":
        return _Fp8MlpCkptOfficial.apply(x, w_up_gate, w_down, fp8_dtype, order)
    if dialect != "deeplinear":
        raise ValueError("dialect must be 'official' or 'deeplinear'")
    return _Fp8MlpCkptOps.apply(x, w_up_gate, w_down, fp8_dtype, order)


class Fp8MLP(torch.nn.Module):
    """SwiGLU MLP on the FP8 linear path (fp8_kernel.py:500-515): up/gate projection, silu(gate) * up, down
    projection, both projections block-wise FP8 (1x128 activation and 128x128 weight scales), no biases.  fp8_dtype
    float8_e5m2 (the reference's default) or float8_e4m3fn.

    dialect "official" (default, what the reference's Fp8MLP computes: its projections are `Fp8Linear`s,
    s = amax / finfo.max) or "deeplinear" (`DeepLinear` projections: clamp 1e4 + eps 1e-8, optional weight cache;
    e4m3fn only).
    Without gradients the activation goes from the up/gate GEMM to the down GEMM through the fused
    SwiGLU + quantizer (one pass, the bf16 activation is never written).  With gradients the default is the
    composition linear -> triton_silu -> linear; `low_memory` (attribute or call argument, as in the
    reference) keeps only the input for the backward pass and recomputes up/gate and the activation there.
    """

    def __init__(self, hidden_size, intermediate_size, order="up-gate", fp8_dtype=E5M2, low_memory=False,
                 device=None, dtype=torch.bfloat16, dialect="official"):
        super().__init__()
        if dialect == "deeplinear":
            _require_e4m3(fp8_dtype, "Fp8MLP(dialect='deeplinear')")
        else:
            _fp8_mode(fp8_dtype, "Fp8MLP")
        assert order in _ORDERS, "please indicate the order of input, up-gate or gate-up"
        if dialect not in ("official", "deeplinear"):
            raise ValueError("dialect must be 'official' or 'deeplinear'")
        if dialect == "official":
            self.up_gate_proj = Fp8Linear(hidden_size, intermediate_size * 2, bias=False, device=device, dtype=dtype,
                                          fp8_dtype=fp8_dtype)
            self.down_proj = Fp8Linear(intermediate_size, hidden_size, bias=False, device=device, dtype=dtype,
                                       fp8_dtype=fp8_dtype)
        else:
            from .fp8 import DeepLinear
            self.up_gate_proj = DeepLinear(hidden_size, intermediate_size * 2, bias=False, device=device, dtype=dtype)
            self.down_proj = DeepLinear(intermediate_size, hidden_size, bias=False, device=device, dtype=dtype)
        self.dialect = dialect
        self.order = order
        self.fp8_dtype = fp8_dtype
        self.low_memory = low_memory

    def forward(self, hidden_states, low_memory=False):
        up, down = self.up_gate_proj, self.down_proj
        w_up, w_down = parameter_of(up, "weight"), parameter_of(down, "weight")
        needs_grad = torch.is_grad_enabled() and (hidden_states.requires_grad or w_up.requires_grad or w_down.requires_grad)
        if not needs_grad and host().ordinary(hidden_states, w_up, w_down):
            # nothing to differentiate and nothing that traces or transforms the call: no autograd function around it
            if self.dialect == "official":
                y = _official_mlp(hidden_states.reshape(-1, hidden_states.size(-1)), w_up, w_down, self.fp8_dtype, self.order)
                return y.view(*hidden_states.shape[:-1], w_down.size(0))
            return _deep_mlp(hidden_states, w_up, w_down, self.order,
                             up._quantized_weight(False, w_up) if up.cache_weight else None,
                             down._quantized_weight(False, w_down) if down.cache_weight else None)
        if not needs_grad or low_memory or self.low_memory:
            if self.dialect == "official":
                return _Fp8MlpCkptOfficial.apply(hidden_states, w_up, w_down, self.fp8_dtype, self.order)
            # cached quantized weights (when the projections cache); the forward needs no transposed copies
            return _Fp8MlpCkptOps.apply(hidden_states, w_up, w_down, self.fp8_dtype, self.order,
                                        up._quantized_weight(False, w_up) if up.cache_weight else None,
                                        down._quantized_weight(False, w_down) if down.cache_weight else None)
        return down(triton_silu(up(hidden_states), self.order))
