"""Autograd for the hot path: the training step's backward through the HIP
kernels (the reference trains through ATen autograd of the same ops,
core/runtime/run_model.py:362-617 over models/attention.py:231-283 and
models/transformer.py:142-300).

- Partition and reverse are adjoint token permutations: every emitted,
  non-pad window token is gathered from exactly one grid token, and reverse
  scatters it back to that token.  So the gradient of partition is reverse
  (grid tokens no window reads get zero) and the gradient of reverse is
  partition (pad window tokens get zero), both on the same geometry.
- The attention core's backward is ``terra_swin_attn_bwd`` (P recomputed
  from q and k; dq, dk, dv, and the bias-table gradient summed over
  windows): an MFMA tile kernel for every bf16 window (8x8, 7x7, padded
  keys), a plain fp32 kernel for fp32 activations.  For a shape neither serves the forward still runs
  and backward() raises NotImplementedError (there is no non-HIP backward).

Each function runs the plain kernel when no input needs a gradient.
"""
from __future__ import annotations

from typing import Optional, Tuple, Union

import torch

from . import kernels
from .kernels import ShiftMask, WindowGeometry, WindowMask

MaskArg = Union[None, torch.Tensor, ShiftMask, WindowMask]


def _needs_grad(*tensors: Optional[torch.Tensor]) -> bool:
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors)


class _Partition(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x: torch.Tensor, geom: WindowGeometry) -> torch.Tensor:
        ctx.geom = geom
        return kernels.swin_partition(x, geom)

    @staticmethod
    def backward(ctx, grad: torch.Tensor):
        return kernels.swin_reverse(grad.contiguous(), ctx.geom), None


class ResidualLink:
    """Hands a half-block's output gradient (the residual's gradient) from the
    scatter's backward to the gather's backward, which adds it into dx in the
    same kernel instead of autograd summing the two paths in a separate pass.
    The scatter then takes its residual detached; the gather's backward runs
    after the scatter's, since the gather's output feeds the scatter."""

    def __init__(self):
        self.grad: Optional[torch.Tensor] = None


class ColumnSumLink:
    """Hands the column sums of a Linear's output gradient (its bias gradient)
    from the backward that produces that gradient, which sums it in the same
    kernel, to the Linear's backward, which then skips its own reduction."""

    def __init__(self):
        self.sums: Optional[torch.Tensor] = None


class _Reverse(torch.autograd.Function):
    """Window reverse + roll + residual.  With bf16 windows and an fp32
    output (autocast's bf16 proj output added to an fp32 shortcut) the kernel
    widens the windows itself, and the backward writes the windows' gradient
    in bf16 (what the cast's backward gives), with the column sums a
    :class:`ColumnSumLink` hands to the producing Linear's bias gradient."""

    @staticmethod
    def forward(ctx, windows: torch.Tensor, geom: WindowGeometry, residual: Optional[torch.Tensor],
                link: Optional[ResidualLink], out_dtype: Optional[torch.dtype],
                bias_sums: Optional[ColumnSumLink]) -> torch.Tensor:
        ctx.geom = geom
        ctx.has_residual = residual is not None
        ctx.link, ctx.bias_sums = link, bias_sums
        ctx.win_dtype = windows.dtype
        return kernels.swin_reverse(windows, geom, residual=residual, out_dtype=out_dtype)

    @staticmethod
    def backward(ctx, grad: torch.Tensor):
        grad = grad.contiguous()
        shape = (ctx.geom.batch, ctx.geom.height, ctx.geom.width, ctx.geom.channels)
        if ctx.win_dtype != grad.dtype:  # bf16 windows, fp32 output
            sums = None
            if ctx.bias_sums is not None:
                sums = torch.zeros(ctx.geom.channels, dtype=torch.float32, device=grad.device)
                ctx.bias_sums.sums = sums
            d_windows = kernels.swin_partition(grad.view(shape), ctx.geom, out_dtype=ctx.win_dtype, column_sums=sums)
        else:
            d_windows = kernels.swin_partition(grad.view(shape), ctx.geom)
        if ctx.link is not None:
            ctx.link.grad = grad.view(shape)
            return d_windows, None, None, None, None, None
        return d_windows, None, (grad if ctx.has_residual else None), None, None, None


class _PartitionLN(torch.autograd.Function):
    """LayerNorm over C + pad + roll + partition (terra_swin_partition_ln),
    backward by terra_swin_partition_ln_bwd: dx, and the weight / bias
    gradients summed over the tokens.  With out_dtype bf16 for fp32 x the
    windows are the fp32 output rounded once to bf16 and their gradient
    arrives in bf16 (the _mixed entry points)."""

    @staticmethod
    def forward(ctx, x, weight, bias, geom, eps, out_dtype, link):
        ctx.geom, ctx.eps, ctx.link = geom, eps, link
        ctx.save_for_backward(x, weight, bias)
        return kernels.swin_partition_ln(x, geom, weight, bias, eps, out_dtype=out_dtype)

    @staticmethod
    def backward(ctx, grad: torch.Tensor):
        x, weight, bias = ctx.saved_tensors
        dw = db = None
        if weight is not None and ctx.needs_input_grad[1]:
            dw = torch.zeros(weight.shape, dtype=torch.float32, device=x.device)
        if bias is not None and ctx.needs_input_grad[2]:
            db = torch.zeros(bias.shape, dtype=torch.float32, device=x.device)
        dres = None
        if ctx.link is not None and ctx.link.grad is not None:  # the residual's gradient, added in the kernel
            dres, ctx.link.grad = ctx.link.grad.to(x.dtype).contiguous(), None
        dx = kernels.swin_partition_ln_backward(grad.contiguous(), x, ctx.geom, weight, ctx.eps, dresidual=dres,
                                                dweight=dw, dbias=db)
        return (dx, None if dw is None else dw.to(weight.dtype), None if db is None else db.to(bias.dtype), None, None,
                None, None)


def linear_input_dtype(x: torch.Tensor) -> torch.dtype:
    """The dtype F.linear computes in for an input like x: bf16 inside a bf16
    autocast region (which casts its fp32 input to bf16), else x's own."""
    return torch.bfloat16 if kernels.autocast_bf16(x) and x.dtype == torch.float32 else x.dtype


def partition_ln(x: torch.Tensor, geom: WindowGeometry, weight: Optional[torch.Tensor],
                 bias: Optional[torch.Tensor], eps: float, out_dtype: Optional[torch.dtype] = None,
                 link: Optional[ResidualLink] = None) -> torch.Tensor:
    """:func:`kernels.swin_partition_ln` with gradients for x and the
    LayerNorm affine parameters.  ``out_dtype`` bf16 for fp32 x writes the
    bf16 copy a following Linear under bf16 autocast would cast to (and takes
    its bf16 gradient), instead of fp32 windows and a cast each way.
    ``link``: the :class:`ResidualLink` of a :func:`reverse` whose residual
    is x; its gradient is then added into dx by this backward's kernel."""
    if _needs_grad(x, weight, bias):
        return _PartitionLN.apply(x, weight, bias, geom, eps, out_dtype, link)
    return kernels.swin_partition_ln(x, geom, weight, bias, eps, out_dtype=out_dtype)


def weight_grad(dy: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """dy^T x for dy [T, out] and x [T, in] (a Linear's weight gradient, the
    contraction over all T tokens), in fp32.  bf16 rows run on the HIP
    weight-gradient kernel, which cuts the tokens into as many slices as fill
    the compute units with (output tile, slice) pairs, sums each in two levels
    and adds them in a fixed order (us, against the library's batched product
    over token slices and its sum, or for other token counts its plain product
    rounded to bf16: 524288 x 768 x 192 204 / 255, 524288 x 576 x 192 176 / 246,
    156672 x 4096 x 1024 1370 / 1562, 50176 x 512 x 128 25 / 31, 16385 x 1024 x 1024
    49 / 140, 2001 x 768 x 192 18 / 21; equal at 524288 x 192 x 192 and 32768 x
    768 x 768; behind, with nothing else on the GPU's queue to wait for, at 300 to
    1000 rows of wide layers, 1000 x 1024 x 1024 21 / 16, where the host's 24 us
    for the library's call hide it).  Other dtypes (and feature counts that
    are no multiple of 16) take the library: for large T in fp16 k slices
    contracted as one batched GEMM with an fp32 output and then summed, since
    hipBLASLt takes no split-K tiles for a contraction this long."""
    T, o = dy.shape
    i = x.shape[1]
    if dy.dtype == torch.bfloat16:
        dy, x = dy.contiguous(), x.contiguous()
        if kernels.weight_grad_supported(dy, x):
            return kernels.weight_grad(dy, x)
    k = next((k for k in (128, 64, 32, 16, 8) if T % k == 0 and T // k >= 2048), 1)
    if k == 1 or dy.dtype not in (torch.bfloat16, torch.float16):
        return (dy.t() @ x).float()
    # The transposed view is the left operand; the right one is contiguous.
    return torch.bmm(dy.view(k, T // k, o).transpose(1, 2), x.reshape(k, T // k, i).contiguous(),
                     out_dtype=torch.float32).sum(0)


def _bf16_linears(x: torch.Tensor, *params: Optional[torch.Tensor]) -> bool:
    """Whether F.linear of bf16 rows like x with these parameters is a bf16
    product: under bf16 autocast, which casts fp32 and fp16 parameters (fp64
    ones it leaves, and F.linear refuses), or with bf16 parameters and no
    autocast."""
    if torch.is_autocast_enabled(x.device.type):
        cast = (torch.bfloat16, torch.float32, torch.float16)
        return kernels.autocast_bf16(x) and all(p is None or p.dtype in cast for p in params)
    return all(p is None or p.dtype == torch.bfloat16 for p in params)


def _pack(weight: torch.Tensor, transpose: bool = False) -> torch.Tensor:
    """:func:`kernels.pack_weight` of a weight of any dtype, which packs bf16
    and fp32 ones; others are rounded to bf16 first, as autocast rounds them."""
    if weight.dtype not in (torch.bfloat16, torch.float32):
        weight = weight.to(torch.bfloat16)
    return kernels.pack_weight(weight, transpose)


def _bias32(bias: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """A bias as the linear kernels read it: contiguous 16-byte aligned fp32."""
    if bias is None:
        return None
    b = bias.float().contiguous()
    return b.clone() if b.data_ptr() % 16 else b


def _short_kernel(x: torch.Tensor, out_features: int) -> bool:
    """The short-row linear kernels serve and fill the chip with rows like x
    (us, against the library's product: 524288 rows of 192 -> 576 130 / 300,
    192 -> 192 60 / 113; 50176 rows of 128 -> 384 12 / 28; with the weight's
    packing, where 256 tiles just fill it: 16384 rows of 192 -> 192 6.0 / 8.5, 5504
    of 192 -> 576 8.2 / 11.8, 4096 of 192 -> 768 with the GELU 9.4 / 16.6)."""
    return (kernels.linear_short_supported(x, x.shape[-1], out_features)
            and kernels.linear_short_fills(x.numel() // x.shape[-1], out_features))


def _linear_kernel(x: torch.Tensor, out_features: int) -> bool:
    """The token-row linear kernels serve and fill the chip with rows like x."""
    return (x.is_contiguous() and x.data_ptr() % 16 == 0 and kernels.linear_supported(x, x.shape[-1], out_features)
            and kernels.linear_fills(x.numel() // x.shape[-1], out_features))


def _input_grad(dy: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """dy @ weight for dy [T, out] in the GEMMs' dtype and a Linear's weight
    [out, in] of any dtype: on the linear kernels where they serve the shape
    and are as fast as the library (156672 rows, 4096 -> 1024: 980-1060 us against 1130-1240 for the
    library's product with an untransposed weight)."""
    if dy.dtype != torch.bfloat16:
        return dy @ weight.to(dy.dtype)
    if _short_kernel(dy, weight.shape[1]):
        return kernels.linear_short(dy, _pack(weight, transpose=True), weight.shape[1])
    if _linear_kernel(dy, weight.shape[1]) and kernels.linear_product_pays(dy.shape[0], weight.shape[1]):
        return kernels.linear(dy, _pack(weight, transpose=True), weight.shape[1])
    return dy @ weight.to(dy.dtype)


def _linear_forward(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]):
    """F.linear in the dtype bf16 autocast gives it; returns the result and x
    and weight in that dtype (for the backward)."""
    dt = torch.bfloat16 if (torch.is_autocast_enabled(x.device.type)
                            and torch.get_autocast_dtype(x.device.type) == torch.bfloat16) else x.dtype
    xc, wc = x.to(dt), weight.to(dt)
    o = weight.shape[0]
    if (dt == torch.bfloat16 and weight.dim() == 2 and weight.shape[1] == x.shape[-1]
            and (bias is None or bias.numel() == o) and _bf16_linears(xc, weight, bias) and _short_kernel(xc, o)):
        return kernels.linear_short(xc, kernels.pack_weight(wc), o, _bias32(bias)), xc, wc
    return torch.nn.functional.linear(xc, wc, None if bias is None else bias.to(dt)), xc, wc


class _Linear(torch.autograd.Function):
    """F.linear for training, in the dtype bf16 autocast gives it (x, weight
    and bias cast to bf16 inside an autocast region, as F.linear's autocast
    rule does; on the HIP linear kernels the bias stays fp32), with the weight
    gradient from :func:`weight_grad`.  The bias gradient comes from a
    :class:`ColumnSumLink` when the output gradient's producer summed it (in
    the order of its own kernel), else from a sum."""

    @staticmethod
    def forward(ctx, x, weight, bias, bias_sums):
        y, xc, wc = _linear_forward(x, weight, bias)
        ctx.save_for_backward(xc, wc)
        ctx.dtypes = (x.dtype, weight.dtype, None if bias is None else bias.dtype)
        ctx.bias_sums = bias_sums
        return y

    @staticmethod
    def backward(ctx, dy: torch.Tensor):
        xc, wc = ctx.saved_tensors
        xd, wd, bd = ctx.dtypes
        dt = xc.dtype  # the product's dtype
        dy2 = dy.reshape(-1, dy.shape[-1]).to(dt)
        dx = dw = db = None
        if ctx.needs_input_grad[0]:
            dx = _input_grad(dy2, wc).view(xc.shape).to(xd)
        if ctx.needs_input_grad[1]:
            dw = weight_grad(dy2, xc.reshape(-1, xc.shape[-1])).to(wd)
        sums = None
        if ctx.bias_sums is not None:
            sums, ctx.bias_sums.sums = ctx.bias_sums.sums, None
        if bd is not None and ctx.needs_input_grad[2]:
            db = (sums if sums is not None and dy.dtype == dt else dy2.sum(0, dtype=torch.float32)).to(bd)
        return dx, dw, db, None


def linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor],
           bias_sums: Optional[ColumnSumLink] = None) -> torch.Tensor:
    """F.linear, through :class:`_Linear` when a gradient is needed.
    ``bias_sums``: a :class:`ColumnSumLink` the backward of the output's
    consumer fills with the output gradient's column sums."""
    if _needs_grad(x, weight, bias):
        return _Linear.apply(x, weight, bias, bias_sums)
    return torch.nn.functional.linear(x, weight, bias)


class _Mlp(torch.autograd.Function):
    """SequentialMlp.forward (models/mlp.py:152-172) for training:
    y = x + fc2(GELU(fc1(LayerNorm(x)))).  The LayerNorm forward and its
    backward (with the residual gradient added in the same kernel) run on
    terra_swin_partition_ln / _bwd over the token rows.  With bf16 GEMMs that
    fill the chip, fc1 and the GELU are one linear kernel that keeps fc1's
    output (156672 rows, C = 1024: 1576 us against 1673 for the library's
    product and torch's GELU; 524288 rows, C = 192: 330 against 631), a bf16
    residual is added in fc2's, and in the backward the product with fc2's
    weight, the GELU derivative and fc1's bias gradient are one
    (1446 against 1972 us; 451 against 778).  Smaller or other shapes run the
    products on hipBLASLt through torch, in the dtypes autocast gave them, and
    the exact (erf) GELU derivative on terra_swin_gelu_bwd with fc1's bias
    gradient summed in the same pass.  Under autocast the output gradient's
    cast to bf16 sums fc2's bias gradient in its pass
    (terra_swin_partition_mixed over the token rows)."""

    @staticmethod
    def forward(ctx, x, ln_w, ln_b, w1, b1, w2, b2, eps):
        C = x.shape[-1]
        rows = x.reshape(-1, C).contiguous()
        geom = kernels.rows_geometry(rows.shape[0], C)
        # Under bf16 autocast fc1 takes a bf16 copy of the fp32 LayerNorm
        # output: the kernel writes that copy directly.
        xn = kernels.swin_partition_ln(rows.view(1, -1, 1, C), geom, ln_w, ln_b, eps,
                                       out_dtype=linear_input_dtype(rows)).view(-1, C)
        y = None
        bf16 = xn.dtype == torch.bfloat16 and _bf16_linears(xn, w1, b1, w2, b2)
        if bf16 and _short_kernel(xn, w1.shape[0]):
            h1, a = kernels.linear_short(xn, _pack(w1), w1.shape[0], _bias32(b1), gelu_keep=True)
        elif bf16 and _linear_kernel(xn, w1.shape[0]) and kernels.linear_gelu_keep_pays(xn.shape[0], C, w1.shape[0]):
            h1, a = kernels.linear_gelu_keep(xn, _pack(w1), w1.shape[0], _bias32(b1))
            if rows.dtype == torch.bfloat16 and w2.shape[0] == C and rows.data_ptr() % 16 == 0 \
                    and _linear_kernel(a, C) and kernels.linear_residual_pays(a.shape[0], a.shape[1], C):
                y = kernels.linear_residual(a, _pack(w2), C, rows, _bias32(b2))
        else:
            h1 = torch.nn.functional.linear(xn, w1, b1)
            a = torch.nn.functional.gelu(h1)
        if y is None:
            h2 = torch.nn.functional.linear(a, w2, b2)
            if h2.dtype == torch.bfloat16 and rows.dtype == torch.float32 and C % 4 == 0 and h2.shape[-1] == C:
                # x + fc2(...) under autocast: the bf16 h2 widened and added to the
                # fp32 rows in one pass (the mixed scatter over an identity frame;
                # bit for bit torch's promoted add).
                y = kernels.swin_reverse(h2.contiguous(), geom, residual=rows.view(1, -1, 1, C),
                                         out_dtype=torch.float32).view(rows.shape)
            else:
                y = rows + h2
        ctx.eps, ctx.geom, ctx.shape = eps, geom, x.shape
        ctx.autocast = torch.is_autocast_enabled(x.device.type)
        ctx.save_for_backward(rows, ln_w, ln_b, xn, h1, a, w1, w2)
        return y.view(x.shape[:-1] + (y.shape[-1],))

    @staticmethod
    def backward(ctx, dy: torch.Tensor):
        rows, ln_w, ln_b, xn, h1, a, w1, w2 = ctx.saved_tensors
        C = rows.shape[-1]
        dy = dy.reshape(-1, dy.shape[-1])
        gemm_dtype = h1.dtype  # the forward GEMMs' dtype (bf16 under autocast)
        T, c_out = dy.shape
        db2 = None
        if dy.dtype == torch.float32 and gemm_dtype == torch.bfloat16 and c_out % 4 == 0 and c_out <= 1024:
            # The cast to the GEMMs' bf16 and fc2's bias gradient (the column
            # sums of the bf16 values) in one pass over the token rows.
            if ctx.needs_input_grad[6]:
                db2 = torch.zeros(c_out, dtype=torch.float32, device=dy.device)
            dh2 = kernels.swin_partition(dy.contiguous().view(1, T, 1, c_out), kernels.rows_geometry(T, c_out),
                                         out_dtype=torch.bfloat16, column_sums=db2).view(T, c_out)
        else:
            dh2 = dy.to(gemm_dtype)
            db2 = dh2.sum(0, dtype=torch.float32) if ctx.needs_input_grad[6] else None
        dw2 = weight_grad(dh2, a.to(gemm_dtype)) if ctx.needs_input_grad[5] else None
        db1 = None
        dh2 = dh2.contiguous()
        if _linear_kernel(dh2, h1.shape[-1]):
            # fc2's input gradient, the GELU derivative and fc1's bias gradient in one kernel.
            if ctx.needs_input_grad[4]:
                db1 = torch.zeros(h1.shape[-1], dtype=torch.float32, device=h1.device)
            dh1 = kernels.linear_gelu_backward(dh2, _pack(w2, transpose=True), h1.shape[-1], h1,
                                               column_sums=db1)
        else:
            da = dh2 @ w2.to(gemm_dtype)
            if kernels.gelu_backward_supported(h1):
                # The GELU derivative and fc1's bias gradient in one pass.
                if ctx.needs_input_grad[4]:
                    db1 = torch.zeros(h1.shape[-1], dtype=torch.float32, device=h1.device)
                dh1 = kernels.gelu_backward(da.contiguous(), h1.contiguous(), column_sums=db1)
            else:
                dh1 = torch.ops.aten.gelu_backward(da, h1)
                db1 = dh1.sum(0, dtype=torch.float32) if ctx.needs_input_grad[4] else None
        dxn = _input_grad(dh1, w1)
        dw1 = weight_grad(dh1, xn.to(gemm_dtype)) if ctx.needs_input_grad[3] else None
        dlw = torch.zeros(C, dtype=torch.float32, device=rows.device) if (
            ln_w is not None and ctx.needs_input_grad[1]) else None
        dlb = torch.zeros(C, dtype=torch.float32, device=rows.device) if (
            ln_b is not None and ctx.needs_input_grad[2]) else None
        # dxn in xn's dtype (bf16 under autocast, read exactly by the kernel).
        dx = kernels.swin_partition_ln_backward(
            dxn.to(xn.dtype).contiguous().view(-1, 1, C), rows.view(1, -1, 1, C), ctx.geom, ln_w, ctx.eps,
            dresidual=dy.to(rows.dtype).contiguous(), dweight=dlw, dbias=dlb)
        cast = lambda g, p: None if g is None else g.to(p.dtype)  # noqa: E731
        return (dx.view(ctx.shape), cast(dlw, ln_w), cast(dlb, ln_b), cast(dw1, w1), cast(db1, w1),
                cast(dw2, w2), cast(db2, w2), None)


def mlp(x: torch.Tensor, ln_w: Optional[torch.Tensor], ln_b: Optional[torch.Tensor], w1: torch.Tensor,
        b1: torch.Tensor, w2: torch.Tensor, b2: torch.Tensor, eps: float) -> torch.Tensor:
    """The MLP half with gradients (see :class:`_Mlp`)."""
    return _Mlp.apply(x, ln_w, ln_b, w1, b1, w2, b2, eps)


def partition(x: torch.Tensor, geom: WindowGeometry) -> torch.Tensor:
    """:func:`kernels.swin_partition` with a gradient (reverse)."""
    if _needs_grad(x):
        return _Partition.apply(x, geom)
    return kernels.swin_partition(x, geom)


def reverse(windows: torch.Tensor, geom: WindowGeometry, residual: Optional[torch.Tensor] = None,
            link: Optional[ResidualLink] = None, out_dtype: Optional[torch.dtype] = None,
            bias_sums: Optional[ColumnSumLink] = None) -> torch.Tensor:
    """:func:`kernels.swin_reverse` with gradients (partition for the windows,
    identity for the residual), in ``out_dtype`` (default: the windows'
    dtype; bf16 windows into fp32 are widened by the kernel, other pairs by a
    cast first).  With ``link`` (the residual is the input of the
    :func:`partition_ln` holding the same link) the residual's gradient goes
    through the link instead of autograd.  ``bias_sums``: the
    :class:`ColumnSumLink` of the :func:`linear` whose output the windows are;
    the bf16 backward fills it."""
    odt = windows.dtype if out_dtype is None else out_dtype
    if odt != windows.dtype and not (windows.dtype == torch.bfloat16 and odt == torch.float32):
        windows = windows.to(odt)
    if link is not None and residual is not None:
        return _Reverse.apply(windows, geom, residual.detach(), link, odt, bias_sums)
    if _needs_grad(windows, residual):
        return _Reverse.apply(windows, geom, residual, None, odt, bias_sums)
    return kernels.swin_reverse(windows, geom, residual=residual, out_dtype=odt)


def _check_backward(q: torch.Tensor, num_heads: int, window_size: Tuple[int, int], n_real: Optional[int]) -> None:
    if not kernels.attention_backward_supported(q, num_heads, window_size, n_real):
        raise NotImplementedError(
            "terra_amd: the attention backward kernels are built for bf16 / fp32 activations, windows up to 8x8 "
            "in at most 64 token rows and head dim 32, 64 or 128, and for bf16 windows of a multiple of 128 tokens "
            f"up to 4096 with head dim 64 or 128 (got {q.dtype}, window {tuple(window_size)}, "
            f"{q.shape[-2]} tokens, n_real {n_real}, head dim {q.shape[-1] // num_heads})")


class _Attention(torch.autograd.Function):
    """q, k, v as separate inputs (any row strides)."""

    @staticmethod
    def forward(ctx, q, k, v, table, num_heads, window_size, scale, mask, n_real, mask_value):
        ctx.cfg = (num_heads, window_size, scale, mask, n_real, mask_value)
        ctx.save_for_backward(q, k, v, table)
        return kernels.window_attention(q, k, v, num_heads, window_size, scale, bias_table=table, mask=mask,
                                        n_real=n_real, mask_value=mask_value)

    @staticmethod
    def backward(ctx, grad: torch.Tensor):
        q, k, v, table = ctx.saved_tensors
        num_heads, window_size, scale, mask, n_real, mask_value = ctx.cfg
        _check_backward(q, num_heads, window_size, n_real)
        dbias = None
        if table is not None and ctx.needs_input_grad[3]:
            dbias = torch.zeros(table.shape, dtype=torch.float32, device=table.device)
        dq, dk, dv = kernels.window_attention_backward(q, k, v, grad.contiguous(), num_heads, window_size, scale,
                                                       bias_table=table, mask=mask, n_real=n_real,
                                                       mask_value=mask_value, dbias=dbias)
        dtable = None if dbias is None else dbias.to(table.dtype)
        return dq, dk, dv, dtable, None, None, None, None, None, None


class _AttentionQKV(torch.autograd.Function):
    """One [B_, N, 3C] projection output as input: the gradients of q, k and v
    are written into one [B_, N, 3C] buffer (the input of the projection's
    backward GEMM), with no slice copies.  With a :class:`ColumnSumLink` the
    bf16 kernel also sums that buffer's columns (the projection's bias
    gradient) while it writes it."""

    @staticmethod
    def forward(ctx, qkv, table, num_heads, window_size, scale, mask, n_real, mask_value, bias_sums):
        C = qkv.shape[-1] // 3
        ctx.cfg = (num_heads, window_size, scale, mask, n_real, mask_value)
        ctx.bias_sums = bias_sums
        ctx.save_for_backward(qkv, table)
        return kernels.window_attention(qkv[..., :C], qkv[..., C:2 * C], qkv[..., 2 * C:], num_heads, window_size,
                                        scale, bias_table=table, mask=mask, n_real=n_real, mask_value=mask_value)

    @staticmethod
    def backward(ctx, grad: torch.Tensor):
        qkv, table = ctx.saved_tensors
        num_heads, window_size, scale, mask, n_real, mask_value = ctx.cfg
        C = qkv.shape[-1] // 3
        _check_backward(qkv[..., :C], num_heads, window_size, n_real)
        dqkv = torch.empty(qkv.shape, dtype=qkv.dtype, device=qkv.device)
        dbias = None
        if table is not None and ctx.needs_input_grad[1]:
            dbias = torch.zeros(table.shape, dtype=torch.float32, device=table.device)
        sums = None
        if ctx.bias_sums is not None and kernels.attention_backward_sums_supported(qkv[..., :C], num_heads,
                                                                                   window_size, n_real):
            sums = torch.zeros(3 * C, dtype=torch.float32, device=qkv.device)
            ctx.bias_sums.sums = sums
        kernels.window_attention_backward(qkv[..., :C], qkv[..., C:2 * C], qkv[..., 2 * C:], grad.contiguous(),
                                          num_heads, window_size, scale, bias_table=table, mask=mask, n_real=n_real,
                                          mask_value=mask_value, dq=dqkv[..., :C], dk=dqkv[..., C:2 * C],
                                          dv=dqkv[..., 2 * C:], dbias=dbias, column_sums=sums)
        dtable = None if dbias is None else dbias.to(table.dtype)
        return dqkv, dtable, None, None, None, None, None, None, None


def window_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, num_heads: int,
                     window_size: Tuple[int, int], scale: float, bias_table: Optional[torch.Tensor] = None,
                     mask: MaskArg = None, n_real: Optional[int] = None,
                     mask_value: float = kernels.MASK_VALUE) -> torch.Tensor:
    """:func:`kernels.window_attention` with gradients for q, k, v and the bias
    table."""
    if _needs_grad(q, k, v, bias_table):
        return _Attention.apply(q, k, v, bias_table, num_heads, tuple(window_size), scale, mask, n_real, mask_value)
    return kernels.window_attention(q, k, v, num_heads, window_size, scale, bias_table=bias_table, mask=mask,
                                    n_real=n_real, mask_value=mask_value)


def window_attention_qkv(qkv: torch.Tensor, num_heads: int, window_size: Tuple[int, int], scale: float,
                         bias_table: Optional[torch.Tensor] = None, mask: MaskArg = None,
                         n_real: Optional[int] = None, mask_value: float = kernels.MASK_VALUE,
                         bias_sums: Optional[ColumnSumLink] = None) -> torch.Tensor:
    """Attention over the column blocks q | k | v of one [B_, N, 3C] tensor,
    with gradients (see :class:`_AttentionQKV`).  ``bias_sums``: the
    :class:`ColumnSumLink` of the :func:`linear` that produced ``qkv``."""
    C = qkv.shape[-1] // 3
    if _needs_grad(qkv, bias_table):
        if not qkv.is_contiguous():
            qkv = qkv.contiguous()
        return _AttentionQKV.apply(qkv, bias_table, num_heads, tuple(window_size), scale, mask, n_real, mask_value,
                                   bias_sums)
    return kernels.window_attention(qkv[..., :C], qkv[..., C:2 * C], qkv[..., 2 * C:], num_heads, window_size,
                                    scale, bias_table=bias_table, mask=mask, n_real=n_real, mask_value=mask_value)


class _AttentionHalf(torch.autograd.Function):
    """SequentialSwinTransformer.forward (models/transformer.py:142-300) for
    training as one function:

        y = x + reverse(proj(attention(qkv(partition(LayerNorm(x))))))

    through the kernels of partition_ln, linear, window_attention_qkv and
    reverse above, in the dtypes bf16 autocast gives each.  One function
    instead of a chain of them: a small block's step is bound by the host
    (fp32, 56x56 tokens, C = 96: 757 us for 230 us of GPU work with separate
    functions, concatenation nodes and a fill per accumulator, 525-690 us so;
    437-625 us, from run to run of the host, with the fp32 kernel that serves
    that shape's whole forward in one launch and keeps what the backward reads)."""

    @staticmethod
    def forward(ctx, x, ln_w, ln_b, qw, kw, vw, qb, kb, vb, pw, pb, table, geom, eps, num_heads, scale, mask, fused):
        C = geom.channels
        w, b = torch.cat((qw, kw, vw), 0), None if qb is None else torch.cat((qb, kb, vb), 0)
        ctx.cfg = (geom, eps, num_heads, scale, mask)
        if fused and x.dtype == torch.float32 and not torch.is_autocast_enabled(x.device.type):
            # The small fp32 configuration: the whole forward in one launch.
            done = kernels.swin_block_f32_train(x, geom, num_heads, scale, w, b, pw, pb, ln_w, ln_b, eps, table, mask)
            if done is not None:
                y, windows, qkv, o = done
                ctx.dtypes = (x.dtype, x.dtype, qw.dtype, None if qb is None else qb.dtype, pw.dtype, pb.dtype)
                ctx.save_for_backward(x, ln_w, ln_b, windows, w, qkv, table, o, pw)
                return y
        windows = kernels.swin_partition_ln(x, geom, ln_w, ln_b, eps, out_dtype=linear_input_dtype(x))
        qkv, xw, wc = _linear_forward(windows, w, b)
        ws = (geom.window, geom.window)
        o = kernels.window_attention(qkv[..., :C], qkv[..., C:2 * C], qkv[..., 2 * C:], num_heads, ws, scale,
                                     bias_table=table, mask=mask)
        p, oc, pwc = _linear_forward(o, pw, pb)
        out_dtype = torch.promote_types(p.dtype, x.dtype)
        if out_dtype != p.dtype and not (p.dtype == torch.bfloat16 and out_dtype == torch.float32):
            p = p.to(out_dtype)
        y = kernels.swin_reverse(p.contiguous(), geom, residual=x.to(out_dtype), out_dtype=out_dtype)
        ctx.dtypes = (windows.dtype, p.dtype, qw.dtype, None if qb is None else qb.dtype, pw.dtype, pb.dtype)
        ctx.save_for_backward(x, ln_w, ln_b, xw, wc, qkv, table, oc, pwc)
        return y

    @staticmethod
    def backward(ctx, dy: torch.Tensor):
        x, ln_w, ln_b, xw, wc, qkv, table, oc, pwc = ctx.saved_tensors
        geom, eps, num_heads, scale, mask = ctx.cfg
        win_dtype, p_dtype, w_dtype, b_dtype, pw_dtype, pb_dtype = ctx.dtypes
        need = ctx.needs_input_grad
        C, dev = geom.channels, x.device
        # Accumulators the kernels add into, in one zeroed buffer.
        sums_p = p_dtype != dy.dtype and need[10]
        sums_qkv = b_dtype is not None and any(need[6:9]) and kernels.attention_backward_sums_supported(
            qkv[..., :C], num_heads, (geom.window, geom.window), None)
        sizes = [C if sums_p else 0, 3 * C if sums_qkv else 0, table.numel() if table is not None and need[11] else 0,
                 C if ln_w is not None and need[1] else 0, C if ln_b is not None and need[2] else 0]
        sizes = [-(-n // 4) * 4 for n in sizes]  # each part 16-byte aligned
        parts = torch.zeros(sum(sizes), dtype=torch.float32, device=dev).split(sizes)
        dpb, dqkvb, dtable, dln_w, dln_b = (t if n else None for t, n in zip(parts, sizes))
        if dpb is not None:
            dpb = dpb[:C]
        if dqkvb is not None:
            dqkvb = dqkvb[:3 * C]
        if dtable is not None:
            dtable = dtable[:table.numel()].view(table.shape)
        if dln_w is not None:
            dln_w = dln_w[:C]
        if dln_b is not None:
            dln_b = dln_b[:C]
        grad = dy.contiguous().view(geom.batch, geom.height, geom.width, C)
        if p_dtype != grad.dtype:  # bf16 windows, fp32 output
            dp = kernels.swin_partition(grad, geom, out_dtype=p_dtype, column_sums=dpb)
        else:
            dp = kernels.swin_partition(grad, geom)
        dp2 = dp.view(-1, C).to(pwc.dtype)
        if need[10] and (dpb is None or dp.dtype != pwc.dtype):
            dpb = dp2.sum(0, dtype=torch.float32)
        dpw = weight_grad(dp2, oc.reshape(-1, C)).to(pw_dtype) if need[9] else None
        dq = dk = dv = dqb = dkb = dvb = dx = None
        if any(need[:9]) or need[11]:
            _check_backward(qkv[..., :C], num_heads, (geom.window, geom.window), None)
            do = _input_grad(dp2, pwc).view(oc.shape).to(qkv.dtype)
            dqkv = torch.empty_like(qkv)
            kernels.window_attention_backward(
                qkv[..., :C], qkv[..., C:2 * C], qkv[..., 2 * C:], do.contiguous(), num_heads,
                (geom.window, geom.window), scale, bias_table=table, mask=mask, dq=dqkv[..., :C],
                dk=dqkv[..., C:2 * C], dv=dqkv[..., 2 * C:], dbias=dtable, column_sums=dqkvb)
            dqkv2 = dqkv.view(-1, 3 * C)
            if any(need[3:6]):
                dw = weight_grad(dqkv2, xw.reshape(-1, C)).to(w_dtype)
                dq, dk, dv = (dw[i * C:(i + 1) * C] if need[3 + i] else None for i in range(3))
            if b_dtype is not None and any(need[6:9]):
                db = (dqkvb if dqkvb is not None else dqkv2.sum(0, dtype=torch.float32)).to(b_dtype)
                dqb, dkb, dvb = (db[i * C:(i + 1) * C] if need[6 + i] else None for i in range(3))
            if any(need[:3]):
                dxw = _input_grad(dqkv2, wc).view(xw.shape).to(win_dtype)
                # The residual's gradient is added in the LayerNorm backward's kernel.
                dx = kernels.swin_partition_ln_backward(
                    dxw.contiguous(), x, geom, ln_w, eps, dresidual=grad.to(x.dtype) if need[0] else None,
                    dweight=dln_w, dbias=dln_b)
        cast = lambda g, t: None if g is None else g.to(t)  # noqa: E731
        return (dx if need[0] else None, None if dln_w is None else dln_w.to(ln_w.dtype),
                None if dln_b is None else dln_b.to(ln_b.dtype), dq, dk, dv, dqb, dkb, dvb, dpw, cast(dpb, pb_dtype),
                None if dtable is None else dtable.to(table.dtype), None, None, None, None, None, None)


def attention_half(x: torch.Tensor, geom: WindowGeometry, norm: torch.nn.LayerNorm, attn: torch.nn.Module,
                   mask: MaskArg, fused: bool = True) -> torch.Tensor:
    """The attention half-block on x [B, H, W, C] with gradients (see
    :class:`_AttentionHalf`); ``attn``: a WindowAttention of plain Linears with
    a biased proj.  ``fused`` False keeps the forward on the staged kernels."""
    q, k, v, proj = attn.q_linear, attn.k_linear, attn.v_linear, attn.proj
    return _AttentionHalf.apply(x, norm.weight, norm.bias, q.weight, k.weight, v.weight, q.bias, k.bias, v.bias,
                                proj.weight, proj.bias, attn._table(), geom, norm.eps, attn.num_heads, attn.scale, mask, fused)
