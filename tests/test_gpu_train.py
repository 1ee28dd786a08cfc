"""The training path's kernels: the backward of the fused LayerNorm +
partition (terra_swin_partition_ln_bwd), alone and inside the block, and the
MLP half's backward (autograd.mlp), against torch autograd of the oracle's
restatement; the mixed-dtype gather / scatter of bf16 autocast and the GELU
backward (terra_swin_gelu_bwd), each with its bias-gradient column sums,
against the separate ops they replace and float64 arithmetic.

Tolerances: fp32 activations, every gradient within 1e-5 of the float64
reference (max-abs relative, per tensor); bf16, within one bf16 rounding of
the output (2^-7 relative) plus 1e-2 of the tensor's max-abs for dx, and
2e-2 max-abs relative for the parameter gradients (fp32 sums over tokens of
bf16 products); module-level bf16 / autocast cases 3e-2 normwise, the
block tests' bound."""
import copy

import pytest
import torch

from helpers import gain_block, params_of
from oracle import swin_oracle as so
from terra_amd import autograd, kernels, workloads
from terra_amd.kernels import WindowGeometry
from terra_amd.transformer import SequentialSwinTransformer

pytestmark = pytest.mark.gpu

CASES = [  # (B, H, W, C, ws, shift, pad, win_row_begin, win_rows, valid)
    (2, 16, 24, 192, 8, 4, (0, 0, 0, 0), 0, None, None),
    (2, 14, 21, 96, 7, 3, (0, 0, 0, 0), 0, None, None),
    (2, 20, 16, 384, 8, 4, (0, 4, 0, 0), 0, 2, (3, 4)),      # slab: rows not emitted, pad windows
    (1, 16, 16, 768, 8, 4, (0, 8, 0, 0), 0, 2, (1, 3)),      # 16 lanes per token
    (1, 16, 8, 1024, 8, 4, (0, 0, 0, 0), 0, None, None),     # C = 1024
    (1, 6, 6, 64, 4, 2, (1, 1, 1, 1), 0, None, None),        # frame padding on every side
]


def _geom(B, H, W, C, ws, s, pad, r0, rows, valid):
    return WindowGeometry(B, H, W, C, ws, s, s, pad, r0, rows, valid)


def _rel(got, ref):
    got, ref = got.double().cpu(), ref.double().cpu()
    return ((got - ref).abs().max() / ref.abs().max()).item()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("residual", [False, True])
def test_partition_ln_backward_matches_autograd(dev, dtype, case, residual):
    B, H, W, C, ws, s, pad, r0, rows, valid = case
    g = _geom(*case)
    x = (workloads.activations((B, H, W, C), 500) * 2 + 0.3).to(dtype)
    w = workloads.activations((C,), 501) * 0.2 + 1.0
    b = workloads.activations((C,), 502) * 0.2
    gw = workloads.activations((g.num_windows, ws * ws, C), 503).to(dtype)
    dres = workloads.activations((B, H, W, C), 504).to(dtype) if residual else None
    cd = torch.float64
    xr = x.to(cd).requires_grad_(True)
    wr = w.to(cd).requires_grad_(True)
    br = b.to(cd).requires_grad_(True)
    win = so.partition_frame(torch.nn.functional.layer_norm(xr, (C,), wr, br, 1e-5), ws, s, s, pad, r0, rows, valid)
    win.backward(gw.to(cd))
    want_dx = xr.grad + (dres.to(cd) if residual else 0)
    dw = torch.zeros(C, device=dev)
    db = torch.zeros(C, device=dev)
    got = kernels.swin_partition_ln_backward(gw.to(dev), x.to(dev), g, w.to(dev), 1e-5,
                                             dresidual=None if dres is None else dres.to(dev), dweight=dw, dbias=db)
    assert got.dtype == dtype and tuple(got.shape) == (B, H, W, C)
    if dtype == torch.float32:
        assert _rel(got, want_dx) <= 1e-5
        assert _rel(dw, wr.grad) <= 1e-5 and _rel(db, br.grad) <= 1e-5
    else:
        err = (got.double().cpu() - want_dx).abs()
        assert bool((err <= 2.0 ** -7 * want_dx.abs() + 1e-2 * want_dx.abs().max()).all()), err.max().item()
        assert _rel(dw, wr.grad) <= 2e-2 and _rel(db, br.grad) <= 2e-2
    # tokens no window reads: dx is the residual gradient alone (or 0)
    reads = so.partition_frame(torch.ones(B, H, W, 1), ws, s, s, pad, r0, rows, valid)
    mask = so.reverse_frame(reads, B, H, W, ws, s, s, pad, r0, rows, valid)[..., 0] == 0
    if mask.any():
        want_free = dres.float()[mask] if residual else torch.zeros_like(got.float().cpu()[mask])
        assert torch.equal(got.float().cpu()[mask], want_free)


def test_partition_ln_backward_in_place_on_residual(dev):
    """dx may be the residual-gradient tensor itself."""
    B, H, W, C, ws, s = 1, 16, 16, 192, 8, 4
    g = WindowGeometry(B, H, W, C, ws, s, s)
    x = workloads.activations((B, H, W, C), 510, torch.bfloat16).to(dev)
    gw = workloads.activations((g.num_windows, 64, C), 511, torch.bfloat16).to(dev)
    dres = workloads.activations((B, H, W, C), 512, torch.bfloat16).to(dev)
    want = kernels.swin_partition_ln_backward(gw, x, g, None, 1e-5, dresidual=dres.clone())
    got = kernels.swin_partition_ln_backward(gw, x, g, None, 1e-5, dresidual=dres, out=dres)
    assert got.data_ptr() == dres.data_ptr()
    assert torch.equal(got, want)


def _mlp_case(C, seed):
    cfg = workloads.CONFIGS["c3"]
    m = workloads.mlp_for(cfg, 1) if C == 192 else workloads.mlp_for(
        workloads.CONFIGS["c4" if C == 768 else "g1"], 1)
    with torch.no_grad():
        m.fc1.weight.mul_(4.0)
        m.fc2.weight.mul_(8.0)
        m.fc1.bias.copy_(workloads.activations(m.fc1.bias.shape, seed) * 0.1)
        m.fc2.bias.copy_(workloads.activations(m.fc2.bias.shape, seed + 1) * 0.1)
        m.norm2.weight.copy_(1.0 + 0.1 * workloads.activations((C,), seed + 2))
        m.norm2.bias.copy_(0.1 * workloads.activations((C,), seed + 3))
    return m


def _oracle_mlp_grads(m, x, gy, cd, bf16_weights=False):
    p = {k: v.detach().to(cd).clone() for k, v in m.state_dict().items()}
    if bf16_weights:
        p = {k: (v.to(torch.bfloat16).to(cd) if k.startswith("fc") else v) for k, v in p.items()}
    p = {k: v.requires_grad_(True) for k, v in p.items()}
    xr = x.to(cd).requires_grad_(True)
    h = torch.nn.functional.layer_norm(xr, (x.shape[-1],), p["norm2.weight"], p["norm2.bias"])
    h = torch.nn.functional.gelu(torch.nn.functional.linear(h, p["fc1.weight"], p["fc1.bias"]))
    y = torch.nn.functional.linear(h, p["fc2.weight"], p["fc2.bias"]) + xr
    y.backward(gy.to(cd))
    return y.detach(), xr.grad, {k: v.grad for k, v in p.items()}


def _normwise(got, ref):
    got, ref = got.double().cpu(), ref.double().cpu()
    return ((got - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("C", [192, 1024])
def test_mlp_backward_fp32(dev, C):
    """fp32 activations and parameters: the HIP LayerNorm forward / backward
    and fp32 GEMMs against float64 autograd, 1e-5 normwise per gradient."""
    m = _mlp_case(C, 520)
    x = workloads.activations((2, 150, C), 521)
    gy = workloads.activations((2, 150, C), 522)
    md = copy.deepcopy(m).to(dev)
    xd = x.to(dev).requires_grad_(True)
    y = md(xd)
    y.backward(gy.to(dev))
    yr, xg, pg = _oracle_mlp_grads(m, x, gy, torch.float64)
    assert _normwise(y.detach(), yr) <= 1e-5
    assert _normwise(xd.grad, xg) <= 1e-5
    for n, p in md.named_parameters():
        assert _normwise(p.grad, pg[n]) <= 1e-5, n


@pytest.mark.parametrize("C", [192, 768])
def test_mlp_backward_autocast(dev, C):
    """The reference's training mode: fp32 input and parameters under bf16
    autocast (bf16 GEMMs); every gradient within 3e-2 normwise of fp32
    autograd on bf16-rounded weights, and the module routes through the HIP
    LayerNorm kernels."""
    m = _mlp_case(C, 530)
    x = workloads.activations((2, 200, C), 531)
    gy = workloads.activations((2, 200, C), 532)
    md = copy.deepcopy(m).to(dev)
    calls = {"fwd": 0, "bwd": 0}
    f0, b0 = kernels.swin_partition_ln, kernels.swin_partition_ln_backward

    def cf(*a, **k):
        calls["fwd"] += 1
        return f0(*a, **k)

    def cb(*a, **k):
        calls["bwd"] += 1
        return b0(*a, **k)

    kernels.swin_partition_ln, kernels.swin_partition_ln_backward = cf, cb
    try:
        xd = x.to(dev).requires_grad_(True)
        with torch.amp.autocast(device_type="cuda", dtype=torch.bfloat16):
            y = md(xd)
        y.backward(gy.to(dev))
    finally:
        kernels.swin_partition_ln, kernels.swin_partition_ln_backward = f0, b0
    assert calls == {"fwd": 1, "bwd": 1}
    assert y.dtype == torch.float32
    yr, xg, pg = _oracle_mlp_grads(m, x, gy, torch.float32, bf16_weights=True)
    assert _normwise(y.detach(), yr) <= 2e-2
    assert _normwise(xd.grad, xg) <= 3e-2
    for n, p in md.named_parameters():
        assert p.grad is not None and p.grad.dtype == torch.float32, n
        assert _normwise(p.grad, pg[n]) <= 3e-2, n


def test_block_training_routes_layernorm_through_hip(dev):
    """A bf16 block's training forward / backward runs its LayerNorm on the
    fused gather and its backward kernel (no torch LayerNorm)."""
    cfg = workloads.CONFIGS["c3"].scaled(16, 32)
    blk = gain_block(workloads.block_for(cfg, 1)).to(dev).to(torch.bfloat16)
    calls = {"bwd": 0}
    b0 = kernels.swin_partition_ln_backward

    def cb(*a, **k):
        calls["bwd"] += 1
        return b0(*a, **k)

    ln_calls = {"n": 0}
    orig_ln = torch.nn.functional.layer_norm

    def count_ln(*a, **k):
        ln_calls["n"] += 1
        return orig_ln(*a, **k)

    kernels.swin_partition_ln_backward = cb
    torch.nn.functional.layer_norm = count_ln
    try:
        x = workloads.activations((1, 16 * 32, cfg.channels), 540, torch.bfloat16).to(dev).requires_grad_(True)
        blk(x).sum().backward()
    finally:
        kernels.swin_partition_ln_backward = b0
        torch.nn.functional.layer_norm = orig_ln
    assert calls["bwd"] == 1 and ln_calls["n"] == 0
    assert blk.norm1.weight.grad is not None and torch.isfinite(blk.norm1.weight.grad.float()).all()


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("residual", [False, True])
def test_partition_ln_mixed_equals_fp32_and_cast(dev, case, residual):
    """The mixed-dtype forms (fp32 x, bf16 windows / bf16 windows gradient)
    that bf16-autocast training uses: the forward equals the fp32 LayerNorm +
    partition followed by a cast to bf16, and the backward equals the fp32
    backward on the bf16 gradient cast to fp32, bit for bit (dγ / dβ up to
    the atomics' summation order)."""
    B, H, W, C, ws, s, pad, r0, rows, valid = case
    g = _geom(*case)
    x = (workloads.activations((B, H, W, C), 510) * 2 + 0.3).to(dev)
    w = (workloads.activations((C,), 511) * 0.2 + 1.0).to(dev)
    b = (workloads.activations((C,), 512) * 0.2).to(dev)
    want = kernels.swin_partition_ln(x, g, w, b, 1e-5, pad_value=0.5).to(torch.bfloat16)
    got = kernels.swin_partition_ln(x, g, w, b, 1e-5, pad_value=0.5, out_dtype=torch.bfloat16)
    assert got.dtype == torch.bfloat16
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    gw = workloads.activations((g.num_windows, ws * ws, C), 513).to(torch.bfloat16).to(dev)
    dres = workloads.activations((B, H, W, C), 514).to(dev) if residual else None
    dw0, db0 = torch.zeros(C, device=dev), torch.zeros(C, device=dev)
    dw1, db1 = torch.zeros(C, device=dev), torch.zeros(C, device=dev)
    want_dx = kernels.swin_partition_ln_backward(gw.float(), x, g, w, 1e-5, dresidual=dres, dweight=dw0, dbias=db0)
    got_dx = kernels.swin_partition_ln_backward(gw, x, g, w, 1e-5, dresidual=dres, dweight=dw1, dbias=db1)
    assert got_dx.dtype == torch.float32
    assert torch.equal(got_dx, want_dx)
    assert _rel(dw1, dw0) < 1e-5 and _rel(db1, db0) < 1e-5


def test_partition_ln_mixed_rejects_other_pairs(dev):
    g = WindowGeometry(1, 8, 8, 64, 8)
    x = torch.zeros((1, 8, 8, 64), dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError):
        kernels.swin_partition_ln(x, g, None, None, 1e-5, out_dtype=torch.float32)
    with pytest.raises(ValueError):
        kernels.swin_partition_ln_backward(torch.zeros((1, 64, 64), dtype=torch.float16, device=dev), x.float(), g,
                                           None, 1e-5)


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("residual", [False, True])
def test_reverse_mixed_equals_widen_and_reverse(dev, case, residual):
    """bf16 windows into an fp32 grid (plus an fp32 residual): bit for bit
    the fp32 reverse of the windows cast to fp32 (the widening is exact and
    the add is the fp32 add either way)."""
    B, H, W, C, ws, s, pad, r0, rows, valid = case
    g = _geom(*case)
    win = workloads.activations((g.num_windows, ws * ws, C), 520).to(torch.bfloat16).to(dev)
    res = (workloads.activations((B, H, W, C), 521) * 3).to(dev) if residual else None
    want = kernels.swin_reverse(win.float(), g, residual=res)
    got = kernels.swin_reverse(win, g, residual=res, out_dtype=torch.float32)
    assert got.dtype == torch.float32
    assert torch.equal(got, want)
    if residual:  # in place on the residual
        res2 = res.clone()
        kernels.swin_reverse(win, g, residual=res2, out=res2, out_dtype=torch.float32)
        assert torch.equal(res2, want)


def _sum_bound(vals: torch.Tensor, dims) -> torch.Tensor:
    """Worst-case error of fp32 summation in any order: n u sum |x| (n terms,
    u = 2^-24), per column."""
    n = 1
    for d in dims:
        n *= vals.shape[d]
    return n * 2.0 ** -24 * vals.double().abs().sum(dims).cpu() + 1e-30


@pytest.mark.parametrize("case", CASES)
def test_partition_mixed_equals_partition_and_cast(dev, case):
    """fp32 grid into bf16 windows: bit for bit the fp32 partition followed
    by a cast (pad slots included), and the column sums of the values written
    within the fp32 summation bound of their float64 sums; the sums
    accumulate over calls."""
    B, H, W, C, ws, s, pad, r0, rows, valid = case
    g = _geom(*case)
    x = (workloads.activations((B, H, W, C), 522) * 3).to(dev)
    want = kernels.swin_partition(x, g, pad_value=0.5).to(torch.bfloat16)
    sums = torch.zeros(C, device=dev)
    got = kernels.swin_partition(x, g, pad_value=0.5, out_dtype=torch.bfloat16, column_sums=sums)
    assert got.dtype == torch.bfloat16
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    ref = want.double().sum((0, 1)).cpu()
    bound = _sum_bound(want, (0, 1))
    assert ((sums.double().cpu() - ref).abs() <= bound).all()
    got2 = kernels.swin_partition(x, g, pad_value=0.5, out_dtype=torch.bfloat16, column_sums=sums)
    assert torch.equal(got2.view(torch.int16), want.view(torch.int16))
    assert ((sums.double().cpu() - 2 * ref).abs() <= 2 * bound).all()
    # without sums; and the identity frame over token rows (the MLP half's cast)
    assert torch.equal(kernels.swin_partition(x, g, pad_value=0.5, out_dtype=torch.bfloat16).view(torch.int16),
                       want.view(torch.int16))
    T = B * H * W
    rows_sums = torch.zeros(C, device=dev)
    flat = kernels.swin_partition(x.view(1, T, 1, C), kernels.rows_geometry(T, C), out_dtype=torch.bfloat16,
                                  column_sums=rows_sums).view(T, C)
    assert torch.equal(flat.view(torch.int16), x.view(T, C).to(torch.bfloat16).view(torch.int16))
    assert ((rows_sums.double().cpu() - flat.double().sum(0).cpu()).abs() <= _sum_bound(flat, (0,))).all()


def _gelu_grad64(g: torch.Tensor, h: torch.Tensor) -> torch.Tensor:
    """d/dh of 0.5 h (1 + erf(h / sqrt 2)) times g, in float64."""
    g, h = g.double().cpu(), h.double().cpu()
    cdf = 0.5 * (1 + torch.erf(h / 2 ** 0.5))
    pdf = torch.exp(-0.5 * h * h) / (2 * torch.pi) ** 0.5
    return g * (cdf + h * pdf)


@pytest.mark.parametrize("dtype,features", [(torch.bfloat16, 256), (torch.bfloat16, 512), (torch.bfloat16, 768),
                                            (torch.bfloat16, 1536),
                                            (torch.bfloat16, 3072), (torch.bfloat16, 4096), (torch.float32, 768),
                                            (torch.float32, 2048)])
@pytest.mark.parametrize("rows", [1, 37, 2053])
def test_gelu_backward(dev, dtype, features, rows):
    """terra_swin_gelu_bwd against the float64 derivative (one rounding to
    the dtype plus fp32 arithmetic: 2^-8 relative for bf16, 1e-6 for fp32,
    with an absolute floor of 1e-6 of the tensor's scale for values that
    cancel to near zero) and against torch's gelu_backward (at most one bf16
    unit in the last place, and equal for at least 99.9 % of the values);
    fc1's bias gradient (the column sums of the values written) within the
    fp32 summation bound."""
    h = (workloads.activations((rows, features), 530) * 2.5).to(dtype).to(dev)
    gy = workloads.activations((rows, features), 531).to(dtype).to(dev)
    sums = torch.zeros(features, device=dev)
    got = kernels.gelu_backward(gy, h, column_sums=sums)
    assert got.dtype == dtype and got.shape == h.shape
    ref = _gelu_grad64(gy, h)
    rel = 2.0 ** -8 if dtype == torch.bfloat16 else 1e-6
    err = (got.double().cpu() - ref).abs()
    assert (err <= rel * ref.abs() + 1e-6 * ref.abs().max()).all(), err.max().item()
    want = torch.ops.aten.gelu_backward(gy, h)
    if dtype == torch.bfloat16:
        gi, wi = got.view(torch.int16).int().cpu(), want.view(torch.int16).int().cpu()
        assert (gi - wi).abs().max().item() <= 1
        assert (gi == wi).float().mean().item() >= 0.999
    else:
        assert ((got - want).abs() <= 1e-6 * want.abs() + 1e-30).float().mean().item() >= 0.999
    assert ((sums.double().cpu() - got.double().sum(0).cpu()).abs() <= _sum_bound(got, (0,))).all()
    # without sums: the same values
    assert torch.equal(kernels.gelu_backward(gy, h), got)


def test_gelu_backward_special_values(dev):
    """Zeros, tiny and huge inputs, infinities and NaN give torch's values."""
    vals = [0.0, -0.0, 1e-30, -1e-30, 2.0 ** -26, -(2.0 ** -20), 0.5, -0.5, 3.0, -3.0, 6.0, -6.0, 32.0, -32.0,
            1e4, -1e4, float("inf"), float("-inf"), float("nan")]
    h = torch.tensor(vals * 8, dtype=torch.float32)[:152].view(1, 152)
    h = torch.cat([h, torch.zeros(1, 8)], 1).to(torch.bfloat16).to(dev)  # 160 features: 20 chunks
    gy = torch.full(h.shape, -1.5, dtype=torch.bfloat16, device=dev)
    got = kernels.gelu_backward(gy, h)
    want = torch.ops.aten.gelu_backward(gy, h)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    fin = ~torch.isnan(want)
    assert torch.equal(got[fin], want[fin])


def test_gelu_backward_rejects_bad_arguments(dev):
    h = torch.zeros((4, 12), dtype=torch.bfloat16, device=dev)  # 24-byte rows
    with pytest.raises(ValueError, match="16-byte"):
        kernels.gelu_backward(h, h)
    h = torch.zeros((4, 16), dtype=torch.float16, device=dev)
    with pytest.raises(TypeError):
        kernels.gelu_backward(h, h)
    h = torch.zeros((4, 16), dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError):
        kernels.gelu_backward(h, h, column_sums=torch.zeros(8, device=dev))
    with pytest.raises(ValueError, match="overlap"):  # dh overlapping dout
        kernels.gelu_backward(h, h.clone(), out=h)


def test_mlp_backward_autocast_routes_through_fused_kernels(dev):
    """Under autocast the MLP half's backward casts the output gradient with
    terra_swin_partition_mixed (fc2's bias gradient summed there) and runs
    the GELU derivative on terra_swin_gelu_bwd (fc1's bias gradient summed
    there): one call each."""
    m = _mlp_case(192, 560)
    md = copy.deepcopy(m).to(dev)
    calls = {"part": 0, "gelu": 0}
    p0, g0 = kernels.swin_partition, kernels.gelu_backward

    def cp(*a, **k):
        if k.get("column_sums") is not None:
            calls["part"] += 1
        return p0(*a, **k)

    def cg(*a, **k):
        calls["gelu"] += 1
        return g0(*a, **k)

    kernels.swin_partition, kernels.gelu_backward = cp, cg
    try:
        x = workloads.activations((2, 96, 192), 561).to(dev).requires_grad_(True)
        with torch.amp.autocast(device_type="cuda", dtype=torch.bfloat16):
            y = md(x)
        y.backward(workloads.activations(tuple(y.shape), 562).to(dev))
    finally:
        kernels.swin_partition, kernels.gelu_backward = p0, g0
    assert calls["part"] == 1 and calls["gelu"] == 1
    assert md.fc1.bias.grad is not None and md.fc2.bias.grad is not None


def test_block_autocast_training_sums_biases_in_kernels(dev):
    """A block's training step under autocast: the scatter's backward writes
    proj's bf16 output gradient with its column sums (terra_swin_partition_mixed)
    and the attention core's backward sums the q | k | v gradient
    (terra_swin_attn_bwd_sums); the forward's scatter widens the bf16 proj
    output itself (terra_swin_reverse_mixed).  The bias gradients equal the
    column sums torch takes of the same gradients, within the fp32 summation
    bound."""
    cfg = workloads.CONFIGS["c3"].scaled(16, 32)
    blk = gain_block(workloads.block_for(cfg, 1)).to(dev)
    calls = {"part": 0, "attn": 0, "rev": 0}
    p0, a0, r0 = kernels.swin_partition, kernels.window_attention_backward, kernels.swin_reverse
    seen = {}

    def cp(*a, **k):
        if k.get("column_sums") is not None:
            calls["part"] += 1
            out = p0(*a, **k)
            seen["dproj"] = out.detach().clone()
            return out
        return p0(*a, **k)

    def ca(*a, **k):
        if k.get("column_sums") is not None:
            calls["attn"] += 1
            outs = a0(*a, **k)
            seen["dqkv"] = torch.cat([t.detach() for t in outs], -1).clone()
            return outs
        return a0(*a, **k)

    def cr(*a, **k):
        if k.get("out_dtype") == torch.float32 and a[0].dtype == torch.bfloat16:
            calls["rev"] += 1
        return r0(*a, **k)

    kernels.swin_partition, kernels.window_attention_backward, kernels.swin_reverse = cp, ca, cr
    try:
        x = workloads.activations((1, 16 * 32, cfg.channels), 570).to(dev).requires_grad_(True)
        with torch.amp.autocast(device_type="cuda", dtype=torch.bfloat16):
            y = blk(x)
        y.backward(workloads.activations(tuple(y.shape), 571).to(dev))
    finally:
        kernels.swin_partition, kernels.window_attention_backward, kernels.swin_reverse = p0, a0, r0
    assert calls == {"part": 1, "attn": 1, "rev": 1}
    C = cfg.channels
    dproj = seen["dproj"].reshape(-1, C)
    want = dproj.double().sum(0).cpu()
    got = blk.attn.proj.bias.grad.double().cpu()
    assert ((got - want).abs() <= dproj.shape[0] * 2.0 ** -24 * dproj.double().abs().sum(0).cpu() + 1e-30).all()
    dqkv = seen["dqkv"].reshape(-1, 3 * C)
    want = dqkv.double().sum(0).cpu()
    bound = dqkv.shape[0] * 2.0 ** -24 * dqkv.double().abs().sum(0).cpu() + 1e-30
    got = torch.cat([blk.attn.q_linear.bias.grad, blk.attn.k_linear.bias.grad, blk.attn.v_linear.bias.grad])
    assert ((got.double().cpu() - want).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("transpose", [False, True])
def test_pack_weight_equals_cast_transpose_and_pack(dev, dtype, transpose):
    for n, k in ((16, 32), (192, 768), (768, 96)):
        w = workloads.activations((k, n) if transpose else (n, k), 580).to(dtype).to(dev)
        p = (w.t() if transpose else w).to(torch.bfloat16).contiguous()
        assert torch.equal(kernels.pack_weight(w, transpose), kernels.pack_linear(p))


LINEAR_GELU_SHAPES = [(1, 64, 256), (257, 128, 512), (700, 192, 768), (256 * 260 + 5, 64, 768), (300, 1024, 4096)]


@pytest.mark.parametrize("rows,k,n", LINEAR_GELU_SHAPES)
def test_linear_gelu_keep(dev, rows, k, n):
    """h is the plain linear kernel's output and y the GELU kernel's, bit for
    bit (edges of the 256-row tiles, several tiles per workgroup)."""
    x = torch.randn(rows, k, device=dev, generator=torch.Generator(dev).manual_seed(581)).bfloat16()
    w = workloads.activations((n, k), 582).to(dev) * k ** -0.5
    b = workloads.activations((n,), 583).to(dev) * 0.1
    pk = kernels.pack_weight(w)
    h, y = kernels.linear_gelu_keep(x, pk, n, b)
    assert torch.equal(h, kernels.linear(x, pk, n, b))
    assert torch.equal(y, kernels.linear(x, pk, n, b, gelu=True))


@pytest.mark.parametrize("rows,k,n", LINEAR_GELU_SHAPES)
def test_linear_gelu_backward(dev, rows, k, n):
    """bf16((dy W2) * slope(h)) against float64: one fp32 sum of k products
    (k u relative to the sum of their magnitudes), one fp32 slope and one bf16
    rounding; tiny, large, infinite and NaN h; the column sums against those
    of the values written, within the fp32 summation bound."""
    g = torch.Generator(dev).manual_seed(584)
    dy = torch.randn(rows, k, device=dev, generator=g).bfloat16()
    h = (torch.randn(rows, n, device=dev, generator=g) * 2).bfloat16()
    special = torch.tensor([0.0, -0.0, 2.0 ** -13, -(2.0 ** -13), 2.0 ** -14, -(2.0 ** -20), 1e-30, 7.96875, -7.96875,
                            8.0, -8.0, 31.0, -31.0, 300.0, -300.0], device=dev).bfloat16()
    h.view(-1)[:special.numel()] = special
    w2 = workloads.activations((k, n), 585).to(dev) * n ** -0.5
    sums = torch.ones(n, device=dev)
    pk = kernels.pack_weight(w2, transpose=True)
    got = kernels.linear_gelu_backward(dy, pk, n, h, column_sums=sums)
    wd, hd = w2.bfloat16().double(), h.double()
    slope = 0.5 * (1 + torch.special.erf(hd / 2 ** 0.5)) + hd * torch.exp(-hd * hd / 2) / (2 * torch.pi) ** 0.5
    want = (dy.double() @ wd) * slope
    mag = dy.double().abs() @ wd.abs()  # what the fp32 sum's rounding scales with
    # the slope in fp32: 2^-22 absolute (erff, expf and their sum); bf16: 2^-8 of the value
    bound = want.abs() * 2.0 ** -8 + mag * (k * 2.0 ** -24 * slope.abs() + 2.0 ** -22) + 1e-30
    assert ((got.double() - want).abs() <= bound).all()
    vals = got.double()
    assert ((sums.double() - 1 - vals.sum(0)).abs() <= (rows + 8) * 2.0 ** -24 * (vals.abs().sum(0) + 1)).all()
    assert torch.equal(got, kernels.linear_gelu_backward(dy, pk, n, h))
    h[0, :3] = torch.tensor([float("inf"), float("-inf"), float("nan")], device=dev).bfloat16()
    bad = kernels.linear_gelu_backward(dy, pk, n, h)
    assert bad[0, :3].isnan().all() and not bad[1:].isnan().any() and not bad[0, 3:].isnan().any()


@pytest.mark.parametrize("x_dtype,C,tokens", [(torch.float32, 192, 21999), (torch.bfloat16, 1024, 16500)])
def test_mlp_training_on_linear_kernels(dev, x_dtype, C, tokens):
    """Rows that fill the chip run fc1 + GELU and the GELU backward on the
    linear kernels; outputs and gradients against float64 autograd of the
    bf16-rounded weights, 1e-2 normwise (the products' bf16 operands)."""
    m = _mlp_case(C, 590)
    x = workloads.activations((tokens, C), 591).to(x_dtype)
    gy = workloads.activations((tokens, C), 592).to(x_dtype)
    md = copy.deepcopy(m).to(dev)
    calls = {"keep": 0, "bwd": 0}
    k0, s0, b0 = kernels.linear_gelu_keep, kernels.linear_short, kernels.linear_gelu_backward

    def ck(*a, **k):
        calls["keep"] += 1
        return k0(*a, **k)

    def cs(*a, **k):
        calls["keep"] += bool(k.get("gelu_keep"))
        return s0(*a, **k)

    def cb(*a, **k):
        calls["bwd"] += 1
        return b0(*a, **k)

    kernels.linear_gelu_keep, kernels.linear_short, kernels.linear_gelu_backward = ck, cs, cb
    try:
        xd = x.to(dev).requires_grad_(True)
        with torch.amp.autocast(device_type="cuda", dtype=torch.bfloat16):
            y = md(xd)
        y.backward(gy.to(dev))
    finally:
        kernels.linear_gelu_keep, kernels.linear_short, kernels.linear_gelu_backward = k0, s0, b0
    assert calls == {"keep": 1, "bwd": 1} and y.dtype == x_dtype
    mref = copy.deepcopy(m).to(dev)
    yr, xg, pg = _oracle_mlp_grads(mref, x.to(dev), gy.to(dev), torch.float64, bf16_weights=True)
    assert _normwise(y.detach(), yr) <= 1e-2
    assert _normwise(xd.grad, xg) <= 1e-2
    for n, p in md.named_parameters():
        assert _normwise(p.grad, pg[n]) <= 1e-2, n


def test_mlp_training_refuses_mixed_dtypes_outside_autocast(dev):
    """bf16 rows with fp32 parameters and no autocast are refused, as F.linear refuses them, at any size."""
    m = _mlp_case(192, 595).to(dev)
    x = workloads.activations((30000, 192), 596).to(torch.bfloat16).to(dev).requires_grad_(True)
    with pytest.raises(RuntimeError):
        m(x)


# (T, out, in): one token, tails of a 32-token stage, widths that fill and do
# not fill the 256 / 192 / 128 tiles, fewer and more stages than LDS buffers,
# slices with a short last one, more tiles than compute units.
WEIGHT_GRAD_SHAPES = [(1, 16, 16), (31, 32, 48), (100, 256, 256), (161, 128, 512), (513, 192, 768), (4099, 400, 336),
                      (20000, 576, 192), (70001, 768, 192), (33, 4096, 4352)]


@pytest.mark.parametrize("T,o,i", WEIGHT_GRAD_SHAPES)
def test_weight_grad(dev, T, o, i):
    """dy^T x against float64: fp32 sums of exact bf16 products, so each entry
    is within T u of the sum of their magnitudes; the same bits twice; the
    tokens past the end (neighbouring memory full of NaN) are not read."""
    g = torch.Generator(dev).manual_seed(600)
    buf_dy = torch.full((T * o + 40 * o,), float("nan"), device=dev, dtype=torch.bfloat16)
    buf_x = torch.full((T * i + 40 * i,), float("nan"), device=dev, dtype=torch.bfloat16)
    dy, x = buf_dy[:T * o].view(T, o), buf_x[:T * i].view(T, i)
    dy.copy_(torch.randn(T, o, device=dev, generator=g))
    x.copy_(torch.randn(T, i, device=dev, generator=g))
    got = kernels.weight_grad(dy, x)
    want = dy.double().t() @ x.double()
    mag = dy.double().abs().t() @ x.double().abs()
    assert got.dtype == torch.float32 and tuple(got.shape) == (o, i)
    assert ((got.double() - want).abs() <= (T + 1) * 2.0 ** -24 * mag).all()
    assert torch.equal(got, kernels.weight_grad(dy, x))


def test_weight_grad_refuses_other_operands(dev):
    dy = torch.zeros(64, 32, device=dev, dtype=torch.bfloat16)
    for bad_dy, bad_x in ((dy.float(), dy.float()), (dy, dy[:32]), (dy.t(), dy.t()), (dy[:0], dy[:0]),
                          (dy[:, :8].contiguous(), dy)):
        with pytest.raises((ValueError, TypeError)):
            kernels.weight_grad(bad_dy, bad_x)


def test_training_accepts_parameters_at_any_offset(dev):
    """Parameters that are views into one flat buffer (4-byte offsets): the same
    gradients as aligned ones."""
    torch.manual_seed(7)
    m = _mlp_case(192, 610).to(dev)
    x = workloads.activations((9000, 192), 611).to(dev)
    gy = workloads.activations((9000, 192), 612).to(dev)

    def grads(shift):
        md = copy.deepcopy(m)
        params = list(md.parameters())
        flat = torch.empty(sum(p.numel() + shift for p in params) + shift, device=dev)
        at = shift
        for p in params:
            flat[at:at + p.numel()].copy_(p.detach().reshape(-1))
            p.data = flat[at:at + p.numel()].view(p.shape)
            at += p.numel() + shift
        xs = x.clone().requires_grad_(True)
        with torch.amp.autocast("cuda", dtype=torch.bfloat16):
            y = md(xs)
        y.backward(gy)
        return [y.detach(), xs.grad] + [p.grad for p in params]

    for a, b in zip(grads(0), grads(1)):
        assert _normwise(a, b) <= 1e-6


# (dtype, autocast, window, C, heads, frozen parameters, x needs a gradient, bias table, q/k/v bias)
HALF_CASES = [
    (torch.float32, False, 7, 96, 3, (), True, True, True),
    (torch.float32, False, 7, 96, 3, ("q_linear.weight", "k_linear.bias", "norm1.bias", "proj.bias"), False, False, True),
    (torch.float32, False, 8, 192, 6, ("proj.weight", "relative_position_bias_table"), True, True, False),
    (torch.float32, True, 8, 192, 6, ("norm1.weight",), True, True, True),
    (torch.bfloat16, False, 8, 128, 4, (), True, True, True),
    (torch.float32, True, 7, 96, 3, ("q_linear", "k_linear", "v_linear", "norm1", "table"), True, False, True),
]


@pytest.mark.parametrize("case", HALF_CASES)
def test_attention_half_matches_the_chain_of_functions(dev, case, monkeypatch):
    """The attention half-block's training step as one function against the
    chain of partition, Linear, core, Linear and reverse it replaces (masked,
    shifted, padded frame): outputs and gradients agree to the rounding of the
    compute dtype, and the same tensors get one."""
    dtype, amp, ws, C, heads, frozen, xgrad, table, qkv_bias = case
    blk = SequentialSwinTransformer(layer_idx=1, height=3 * ws - 2, width=4 * ws, embedding_dim=C, window_size=ws,
                                    num_heads=heads, use_relative_position_bias=table, pad=(1, 1, 0, 0),
                                    land_mask=workloads.land_mask(3 * ws - 2, 4 * ws, seed=81))
    workloads.init_block_params(blk, 1)
    blk = gain_block(blk)
    if not qkv_bias:
        for lin in (blk.attn.q_linear, blk.attn.k_linear, blk.attn.v_linear):
            lin.bias = None
    blk = blk.to(dev, dtype)
    for n, p in blk.named_parameters():
        p.requires_grad_(not any(f in n for f in frozen))
    x0 = workloads.activations((2, (3 * ws - 2) * 4 * ws, C), 620).to(dev, dtype)
    gy = workloads.activations(tuple(x0.shape), 621).to(dev, dtype)
    calls = []
    orig = autograd.attention_half
    monkeypatch.setattr(autograd, "attention_half", lambda *a: calls.append(1) or orig(*a))

    def step():
        x = x0.clone().requires_grad_(xgrad)
        blk.zero_grad(set_to_none=True)
        with torch.amp.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
            y = blk(x)
        y.backward(gy)
        return {"y": y.detach(), "x": x.grad, **{n: p.grad for n, p in blk.named_parameters()}}

    got = step()
    assert calls == [1]
    monkeypatch.setattr(blk, "_one_function", lambda x: False, raising=False)
    want = step()
    assert calls == [1]
    # One rounding of the compute dtype and its sums' order on either side.
    tol = 2.0 ** -8 if amp or dtype == torch.bfloat16 else 1e-5
    for name, b in want.items():
        a = got[name]
        assert (a is None) == (b is None)
        if b is not None:
            assert a.dtype == b.dtype and a.shape == b.shape
            # k's bias shifts a query's logits alike, so its exact gradient is
            # zero: what is left is rounding, on the scale of q's and v's.
            scale = want["attn.v_linear.bias"] if name == "attn.k_linear.bias" else b
            assert (a.double() - b.double()).norm() <= tol * scale.double().norm(), name


def test_attention_half_keeps_the_chain_for_other_calls(dev, monkeypatch):
    """A subclassed projection, and a call with only proj trainable, stay on
    the chain."""
    monkeypatch.setattr(autograd, "attention_half", None)
    for change in ("subclass", "frozen"):
        blk = SequentialSwinTransformer(layer_idx=0, height=14, width=14, embedding_dim=96, window_size=7, num_heads=3)
        if change == "subclass":
            blk.attn.q_linear.__class__ = type("L", (torch.nn.Linear,), {})
        else:
            blk.requires_grad_(False)
            blk.attn.proj.requires_grad_(True)
        blk = blk.to(dev)
        blk(torch.randn(1, 196, 96, device=dev)).sum().backward()
        assert blk.attn.proj.weight.grad is not None


@pytest.mark.parametrize("x_dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("C,tokens", [(192, 9000), (1024, 16500)])
def test_mlp_training_casts_fp16_parameters_under_autocast(dev, C, tokens, x_dtype):
    """fp16 parameters in a bf16 autocast region, which casts them, with rows
    that fill the chip: the gradients of the fp16 values in float64, 1e-2
    normwise (bf16 operands, weights rounded to bf16)."""
    m = _mlp_case(C, 630).to(dev, torch.float16)
    x = workloads.activations((tokens, C), 631).to(dev, x_dtype)
    gy = workloads.activations((tokens, C), 632).to(dev)
    xd = x.clone().requires_grad_(True)
    with torch.amp.autocast("cuda", dtype=torch.bfloat16):
        y = m(xd)
    y.backward(gy.to(y.dtype))
    yr, xg, pg = _oracle_mlp_grads(m, x, gy, torch.float64, bf16_weights=True)
    assert _normwise(y.detach(), yr) <= 1e-2 and _normwise(xd.grad, xg) <= 1e-2
    for n, p in m.named_parameters():
        assert p.grad.dtype == torch.float16 and _normwise(p.grad, pg[n]) <= 1e-2, n


def test_mlp_training_refuses_fp64_parameters_under_autocast(dev):
    """Autocast leaves fp64 parameters as they are and F.linear refuses them, at any size."""
    x = workloads.activations((9000, 192), 633).to(dev).requires_grad_(True)
    for name in ("weight", "bias"):
        m = _mlp_case(192, 634).to(dev)
        setattr(m.fc1, name, torch.nn.Parameter(getattr(m.fc1, name).detach().double()))
        with torch.amp.autocast("cuda", dtype=torch.bfloat16), pytest.raises(RuntimeError):
            m(x)


def test_linear_gelu_backward_slope_of_every_bf16_value(dev):
    """The slope in the linear kernel's epilogue against the GELU backward
    kernel's, bit for bit, over all 2^16 values of h: a product of 2^60 shows
    the tails, where the slope is far below fp32's resolution of 1."""
    h = torch.arange(1 << 16, device=dev).to(torch.int32).to(torch.int16).view(torch.bfloat16).view(256, 256)
    dy = torch.zeros(256, 64, device=dev, dtype=torch.bfloat16)
    dy[:, 0] = 2.0 ** 60
    w2 = torch.zeros(64, 256, device=dev)
    w2[0] = 1.0
    got = kernels.linear_gelu_backward(dy, kernels.pack_weight(w2, transpose=True), 256, h)
    want = kernels.gelu_backward(torch.full_like(h, 2.0 ** 60), h)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(0.0), want.nan_to_num(0.0))


@pytest.mark.parametrize("tokens,launches", [(6001, (0, 1, 0)), (17000, (1, 1, 0)), (26000, (1, 1, 1))])
def test_mlp_training_takes_the_linear_kernels_where_they_pay(dev, tokens, launches, monkeypatch):
    """fc1 + GELU, the GELU backward and fc1's input gradient (1024 features)
    against float64 on either side of each rule."""
    m = _mlp_case(1024, 640).to(dev)
    x, gy = (workloads.activations((tokens, 1024), s).to(dev, torch.bfloat16) for s in (641, 642))
    calls = []
    names = ("linear_gelu_keep", "linear_gelu_backward", "linear")
    for name in names:
        real = getattr(kernels, name)
        monkeypatch.setattr(kernels, name, lambda *a, name=name, real=real, **k: calls.append(name) or real(*a, **k))
    xd = x.clone().requires_grad_(True)
    with torch.amp.autocast("cuda", dtype=torch.bfloat16):
        y = m(xd)
    y.backward(gy)
    assert tuple(calls.count(n) for n in names) == launches
    yr, xg, pg = _oracle_mlp_grads(m, x, gy, torch.float64, bf16_weights=True)
    assert _normwise(y.detach(), yr) <= 1e-2 and _normwise(xd.grad, xg) <= 1e-2
    for n, p in m.named_parameters():
        assert _normwise(p.grad, pg[n]) <= 1e-2, n


@pytest.mark.parametrize("mean", [0.0, 0.3])
@pytest.mark.parametrize("T,o,i", [(156672, 4096, 1024), (156673, 3072, 1024), (524288, 768, 192)])
def test_weight_grad_sums_long_contractions_in_two_levels(dev, T, o, i, mean):
    """Normwise error against float64 over 64 output features.  fp32 sums of n
    independent terms in one chain are off by about 3.6e-8 sqrt(n / 32) of the
    result (n / 32 MFMA steps, measured); 32 steps a chain and 77 chains a slice
    leave 2.0e-7 and 1.5e-7.  One chain per slice gave 1.3e-6, 1.1e-6 and 5.2e-7,
    the library's sums over 64 and 128 slices 3.1e-7 and 4.1e-7."""
    g = torch.Generator(dev).manual_seed(601)
    dy = (torch.randn(T, o, device=dev, generator=g) + mean).bfloat16()
    x = (torch.randn(T, i, device=dev, generator=g) + mean).bfloat16()
    got = kernels.weight_grad(dy, x)[:64].double()
    want = dy[:, :64].double().t().contiguous() @ x.double()
    assert ((got - want).norm() / want.norm()).item() <= 3e-7


@pytest.mark.parametrize("T,o,i", [(1023, 256, 128), (1024, 512, 256), (1025, 192, 384), (2049, 208, 144), (5000, 3072, 1024),
                                   (16385, 3072, 1024), (40000, 1152, 1152), (600, 16, 4096), (600, 4096, 16)])
def test_weight_grad_tiles_and_folds(dev, T, o, i):
    """Every tile shape, chains that end at, before and after the end of a
    slice, one and several rounds of slices, grids of tiles longer on either
    side: within T u of the sum of magnitudes, the same bits twice."""
    g = torch.Generator(dev).manual_seed(602)
    dy, x = (torch.randn(T, n, device=dev, generator=g).bfloat16() for n in (o, i))
    got = kernels.weight_grad(dy, x)
    want, mag = dy.double().t().contiguous() @ x.double(), dy.double().abs().t().contiguous() @ x.double().abs()
    assert ((got.double() - want).abs() <= (T + 1) * 2.0 ** -24 * mag).all()
    assert torch.equal(got, kernels.weight_grad(dy, x))
