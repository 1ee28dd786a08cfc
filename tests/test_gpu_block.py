"""The drop-in SequentialSwinTransformer against the oracle's restatement of
the reference block, on identical seeded inputs and weights.

Weights are scaled (helpers.gain_block) so that the attention term y - x is
O(1): with the reference's std-0.02 init it is ~0.02 and a check on y alone
would see mostly the residual.  Tolerances:
  fp32: max-abs relative error on y <= 1e-5, and normwise relative error on
        y - x <= 1e-5 (the contract's fp32 bound; the GEMMs differ from the
        CPU's only in summation order);
  bf16: max-abs relative error on y <= 2e-2, normwise on y - x <= 3e-2,
        against the fp32 oracle on the bf16-rounded weights.
"""
import pytest
import torch

from helpers import assert_block_matches, gain_block, params_of
from oracle import swin_oracle as so
from terra_amd import kernels, workloads
from terra_amd.attention import WindowAttention
from terra_amd.transformer import SequentialSwinTransformer

pytestmark = pytest.mark.gpu

TOL = {torch.float32: (1e-5, 1e-5), torch.bfloat16: (2e-2, 3e-2)}


def _block_case(dev, cfg, layer, dtype, land=None, seed=300, gain=True):
    blk = workloads.block_for(cfg, layer, land=land)
    if gain:
        gain_block(blk)
    blk = blk.to(dev).to(dtype)
    x = workloads.activations((cfg.batch, cfg.height * cfg.width, cfg.channels), seed, dtype)
    with torch.no_grad():
        y = blk(x.to(dev))
    ref = so.swin_block_attention(x, cfg.height, cfg.width, cfg.window, blk.shift_size, cfg.heads, params_of(blk),
                                  land=land, pad=cfg.pad, win_row_begin=cfg.win_row_begin, win_rows=cfg.win_rows,
                                  valid=cfg.valid)
    return y, ref, x


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("layer", [0, 1])
def test_block_c1_c2_shapes(dev, dtype, layer):
    cfg = workloads.CONFIGS["c2"].scaled(28, 42, batch=2)  # ws 7, shift 3 on odd layers
    y, ref, x = _block_case(dev, cfg, layer, dtype)
    assert_block_matches(y, ref, x, *TOL[dtype])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_block_c3_shape_with_land(dev, dtype):
    cfg = workloads.CONFIGS["c3"].scaled(64, 128)
    land = workloads.land_mask(64, 128, seed=301)
    y, ref, x = _block_case(dev, cfg, 1, dtype, land=land)
    assert_block_matches(y, ref, x, *TOL[dtype])


def test_block_c1_fp32_reference_init(dev):
    """c1 as BASELINE states it (fp32, std-0.02 weights, no gain): the contract's
    1e-5 on y and on the attention term."""
    cfg = workloads.CONFIGS["c1"]
    y, ref, x = _block_case(dev, cfg, 0, torch.float32, gain=False)
    assert_block_matches(y, ref, x, 1e-5, 1e-5, min_delta=1e-3)


def test_block_c5_slab(dev):
    cfg = workloads.CONFIGS["c5"]
    land = workloads.land_mask(cfg.height, cfg.width, seed=302)
    y, ref, x = _block_case(dev, cfg, 1, torch.bfloat16, land=land)
    assert_block_matches(y, ref, x, *TOL[torch.bfloat16])
    # slab rows 0..3 take their SW-MSA output from the previous rank: here the
    # residual passes through unchanged
    yb = y.view(cfg.batch, cfg.height, cfg.width, cfg.channels).cpu()
    xb = x.view(cfg.batch, cfg.height, cfg.width, cfg.channels)
    assert torch.equal(yb[:, :4], xb[:, :4])


@pytest.mark.parametrize("layer", [0, 1])
def test_block_c4_shape(dev, layer):
    """The reference model's block (C=768, 12 heads of dim 64) at full size,
    W-MSA and SW-MSA."""
    cfg = workloads.CONFIGS["c4"]
    y, ref, x = _block_case(dev, cfg, layer, torch.bfloat16)
    assert_block_matches(y, ref, x, *TOL[torch.bfloat16])


@pytest.mark.parametrize("layer", [0, 1])
def test_block_g1_shape(dev, layer):
    """TERRA's shipped pretrain block (C=1024, 8 heads of dim 128, window 8,
    288x544 tokens) at full size, W-MSA and SW-MSA."""
    cfg = workloads.CONFIGS["g1"]
    y, ref, x = _block_case(dev, cfg, layer, torch.bfloat16, seed=305)
    assert_block_matches(y, ref, x, *TOL[torch.bfloat16])


def test_block_g1_takes_the_proj_scatter_kernel(dev, monkeypatch):
    """bf16 inference at C = 1024 projects, reverses and adds the residual in
    one linear-kernel launch (and matches the oracle: the g1 tests above)."""
    calls = []
    real = kernels.linear_residual

    def spy(*a, **k):
        calls.append(k.get("geom"))
        return real(*a, **k)

    monkeypatch.setattr(kernels, "linear_residual", spy)
    cfg = workloads.CONFIGS["g1"].scaled(16, 32)
    y, ref, x = _block_case(dev, cfg, 1, torch.bfloat16, seed=308)
    assert len(calls) == 1 and calls[0] is not None
    assert_block_matches(y, ref, x, *TOL[torch.bfloat16])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_block_g1_small_with_land(dev, dtype):
    """Head dim 128 in fp32 (the contract's 1e-5) and bf16, SW-MSA with a land
    mask, on a reduced grid."""
    cfg = workloads.CONFIGS["g1"].scaled(16, 32)
    land = workloads.land_mask(16, 32, seed=306)
    y, ref, x = _block_case(dev, cfg, 1, dtype, land=land, seed=307)
    assert_block_matches(y, ref, x, *TOL[dtype])


def test_block_c4_small_sw_msa_with_land(dev):
    """C=768, 12 heads, SW-MSA with a land mask on a small grid."""
    cfg = workloads.CONFIGS["c4"].scaled(32, 48)
    land = workloads.land_mask(32, 48, seed=303)
    y, ref, x = _block_case(dev, cfg, 1, torch.bfloat16, land=land, seed=304)
    assert_block_matches(y, ref, x, *TOL[torch.bfloat16])


def test_c2_basic_layer_wmsa_then_swmsa_with_mlp(dev):
    """Config 2: W-MSA block, MLP, SW-MSA block (shift 3, 9-region mask), MLP,
    with gained weights, checked on the output and on the change the four
    halves make to x."""
    cfg = workloads.CONFIGS["c2"]
    dtype = torch.bfloat16
    blocks = [gain_block(workloads.block_for(cfg, 0)), workloads.mlp_for(cfg, 0),
              gain_block(workloads.block_for(cfg, 1), seed=420), workloads.mlp_for(cfg, 1)]
    for m in (blocks[1], blocks[3]):
        with torch.no_grad():
            m.fc1.weight.mul_(4.0)
            m.fc2.weight.mul_(8.0)
    x = workloads.activations((cfg.batch, cfg.height * cfg.width, cfg.channels), 310, dtype)
    y = x.to(dev)
    with torch.no_grad():
        for b in blocks:
            y = b.to(dev).to(dtype)(y)
    r = x.float()
    for b in blocks:
        p = params_of(b)
        if hasattr(b, "fc1"):
            r = so.mlp(r, p)
        else:
            r = so.swin_block_attention(r, cfg.height, cfg.width, cfg.window, b.shift_size, cfg.heads, p)
    assert blocks[2].shift_size == 3
    assert_block_matches(y, r.view(cfg.batch, cfg.height * cfg.width, cfg.channels), x, 2e-2, 3e-2)


def test_window_attention_rejects_wrong_out(dev):
    q = workloads.activations((4, 64, 64), 320, torch.bfloat16).to(dev)
    with pytest.raises(ValueError, match="out must be a torch.bfloat16 tensor"):
        kernels.window_attention(q, q, q, 2, (8, 8), 0.2, out=torch.empty(4, 64, 64, device=dev))


def test_c4_chain_alternating_blocks_with_mlp(dev):
    """Four blocks at the reference model's width (C=768, 12 heads of dim 64,
    window 8): W-MSA and SW-MSA alternating by layer index (shift from
    models/transformer.py:88), each followed by its MLP half, in the order
    BasicLayer runs them (models/reference_model/parallel_layers.py:151-153),
    through the drop-ins (fused MLP kernel, fused attention half-block)
    against the oracle chain, on a reduced grid."""
    cfg = workloads.CONFIGS["c4"].scaled(32, 64)
    dtype = torch.bfloat16
    layers = []
    for layer in range(4):
        layers.append(gain_block(workloads.block_for(cfg, layer), seed=430 + 10 * layer))
        m = workloads.mlp_for(cfg, layer)
        with torch.no_grad():
            m.fc1.weight.mul_(4.0)
            m.fc2.weight.mul_(4.0)
        layers.append(m)
    assert [b.shift_size for b in layers[::2]] == [0, 4, 0, 4]
    x = workloads.activations((cfg.batch, cfg.height * cfg.width, cfg.channels), 440, dtype)
    y = x.to(dev)
    with torch.no_grad():
        for b in layers:
            y = b.to(dev).to(dtype)(y)
    r = x.float()
    for b in layers:
        p = params_of(b)
        if hasattr(b, "fc1"):
            r = so.mlp(r, p)
        else:
            r = so.swin_block_attention(r, cfg.height, cfg.width, cfg.window, b.shift_size, cfg.heads, p)
    assert_block_matches(y, r.view(cfg.batch, cfg.height * cfg.width, cfg.channels), x, 2e-2, 3e-2)


def test_c4_stack_24_blocks_full_size(dev):
    """The c4 model's Swin stack at full size: 24 blocks at 128x256 tokens
    (C=768, 12 heads of dim 64, window 8), W-MSA and SW-MSA alternating by
    layer index (models/transformer.py:88), each followed by its MLP half, in
    BasicLayer's order (models/reference_model/parallel_layers.py:151-153).
    - every half: the fused kernel against the five-stage path (torch's ops
      for the MLP) on the same input, and every output finite;
    - the first two block pairs against the oracle chain;
    - end to end: the fused chain against the five-stage chain run
      separately, normwise on y - x (error growth through depth).
    Weights: the reference init with q/k x4 (O(1) logits), proj x4, bias
    table x25, fc1 and fc2 x2, so each half changes its input visibly while
    the residual stream stays bounded over 48 halves."""
    cfg = workloads.CONFIGS["c4"]
    dtype = torch.bfloat16
    halves = []
    for layer in range(24):
        blk = workloads.block_for(cfg, layer)
        with torch.no_grad():
            for lin in (blk.attn.q_linear, blk.attn.k_linear):
                lin.weight.mul_(4.0)
            blk.attn.proj.weight.mul_(4.0)
            blk.attn.relative_position_bias_table.mul_(25.0)
        m = workloads.mlp_for(cfg, layer)
        with torch.no_grad():
            m.fc1.weight.mul_(2.0)
            m.fc2.weight.mul_(2.0)
        halves += [blk, m]
    assert [b.shift_size for b in halves[::2]] == [0, 4] * 12
    x = workloads.activations((cfg.batch, cfg.height * cfg.width, cfg.channels), 450, dtype)
    gpu = [h.to(dev).to(dtype) for h in halves]

    def run(h, inp, fused):
        if hasattr(h, "fc1"):
            h.use_fused_mlp = fused
        else:
            h.use_fused_block = fused
        try:
            with torch.no_grad():
                return h(inp)
        finally:
            h.use_fused_mlp = h.use_fused_block = True

    y = x.to(dev)
    y_five = x.to(dev)
    outs = []
    for i, h in enumerate(gpu):
        y_f = run(h, y, True)
        y_u = run(h, y, False)
        assert torch.isfinite(y_f.float()).all() and torch.isfinite(y_u.float()).all(), i
        d_u = (y_u.float() - y.float())
        tol = 2.0 ** -7 * y_u.float().abs() + 2e-2 * d_u.abs().max()
        assert bool(((y_f.float() - y_u.float()).abs() <= tol).all()), (i, float((y_f.float() - y_u.float()).abs().max()))
        y = y_f
        y_five = run(h, y_five, False)
        if i == 3:
            outs.append(y.cpu())
    # the first two block pairs (four halves) against the oracle chain
    r = x.float()
    for h in halves[:4]:
        p = params_of(h)
        if hasattr(h, "fc1"):
            r = so.mlp(r, p)
        else:
            r = so.swin_block_attention(r, cfg.height, cfg.width, cfg.window, h.shift_size, cfg.heads, p)
    assert_block_matches(outs[0], r.view_as(x), x, 2e-2, 3e-2)
    # end to end through 48 halves: the two chains stay together
    d_f = y.double().cpu() - x.double()
    d_u = y_five.double().cpu() - x.double()
    assert torch.isfinite(d_f).all()
    growth = (torch.linalg.vector_norm(d_f - d_u) / torch.linalg.vector_norm(d_u)).item()
    print(f"24-block stack: |y - x| max {d_u.abs().max().item():.3f}, fused vs five-stage normwise {growth:.3e}")
    assert growth <= 5e-2, growth


# (channels, heads, window, height, width, dtype): the fp32 kernel, the scatter launch of other windows and of 8x8 ones
ONE_LAUNCH_BLOCKS = [(96, 3, 7, 28, 28, torch.float32), (512, 4, 32, 256, 128, torch.bfloat16),
                     (256, 2, 8, 16, 16, torch.bfloat16)]


@pytest.mark.parametrize("C,heads,ws,H,W,dtype", ONE_LAUNCH_BLOCKS)
@pytest.mark.parametrize("how", ["hook", "pre-hook", "global hook", "subclass", "instance forward"])
def test_one_launch_blocks_keep_the_call_of_attn(dev, C, heads, ws, H, W, dtype, how):
    """Forward hooks on attn and a forward of its own are seen where proj or
    the whole half-block would otherwise run in one launch."""
    blk = SequentialSwinTransformer(layer_idx=0, height=H, width=W, embedding_dim=C, window_size=ws, num_heads=heads,
                                    use_attn_mask=False, use_relative_position_bias=False)
    blk = blk.to(dev, dtype)
    x = workloads.activations((1, H * W, C), 90).to(dev, dtype)
    calls = []
    handle = None
    orig = blk.attn.forward
    if how == "hook":
        blk.attn.register_forward_hook(lambda m, a, out: calls.append(1))
    elif how == "pre-hook":
        blk.attn.register_forward_pre_hook(lambda m, a: calls.append(1))
    elif how == "global hook":
        handle = torch.nn.modules.module.register_module_forward_hook(
            lambda m, a, out: calls.append(1) if m is blk.attn else None)
    elif how == "subclass":
        blk.attn.__class__ = type("Own", (WindowAttention,), {"forward": lambda self, *a, **k: calls.append(1) or orig(*a, **k)})
    else:
        blk.attn.forward = lambda *a, **k: calls.append(1) or orig(*a, **k)
    try:
        with torch.no_grad():
            blk(x)
    finally:
        if handle is not None:
            handle.remove()
    assert calls == [1]


@pytest.mark.parametrize("C,heads,ws,H,W,dtype", ONE_LAUNCH_BLOCKS)
@pytest.mark.parametrize("own", [None, "attend", "qkv"])
def test_one_launch_blocks_of_a_subclass(dev, C, heads, ws, H, W, dtype, own, monkeypatch):
    """A subclass of WindowAttention that keeps its forward takes the launches
    that WindowAttention takes; one with an attend or qkv of its own has it
    called (the scatter launch starts behind attend)."""
    blk = SequentialSwinTransformer(layer_idx=0, height=H, width=W, embedding_dim=C, window_size=ws, num_heads=heads,
                                    use_attn_mask=False, use_relative_position_bias=False)
    blk = blk.to(dev, dtype)
    x = workloads.activations((1, H * W, C), 91).to(dev, dtype)
    entry = {7: "swin_block_f32", 32: "linear_scatter", 8: "linear_residual"}[ws]
    launches, calls = [], []
    real = getattr(kernels, entry)
    monkeypatch.setattr(kernels, entry, lambda *a, **k: launches.append(1) or real(*a, **k))
    methods = {}
    if own is not None:
        orig = getattr(blk.attn, own)
        methods[own] = lambda self, *a, **k: calls.append(1) or orig(*a, **k)
    blk.attn.__class__ = type("Own", (WindowAttention,), methods)
    with torch.no_grad():
        blk(x)
    assert len(calls) == (own is not None)
    assert len(launches) == (own is None or ws != 7)


@pytest.mark.parametrize("C,heads,ws,H,W", [(512, 4, 32, 256, 128), (256, 2, 8, 16, 16)])
def test_bf16_block_takes_x_at_any_offset(dev, C, heads, ws, H, W):
    """x two bytes off an 8-byte boundary, behind a norm that is not fused: the
    residual the scatter launch does not read goes through the staged path, to
    the bf16 roundings of the product and of the sum."""
    blk = SequentialSwinTransformer(layer_idx=0, height=H, width=W, embedding_dim=C, window_size=ws, num_heads=heads,
                                    use_attn_mask=False, use_relative_position_bias=False,
                                    norm_layer=type("Norm", (torch.nn.LayerNorm,), {})).to(dev, torch.bfloat16)
    buf = workloads.activations((H * W * C + 1,), 91).to(dev, torch.bfloat16)
    x = buf[1:].view(1, H * W, C)
    assert x.data_ptr() % 8 == 2
    with torch.no_grad():
        got, want = blk(x), blk(x.clone())
    assert (got.float() - want.float()).norm() <= 2.0 ** -8 * want.float().norm()
