"""The work a user of this framework has it do, as measurable cases.

A case is one pass of one half of a Swin block through the drop-in modules:
the attention half (``SequentialSwinTransformer``) or the MLP half
(``SequentialMlp``), either a forward without gradients or a training pass
(forward, backward, every parameter's gradient).  ``listed()`` holds the
configurations of ``terra_amd.workloads``; ``draw()`` gives other grids,
widths, data types and options of the same ranges, odd sizes among them.

Weights have the scale of a trained block (outputs of each Linear of order
one, a bias table that matters), so that no term hides behind the residual.
"""
from __future__ import annotations

import contextlib
import math

import torch
import torch.nn.functional as F

from terra_amd.mlp import SequentialMlp
from terra_amd.transformer import SequentialSwinTransformer

DEVICE = "cuda"
# Widths of the repository's configurations: channels -> (heads, window).
WIDTHS = {96: (3, 7), 128: (4, 7), 192: (6, 8), 384: (12, 8), 768: (12, 8), 1024: (8, 8)}


def _attn(channels, height, width, *, name=None, batch=1, window=None, shift=True, mask=True, bias=True, land=False,
          pad_bottom=0, pad_right=0, win_rows=0, valid_begin=0, valid_end=0, train=False, x="bf16", params="bf16"):
    heads, win = WIDTHS[channels]
    case = dict(half="attention", train=train, x=x, params=params, batch=batch, height=height, width=width,
                channels=channels, heads=heads, window=window or win, shift=shift, mask=mask, bias=bias, land=land,
                pad_bottom=pad_bottom, pad_right=pad_right, win_rows=win_rows, valid_begin=valid_begin,
                valid_end=valid_end)
    return dict(case, name=name) if name else case


def _mlp(channels, tokens, *, name=None, batch=1, train=False, x="bf16", params="bf16"):
    case = dict(half="mlp", train=train, x=x, params=params, batch=batch, tokens=tokens, channels=channels)
    return dict(case, name=name) if name else case


def listed():
    return [
        # One small fp32 image (56x56 tokens, 7x7 windows, no shift): the shortest call there is, a chain of small
        # launches, as in a correctness run or an interactive forecast on a small grid.
        _attn(96, 56, 56, name="attn_fp32_c96", shift=False, x="fp32", params="fp32"),
        # The same block trained in fp32 with the shift and its mask: what a correctness run of the training does.
        _attn(96, 56, 56, name="train_attn_fp32_c96", train=True, x="fp32", params="fp32"),
        # A small batch of 112x112 grids, bf16, shifted 7x7 windows (49 tokens: ragged against every tile).
        _attn(128, 112, 112, name="attn_c128", batch=4),
        # The benchmark's step: 512x1024 tokens, shifted windows, land mask, bf16 inference.
        _attn(192, 512, 1024, name="attn_c192", land=True),
        # The MLP half that follows it.
        _mlp(192, 512 * 1024, name="mlp_c192"),
        # One rank's ragged slab of a window-parallel grid: pad windows at both ends, halo rows, land.
        _attn(384, 296, 512, name="attn_c384_slab", batch=2, land=True, pad_bottom=8, win_rows=37, valid_begin=27,
              valid_end=2358),
        # A wide stack's MLP half on a 128x256 grid: fp32 parameters under bf16 autocast, as the model evaluates.
        _mlp(768, 128 * 256, name="mlp_c768_autocast", params="fp32"),
        # The pretraining block's attention half (288x544 grid, 8 heads of dim 128), inference.
        _attn(1024, 288, 544, name="attn_c1024"),
        # The correctness configuration of the same grid: 32x32 windows, no bias, no mask.
        _attn(1024, 288, 544, name="attn_c1024_w32", window=32, mask=False, bias=False),
        # Training under bf16 autocast with fp32 parameters and fp32 activations, both halves of the benchmark's block.
        _attn(192, 512, 1024, name="train_attn_c192", land=True, train=True, x="fp32", params="fp32"),
        _mlp(192, 512 * 1024, name="train_mlp_c192", train=True, x="fp32", params="fp32"),
        # Training of the pretraining block's MLP half: bf16 activations (a bf16 residual stream), fp32 parameters.
        _mlp(1024, 288 * 544, name="train_mlp_c1024", train=True, params="fp32"),
    ]


def draw(rng):
    """One more case: any width, both halves, inference and training, small to large grids."""
    channels = rng.choice((96, 128, 192, 192, 384, 768, 1024))
    train = rng.random() < 0.5
    small = channels == 96  # the fp32 configuration
    most = (2e7 if small else 1e8) / channels
    tokens = int(math.exp(rng.uniform(math.log(2000), math.log(most))))
    # fp32 throughout at C = 96; else bf16 parameters, or fp32 ones under autocast with bf16 or fp32 activations.
    x, params = ("fp32", "fp32") if small else rng.choice((("bf16", "bf16"), ("bf16", "fp32"), ("fp32", "fp32")))
    if train and not small and params == "bf16":
        params = "fp32"
    if rng.random() < 0.4:
        return _mlp(channels, tokens | 1, train=train, x=x, params=params)
    heads, window = WIDTHS[channels]
    if channels == 1024 and rng.random() < 0.2:
        rows = max(1, min(9, int(math.sqrt(tokens) / 32)))
        cols = max(1, tokens // (rows * 1024))
        return _attn(channels, 32 * rows, 32 * cols, window=32, mask=False, bias=False, shift=rng.random() < 0.5,
                     train=train, x=x, params=params)
    batch = rng.choice((1, 1, 1, 2, 3))
    windows = max(4, tokens // (batch * window * window))
    rows = max(2, int(math.sqrt(windows) * rng.uniform(0.5, 1.0)))
    cols = max(2, windows // rows)
    odd = rng.random() < 0.3  # a grid that is no whole number of windows, padded by the model
    pad_bottom, pad_right = (rng.randrange(window), rng.randrange(window)) if odd else (0, 0)
    shift = rng.random() < 0.7
    return _attn(channels, rows * window - pad_bottom, cols * window - pad_right, batch=batch, shift=shift,
                 mask=rng.random() < 0.9, land=rng.random() < 0.3, pad_bottom=pad_bottom, pad_right=pad_right,
                 train=train, x=x, params=params)


def _dtype(name):
    return torch.float32 if name == "fp32" else torch.bfloat16


def _autocast(case):
    """fp32 parameters with a bf16 half-block: the framework's autocast mode."""
    return case["params"] == "fp32" and case["channels"] != 96


def _rows(case):
    return case["tokens"] if case["half"] == "mlp" else case["height"] * case["width"]


def _inputs(case, seed):
    """x, the output gradient, the land grid and the parameters, on the device, from the seed alone."""
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    C = case["channels"]

    def normal(*shape, std=1.0, mean=0.0, dtype=None):
        t = torch.randn(*shape, generator=g, device=DEVICE) * std + mean
        return t.to(_dtype(dtype or case["params"]))

    shape = (case["batch"], _rows(case), C)
    t = {"x": normal(*shape, dtype=case["x"])}
    if case["train"]:
        t["dy"] = normal(*shape, dtype=case["x"])
    p = {}
    norm = "norm1" if case["half"] == "attention" else "norm2"
    p[norm + ".weight"] = normal(C, std=0.1, mean=1.0)
    p[norm + ".bias"] = normal(C, std=0.1)
    if case["half"] == "attention":
        if case["bias"]:
            n = (2 * case["window"] - 1) ** 2
            p["attn.relative_position_bias_table"] = normal(n, case["heads"], std=0.5)
        for lin in ("q_linear", "k_linear", "v_linear", "proj"):
            p[f"attn.{lin}.weight"] = normal(C, C, std=C ** -0.5)
            p[f"attn.{lin}.bias"] = normal(C, std=0.1)
        if case["land"]:
            H, W = case["height"], case["width"]
            z = torch.randn(1, 1, max(2, H // 24), max(2, W // 24), generator=g, device=DEVICE)
            z = F.interpolate(z, size=(H, W), mode="bilinear")[0, 0]
            t["land"] = z > torch.sort(z.flatten()).values[int(0.7 * H * W)]  # blobs over 30 % of the grid
    else:
        p["fc1.weight"] = normal(4 * C, C, std=C ** -0.5)
        p["fc1.bias"] = normal(4 * C, std=0.1)
        p["fc2.weight"] = normal(C, 4 * C, std=(4 * C) ** -0.5)
        p["fc2.bias"] = normal(C, std=0.1)
    t["params"] = p
    return t


def prepare(case, seed):
    t = _inputs(case, seed)
    with torch.device(DEVICE):
        if case["half"] == "mlp":
            module = SequentialMlp(case["channels"], 4 * case["channels"])
        else:
            module = SequentialSwinTransformer(
                layer_idx=1 if case["shift"] else 0, height=case["height"], width=case["width"],
                embedding_dim=case["channels"], window_size=case["window"], num_heads=case["heads"],
                use_attn_mask=case["mask"], use_relative_position_bias=case["bias"], land_mask=t.get("land"),
                pad=(0, case["pad_bottom"], 0, case["pad_right"]), win_rows=case["win_rows"] or None,
                valid_windows=(case["valid_begin"], case["valid_end"]) if case["valid_end"] else None)
    module = module.to(DEVICE).to(_dtype(case["params"]))
    with torch.no_grad():
        for name, p in module.named_parameters():
            p.copy_(t["params"][name])
    state = dict(module=module, x=t["x"], autocast=_autocast(case), train=case["train"])
    if case["train"]:
        state["x"].requires_grad_(True)
        state["dy"] = t["dy"]
    return state


def _gradients(half, get):
    """The gradients in a fixed order.  The three q, k, v bias gradients are one tensor: the softmax does not see a
    constant added to every key, so the k bias has a gradient of zero, which rounding alone would be judged by."""
    if half == "mlp":
        names = ["norm2.weight", "norm2.bias", "fc1.weight", "fc1.bias", "fc2.weight", "fc2.bias"]
        return {n: get(n) for n in names}
    out = {n: get(n) for n in ["norm1.weight", "norm1.bias", "attn.q_linear.weight", "attn.k_linear.weight",
                               "attn.v_linear.weight", "attn.proj.weight", "attn.proj.bias"]}
    out["attn.qkv.bias"] = torch.cat([get(f"attn.{n}_linear.bias") for n in "qkv"])
    table = get("attn.relative_position_bias_table")
    if table is not None:
        out["attn.relative_position_bias_table"] = table
    return out


def run(state):
    module, x = state["module"], state["x"]
    amp = torch.amp.autocast("cuda", dtype=torch.bfloat16) if state["autocast"] else contextlib.nullcontext()
    if not state["train"]:
        with torch.no_grad(), amp:
            return module(x)
    module.zero_grad(set_to_none=True)
    x.grad = None
    with amp:
        y = module(x)
    y.backward(state["dy"])
    grads = {n: p.grad for n, p in module.named_parameters()}
    half = "mlp" if isinstance(module, SequentialMlp) else "attention"
    return {"y": y.detach(), "dx": x.grad, **_gradients(half, grads.get)}


def _window_tokens(case):
    """Tokens of the windows that are computed (a slab's pad windows left out)."""
    H, W, ws = case["height"] + case["pad_bottom"], case["width"] + case["pad_right"], case["window"]
    if case["valid_end"]:
        return case["batch"] * (case["valid_end"] - case["valid_begin"]) * ws * ws
    return case["batch"] * (case["win_rows"] or H // ws) * ws * W


def work(case):
    C, tokens = case["channels"], case["batch"] * _rows(case)
    elt = 4 if case["x"] == "fp32" else 2
    weight_elt = 4 if case["params"] == "fp32" else 2
    if case["half"] == "mlp":
        weights, flops = 8 * C * C, 16 * C * C * tokens
    else:
        weights = 4 * C * C
        t = _window_tokens(case)
        flops = 8 * C * C * t + 4 * case["window"] ** 2 * C * t
    passes = 2 if case["train"] else 1  # x -> y, and dy -> dx and the weight gradients
    return {"bytes": passes * (2 * tokens * C * elt + weights * weight_elt), "flops": flops * (3 if case["train"] else 1)}


def tolerance(case):
    # Measured against 64 bits, times about four (the order of long fp32 sums differs between implementations).
    # fp32 throughout: 1e-7 (forward) to 1.1e-6 (weight gradients of 3136 tokens), growing with the tokens summed.
    if case["channels"] == 96:
        return {"rel": 1e-5}
    # bf16 operands and results, fp32 sums: forward 0.0018 to 0.0029, ...
    if not case["train"]:
        return {"rel": 1.2e-2, "max": 0.1}
    # ... gradients of the MLP half up to 0.0046, of the attention half (q and k weights) up to 0.0067.
    return {"rel": 1.8e-2 if case["half"] == "mlp" else 2.7e-2}


def _exact_attention(case, t, p, x):
    C, nh, ws = case["channels"], case["heads"], case["window"]
    B, H, W = case["batch"], case["height"], case["width"]
    s = ws // 2 if case["shift"] else 0
    Hp, Wp = H + case["pad_bottom"], W + case["pad_right"]
    n = ws * ws
    rows, cols = case["win_rows"] or Hp // ws, Wp // ws

    def cut(grid):  # [B, Hp, Wp, c] -> [B, emitted windows, n, c]
        w = grid.view(grid.shape[0], Hp // ws, ws, cols, ws, -1).permute(0, 1, 3, 2, 4, 5)
        return w[:, :rows].reshape(grid.shape[0], rows * cols, n, -1)

    live = torch.ones(rows * cols, dtype=torch.bool, device=x.device)
    if case["valid_end"]:
        live[:] = False
        live[case["valid_begin"]:case["valid_end"]] = True
    z = F.layer_norm(x, (C,), p["norm1.weight"], p["norm1.bias"]).view(B, H, W, C)
    z = torch.roll(F.pad(z, (0, 0, 0, case["pad_right"], 0, case["pad_bottom"])), (-s, -s), (1, 2))
    win = cut(z)[:, live].reshape(-1, n, C)
    split = lambda a: a.view(-1, n, nh, C // nh).transpose(1, 2).contiguous()  # noqa: E731
    q, k, v = (split(F.linear(win, p[f"attn.{m}_linear.weight"], p[f"attn.{m}_linear.bias"])) for m in "qkv")
    logits = (q * (C // nh) ** -0.5) @ k.transpose(-2, -1).contiguous()
    if case["bias"]:
        i = torch.arange(n, device=x.device)
        dh, dw = i[:, None] // ws - i // ws + ws - 1, i[:, None] % ws - i % ws + ws - 1
        logits = logits + p["attn.relative_position_bias_table"][dh * (2 * ws - 1) + dw].permute(2, 0, 1)
    extra = torch.zeros(int(live.sum()), n, n, dtype=torch.float64, device=x.device)
    if s and case["mask"]:
        part = lambda m: ((torch.arange(m, device=x.device) >= m - ws).long()  # noqa: E731
                          + (torch.arange(m, device=x.device) >= m - s).long())
        region = cut((3 * part(Hp)[:, None] + part(Wp)).view(1, Hp, Wp, 1))[0, live, :, 0]
        extra = torch.where(region[:, :, None] != region[:, None, :], extra - 100.0, extra)
    if "land" in t:
        land = F.pad(t["land"].double(), (0, case["pad_right"], 0, case["pad_bottom"]))
        land = cut(torch.roll(land, (-s, -s), (0, 1)).view(1, Hp, Wp, 1))[0, live, :, 0]
        extra = extra - 100.0 * land[:, None, :]
    if (s and case["mask"]) or "land" in t:
        logits = (logits.view(B, -1, nh, n, n) + extra[:, None]).view(-1, nh, n, n)
    o = (torch.softmax(logits, -1) @ v).transpose(1, 2).reshape(-1, n, C)
    o = F.linear(o, p["attn.proj.weight"], p["attn.proj.bias"])
    full = torch.zeros(B, (Hp // ws) * cols, n, C, dtype=torch.float64, device=x.device)
    index = torch.nonzero(live)[:, 0]
    full = full.index_copy(1, index, o.view(B, -1, n, C))
    grid = full.view(B, Hp // ws, cols, ws, ws, C).permute(0, 1, 3, 2, 4, 5).reshape(B, Hp, Wp, C)
    grid = torch.roll(grid, (s, s), (1, 2))[:, :H, :W]
    return x + grid.reshape(B, H * W, C)


def _exact_mlp(p, x):
    z = F.layer_norm(x, (x.shape[-1],), p["norm2.weight"], p["norm2.bias"])
    return x + F.linear(F.gelu(F.linear(z, p["fc1.weight"], p["fc1.bias"])), p["fc2.weight"], p["fc2.bias"])


def exact(case, seed):
    t = _inputs(case, seed)
    p = {n: v.double().requires_grad_(case["train"]) for n, v in t["params"].items()}
    x = t["x"].double().requires_grad_(case["train"])
    with contextlib.nullcontext() if case["train"] else torch.no_grad():
        y = _exact_mlp(p, x) if case["half"] == "mlp" else _exact_attention(case, t, p, x)
    if not case["train"]:
        return y
    names = list(p)
    grads = torch.autograd.grad(y, [x] + [p[n] for n in names], t["dy"].double())
    by_name = dict(zip(names, grads[1:]))
    return {"y": y.detach(), "dx": grads[0], **_gradients(case["half"], by_name.get)}
