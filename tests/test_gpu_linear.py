"""GPU parity of the token-row linear kernels (terra_swin_linear,
terra_swin_linear_residual): the GEMM against a float64 CPU product of the
same bf16 operands, and the epilogues (GELU, residual add, the scatter back to
the grid) bit-exact where the GEMM is exact (an identity weight)."""
import pytest
import torch

from oracle import swin_oracle as so
from terra_amd import _lib as L
from terra_amd import kernels, workloads
from terra_amd.kernels import WindowGeometry

pytestmark = pytest.mark.gpu


def _weights(n, k, seed, scale=0.03):
    w = (workloads.activations((n, k), seed) * scale).to(torch.bfloat16)
    b = workloads.activations((n,), seed + 1) * 0.1
    return w, b


def _ref_linear(x, w, b):
    """float64 x W^T + b of the bf16 operands (the fp32-bias module's sum)."""
    return x.double() @ w.double().t() + b.double()


def _assert_bf16_close(got, want64, what):
    """got (bf16) against the exact sum rounded to bf16: fp32 accumulation in
    another order may land one bf16 step away, nothing more."""
    got = got.double().cpu()
    want = want64.float().bfloat16().double()
    step = want.abs().clamp_min(2.0 ** -30) * 2.0 ** -7  # one bf16 ulp or less
    bad = (got - want).abs() > step + 1e-6
    assert bad.float().mean().item() < 1e-3, f"{what}: {int(bad.sum())} of {bad.numel()} values off by more than 1 ulp"
    rel = ((got - want64).norm() / want64.norm()).item()
    assert rel < 4e-3, f"{what}: normwise error {rel:.2e}"


@pytest.mark.parametrize("rows,k,n", [(512, 64, 256), (700, 1024, 1024), (300, 1024, 4096), (256, 4096, 1024),
                                      (1, 64, 256)])
def test_linear_store_against_float64(dev, rows, k, n):
    x = workloads.activations((rows, k), 11).to(torch.bfloat16)
    w, b = _weights(n, k, 12)
    got = kernels.linear(x.to(dev), kernels.pack_linear(w.to(dev)), n, b.to(dev))
    torch.cuda.synchronize()
    _assert_bf16_close(got, _ref_linear(x, w, b), f"linear {rows}x{k}->{n}")


def test_linear_without_bias_and_strided_rows_of_a_batch(dev):
    x = workloads.activations((3, 100, 256), 13).to(torch.bfloat16)
    w, _ = _weights(512, 256, 14)
    got = kernels.linear(x.to(dev), kernels.pack_linear(w.to(dev)), 512)
    assert got.shape == (3, 100, 512)
    _assert_bf16_close(got.reshape(-1, 512), x.reshape(-1, 256).double() @ w.double().t(), "no bias")


def _special_inputs(rows, n):
    """bf16 pre-activations covering the GELU table and its closed forms."""
    x = workloads.activations((rows, n), 15) * 3.0
    # (no inf / nan: the identity GEMM multiplies them by the zeros of W)
    specials = torch.tensor([0.0, -0.0, 2.0 ** -30, -(2.0 ** -30), 2.0 ** -22, -(2.0 ** -22), 31.875, -31.875, 32.0,
                             -32.0, 100.0, -100.0, 3e4, -3e4, 1e-3, -1e-3, 5.5, -5.5])
    x.view(-1)[: specials.numel()] = specials
    x.view(-1)[-specials.numel():] = specials
    return x.to(torch.bfloat16)


def test_linear_gelu_bit_exact_with_identity_weight(dev):
    """W = I and a bf16 bias keep the sum exact (x + b in fp32, one rounding),
    so the output must equal nn.GELU of that bf16 tensor bit for bit,
    including the closed forms outside the table (|x| < 2^-22, |x| >= 32)."""
    rows, n = 300, 256
    x = _special_inputs(rows, n)
    b = (workloads.activations((n,), 16) * 0.5).to(torch.bfloat16).float()
    b[:32] = 0.0  # the special values of the first and last rows stay as they are
    b[-32:] = 0.0
    eye = torch.eye(n, dtype=torch.bfloat16)
    got = kernels.linear(x.to(dev), kernels.pack_linear(eye.to(dev)), n, b.to(dev), gelu=True)
    pre = (x.float() + b).bfloat16()
    want = torch.nn.functional.gelu(pre.to(dev))  # the module's op on the same bf16 tensor
    torch.cuda.synchronize()
    assert torch.equal(got.isnan(), want.isnan())
    ok = ~want.isnan()
    assert torch.equal(got[ok], want[ok])


@pytest.mark.parametrize("rows,k,n", [(513, 1024, 4096), (256, 256, 512)])
def test_linear_gelu_against_float64(dev, rows, k, n):
    x = workloads.activations((rows, k), 17).to(torch.bfloat16)
    w, b = _weights(n, k, 18, scale=0.06)
    got = kernels.linear(x.to(dev), kernels.pack_linear(w.to(dev)), n, b.to(dev), gelu=True).double().cpu()
    pre = _ref_linear(x, w, b).float().bfloat16().double()
    want = 0.5 * pre * (1.0 + torch.special.erf(pre / 2.0 ** 0.5))
    # the pre-activation may sit one bf16 step away (summation order); GELU's slope is below 1.13
    err = (got - want).abs()
    assert (err <= pre.abs() * 2.0 ** -7 * 1.2 + want.abs() * 2.0 ** -8 + 1e-6).float().mean().item() > 0.999
    assert ((got - want).norm() / want.norm()).item() < 4e-3


def test_linear_residual_bit_exact_with_identity_weight(dev):
    rows, n = 777, 512
    x = workloads.activations((rows, n), 19).to(torch.bfloat16)
    r = workloads.activations((rows, n), 20).to(torch.bfloat16)
    b = (workloads.activations((n,), 21) * 0.25).to(torch.bfloat16).float()
    eye = torch.eye(n, dtype=torch.bfloat16)
    got = kernels.linear_residual(x.to(dev), kernels.pack_linear(eye.to(dev)), n, r.to(dev), b.to(dev)).cpu()
    want = r + (x.float() + b).bfloat16()  # bf16 + bf16: fp32 sum, one rounding
    assert torch.equal(got, want)


def test_linear_residual_in_place_against_float64(dev):
    rows, k, n = 600, 4096, 1024
    x = workloads.activations((rows, k), 22).to(torch.bfloat16)
    r = workloads.activations((rows, n), 23).to(torch.bfloat16)
    w, b = _weights(n, k, 24, scale=0.01)
    rd = r.to(dev)
    got = kernels.linear_residual(x.to(dev), kernels.pack_linear(w.to(dev)), n, rd, b.to(dev), out=rd)
    assert got.data_ptr() == rd.data_ptr()
    y = _ref_linear(x, w, b).float().bfloat16().double()
    want = r.double() + y
    got = got.double().cpu()
    assert ((got - want).norm() / want.norm()).item() < 4e-3
    assert ((got - want).abs() <= want.abs() * 2.0 ** -7 + y.abs() * 2.0 ** -7 + 1e-6).float().mean().item() > 0.999


SCATTER_CASES = [  # (B, H, W, shift, pad): every window of the padded frame emitted
    (2, 16, 24, 4, (0, 0, 0, 0)),
    (1, 20, 36, 4, (0, 4, 0, 4)),
    (2, 13, 21, 0, (1, 2, 0, 3)),
    (1, 24, 40, 3, (0, 0, 0, 0)),
]


@pytest.mark.parametrize("case", SCATTER_CASES)
def test_linear_scatter_bit_exact_with_identity_weight(dev, case):
    """W = I: y must be the oracle's window reverse (+ roll, crop) plus the
    residual, bit for bit: the row map of the epilogue is the partition's."""
    B, H, W, s, pad = case
    C = 256
    geom = WindowGeometry(B, H, W, C, 8, s, s, pad)
    win = workloads.activations((geom.num_windows, 64, C), 25).to(torch.bfloat16)
    r = workloads.activations((B, H, W, C), 26).to(torch.bfloat16)
    eye = torch.eye(C, dtype=torch.bfloat16)
    got = kernels.linear_residual(win.to(dev), kernels.pack_linear(eye.to(dev)), C, r.to(dev), None, geom=geom).cpu()
    want = so.reverse_frame(win, B, H, W, 8, s, s, pad, residual=r)
    assert torch.equal(got, want)


SCATTER_ANY_CASES = [  # (B, H, W, window, shift, pad)
    (2, 64, 96, 32, 16, (0, 0, 0, 0)),
    (3, 14, 21, 7, 3, (0, 0, 0, 0)),
    (2, 13, 19, 7, 0, (1, 0, 0, 2)),
    (1, 30, 50, 16, 5, (1, 1, 7, 7)),
    (2, 5, 9, 1, 0, (0, 0, 0, 0)),
    (1, 3, 3, 3, 1, (0, 0, 0, 0)),
    (2, 16, 24, 8, 4, (0, 0, 0, 0)),
]


@pytest.mark.parametrize("case", SCATTER_ANY_CASES)
def test_linear_scatter_any_window_bit_exact_with_identity_weight(dev, case):
    """As above for windows of other sizes (terra_swin_linear_scatter)."""
    B, H, W, ws, s, pad = case
    C = 256
    geom = WindowGeometry(B, H, W, C, ws, s, s, pad)
    win = workloads.activations((geom.num_windows, ws * ws, C), 35).to(torch.bfloat16)
    r = workloads.activations((B, H, W, C), 36).to(torch.bfloat16)
    wd = kernels.pack_linear(torch.eye(C, dtype=torch.bfloat16).to(dev))
    got = kernels.linear_scatter(win.to(dev), wd, C, r.to(dev), geom)
    assert torch.equal(got.cpu(), so.reverse_frame(win, B, H, W, ws, s, s, pad, residual=r))
    if ws != 8:  # the other entry keeps refusing these windows
        with pytest.raises((ValueError, RuntimeError, NotImplementedError), match="8x8"):
            kernels.linear_residual(win.to(dev), wd, C, r.to(dev), geom=geom)


def test_block_window32_takes_the_scatter_launch(dev, monkeypatch):
    """A window-32 block whose rows fill the chip projects, reverses and adds the
    residual in one launch; the staged order gives the same to bf16 rounding."""
    from terra_amd.transformer import SequentialSwinTransformer
    blk = SequentialSwinTransformer(layer_idx=1, height=256, width=128, embedding_dim=512, window_size=32, num_heads=4,
                                    use_attn_mask=False, use_relative_position_bias=False)
    workloads.init_block_params(blk, 1)
    blk = blk.to(dev, torch.bfloat16)
    x = workloads.activations((1, 256 * 128, 512), 37).to(dev, torch.bfloat16)
    calls = []
    real = kernels.linear_scatter
    monkeypatch.setattr(kernels, "linear_scatter", lambda *a, **k: calls.append(1) or real(*a, **k))
    with torch.no_grad():
        y = blk(x)
        assert calls == [1]
        monkeypatch.setattr(kernels, "linear_fills", lambda *a: False)
        want = blk(x)
        assert calls == [1]
    # Two bf16 roundings (the product, the sum) on either side.
    assert ((y - x).float() - (want - x).float()).norm() <= 2.0 ** -7 * (want - x).float().norm()


@pytest.mark.parametrize("shape", [(1, 32, 48), (1, 288, 544)], ids=["small", "g1-grid"])
def test_linear_scatter_matches_proj_then_reverse(dev, shape):
    """proj + reverse + residual in one kernel against the five-stage order
    (torch's bf16 Linear, then the reverse kernel), C = 1024."""
    B, H, W = shape
    C = 1024
    geom = WindowGeometry(B, H, W, C, 8, 4, 4)
    o = workloads.activations((geom.num_windows, 64, C), 27).to(torch.bfloat16).to(dev)
    x = workloads.activations((B, H, W, C), 28).to(torch.bfloat16).to(dev)
    w, b = _weights(C, C, 29, scale=0.02)
    wd, bd = w.to(dev), b.to(dev)
    got = kernels.linear_residual(o, kernels.pack_linear(wd), C, x, bd, geom=geom)
    proj = torch.nn.functional.linear(o, wd, bd.to(torch.bfloat16))
    want = kernels.swin_reverse(proj.contiguous(), geom, residual=x)
    torch.cuda.synchronize()
    d = (got.float() - want.float())
    assert torch.isfinite(got.float()).all()
    assert (d.norm() / want.float().norm()).item() < 4e-3
    y = (want.float() - x.float())
    assert ((got.float() - x.float() - y).norm() / y.norm()).item() < 2e-2


@pytest.mark.parametrize("k", [64, 128, 192, 320])
def test_linear_many_tiles_per_workgroup(dev, k):
    """1028 tiles over 256 workgroups: the load stream runs across tile
    boundaries with 1, 2, 3 and 5 stages per tile (odd counts swap the token
    fragment registers), past output stores still in flight, into a last tile
    of 77 rows; against the same rows computed as one small call each."""
    rows, n = 256 * 513 + 77, 512
    x = torch.randn(rows, k, device=dev, dtype=torch.bfloat16, generator=torch.Generator(dev).manual_seed(30))
    w, b = _weights(n, k, 31)
    pk, bd = kernels.pack_linear(w.to(dev)), b.to(dev)
    got = kernels.linear(x, pk, n, bd)
    ref = x.double() @ w.to(dev).double().t() + bd.double()
    # one fp32 sum of k products in another order: within a bf16 step of the exact sum's rounding
    assert ((got.double() - ref).abs() <= ref.abs() * 2.0 ** -7 + 1e-5).all()
    for r0 in (0, 256 * 255, rows - 333):
        assert torch.equal(got[r0:r0 + 333], kernels.linear(x[r0:r0 + 333].contiguous(), pk, n, bd))
    r = torch.randn(rows, n, device=dev, dtype=torch.bfloat16, generator=torch.Generator(dev).manual_seed(32))
    assert torch.equal(kernels.linear_residual(x, pk, n, r, bd), r + got)


def test_linear_row_stride_past_the_descriptor(dev):
    """A 16.8 MB output row stride: 256 rows span more than a buffer
    descriptor, so the 64-bit store form runs; the same values as contiguous."""
    rows, k, n, stride = 300, 64, 256, (1 << 23) + 8
    x = workloads.activations((rows, k), 33).to(torch.bfloat16).to(dev)
    w, b = _weights(n, k, 34)
    pk, bd = kernels.pack_linear(w.to(dev)), b.to(dev)
    y = torch.empty((rows - 1) * stride + n, dtype=torch.bfloat16, device=dev)
    for gelu in (0, 1):
        st = L.load().terra_swin_linear(x.data_ptr(), y.data_ptr(), L.DTYPE_BF16, rows, k, n, k, stride,
                                        pk.data_ptr(), bd.data_ptr(), gelu, None)
        torch.cuda.synchronize()
        assert st == 0, L.last_error()
        assert torch.equal(y.as_strided((rows, n), (stride, 1)), kernels.linear(x, pk, n, bd, gelu=bool(gelu)))


def test_linear_scatter_grid_past_the_descriptor(dev):
    """A grid of 4.3 GB (2904 x 2904 tokens of 256 channels): the 64-bit
    addresses of the scatter, bit for bit the reverse kernel's (W = I)."""
    H = W = 2904
    C = 256
    geom = WindowGeometry(1, H, W, C, 8, 4, 4)
    g = torch.Generator(dev).manual_seed(35)
    win = torch.randn(geom.num_windows, 64, C, device=dev, dtype=torch.bfloat16, generator=g)
    r = torch.randn(1, H, W, C, device=dev, dtype=torch.bfloat16, generator=g)
    eye = torch.eye(C, dtype=torch.bfloat16, device=dev)
    got = kernels.linear_residual(win, kernels.pack_linear(eye), C, r, None, geom=geom)
    assert torch.equal(got, kernels.swin_reverse(win, geom, residual=r))


def test_linear_empty_rows(dev):
    x = torch.empty(0, 256, dtype=torch.bfloat16, device=dev)
    w = kernels.pack_linear(torch.zeros(256, 256, dtype=torch.bfloat16, device=dev))
    assert kernels.linear(x, w, 256).shape == (0, 256)
    assert kernels.linear_residual(x, w, 256, torch.empty(0, 256, dtype=torch.bfloat16, device=dev)).shape == (0, 256)


# (rows, in, out): one row, a tail row, whole tiles, feature blocks of 192 and
# 128, one and several blocks, more tiles than resident workgroups.
SHORT_SHAPES = [(1, 192, 192), (64, 128, 128), (65, 192, 128), (300, 128, 192), (500, 128, 512), (777, 192, 1024),
                (70001, 192, 576), (120000, 128, 384), (90000, 192, 768)]


@pytest.mark.parametrize("rows,k,n", SHORT_SHAPES)
def test_linear_short(dev, rows, k, n):
    """The short-row linear kernel against float64 (one fp32 sum of k products
    and its bf16 rounding), with and without bias, and its GELU pair: h the
    same bits, y torch's GELU of h; memory past the outputs untouched."""
    x = torch.randn(rows, k, device=dev, generator=torch.Generator(dev).manual_seed(40)).bfloat16()
    w, b = _weights(n, k, 41, scale=k ** -0.5)
    pk, bd = kernels.pack_linear(w.to(dev)), b.to(dev)
    y = kernels.linear_short(x, pk, n, bd)
    ref = x.double() @ w.to(dev).double().t()
    mag = x.double().abs() @ w.to(dev).double().abs().t() + bd.double().abs()
    assert ((y.double() - ref - bd.double()).abs() <= (ref + bd.double()).abs() * 2.0 ** -8 + mag * k * 2.0 ** -24).all()
    assert ((kernels.linear_short(x, pk, n).double() - ref).abs() <= ref.abs() * 2.0 ** -8 + mag * k * 2.0 ** -24).all()
    h, a = kernels.linear_short(x, pk, n, bd, gelu_keep=True)
    assert torch.equal(h, y) and torch.equal(a, torch.nn.functional.gelu(h))
    guard = torch.full((rows * n + 4096,), 7.0, device=dev, dtype=torch.bfloat16)
    st = L.load().terra_swin_linear_short(x.data_ptr(), guard.data_ptr(), None, L.DTYPE_BF16, rows, k, n, pk.data_ptr(),
                                          bd.data_ptr(), 0, None)
    torch.cuda.synchronize()
    assert st == 0 and torch.equal(guard[:rows * n].view(rows, n), y) and bool((guard[rows * n:] == 7.0).all())


@pytest.mark.parametrize("C,tokens,amp", [(256, 65300, False), (1024, 16385, True), (256, 4097, False)])
def test_mlp_inference_fc2_on_the_residual_epilogue(dev, C, tokens, amp, monkeypatch):
    """SequentialMlp at widths the one-kernel MLP does not take: fc2 + residual
    run on the linear kernel where the rows fill the chip, with the library's
    result to the bf16 roundings of the product and of the sum."""
    from terra_amd.mlp import SequentialMlp
    torch.manual_seed(9)
    m = SequentialMlp(C, 4 * C).to(dev, torch.float32 if amp else torch.bfloat16)
    x = workloads.activations((1, tokens, C), 38).to(dev, torch.bfloat16)
    calls = []
    real, fills = kernels.linear_residual, kernels.linear_fills(tokens, C)
    monkeypatch.setattr(kernels, "linear_residual", lambda *a, **k: calls.append(1) or real(*a, **k))
    with torch.no_grad(), torch.amp.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
        y = m(x)
        assert len(calls) == int(fills)
        monkeypatch.setattr(kernels, "linear_fills", lambda *a: False)
        want = m(x)
    assert y.dtype == want.dtype
    assert (y.float() - want.float()).norm() <= 2.0 ** -7 * want.float().norm()


def test_window32_block_adds_the_bias_that_f_linear_adds(dev, monkeypatch):
    """fp32 parameters under bf16 autocast: F.linear rounds proj's bias to bf16.
    The scatter launch gives the staged path's result but for the order of the
    fp32 sums, which moves a product of 512 terms across a bf16 rounding for
    about one value in a thousand; an unrounded bias moves one in ten."""
    from terra_amd.transformer import SequentialSwinTransformer
    blk = SequentialSwinTransformer(layer_idx=1, height=256, width=128, embedding_dim=512, window_size=32, num_heads=4,
                                    use_attn_mask=False, use_relative_position_bias=False)
    workloads.init_block_params(blk, 1)
    blk.attn.proj.bias.data.copy_(workloads.activations((512,), 39))
    blk = blk.to(dev)
    x = workloads.activations((1, 256 * 128, 512), 37).to(dev, torch.bfloat16)
    calls = []
    real = kernels.linear_scatter
    monkeypatch.setattr(kernels, "linear_scatter", lambda *a, **k: calls.append(1) or real(*a, **k))
    with torch.no_grad(), torch.amp.autocast("cuda", dtype=torch.bfloat16):
        y = blk(x)
        monkeypatch.setattr(kernels, "linear_fills", lambda *a: False)
        want = blk(x)
    assert calls == [1] and (y != want).float().mean() <= 0.01


@pytest.mark.parametrize("C,tokens", [(256, 65300), (1024, 16385)])
def test_mlp_fc2_adds_the_bias_that_f_linear_adds(dev, C, tokens, monkeypatch):
    """As above for fc2 + residual in SequentialMlp."""
    from terra_amd.mlp import SequentialMlp
    torch.manual_seed(10)
    m = SequentialMlp(C, 4 * C).to(dev)
    m.fc2.bias.data.copy_(workloads.activations((C,), 39))
    x = workloads.activations((1, tokens, C), 38).to(dev, torch.bfloat16)
    with torch.no_grad(), torch.amp.autocast("cuda", dtype=torch.bfloat16):
        y = m(x)
        monkeypatch.setattr(kernels, "linear_fills", lambda *a: False)
        want = m(x)
    assert (y != want).float().mean() <= 0.01


@pytest.mark.parametrize("C,tokens,launches", [(1024, 16896, 0), (1024, 24576, 1), (512, 33000, 0), (256, 66000, 0),
                                               (256, 73728, 1)])
def test_mlp_inference_takes_the_residual_launch_where_it_pays(dev, C, tokens, launches, monkeypatch):
    from terra_amd.mlp import SequentialMlp
    m = SequentialMlp(C, 4 * C).to(dev, torch.bfloat16)
    calls = []
    real = kernels.linear_residual
    monkeypatch.setattr(kernels, "linear_residual", lambda *a, **k: calls.append(1) or real(*a, **k))
    with torch.no_grad():
        m(torch.randn(1, tokens, C, device=dev, dtype=torch.bfloat16))
    assert len(calls) == launches
