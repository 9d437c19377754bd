"""GPU: fused residual add + RMSNorm and SiLU-gated product vs torch.

Bars: the residual sum x + delta is bit-exact with torch's bf16 add; the
normalised output is within one bf16 rounding of an fp32 evaluation of
rms_norm(x + delta) * w (and of torch's F.rms_norm); SiLU * up is within one
bf16 ulp of torch's F.silu(g) * u.  The model's prefill logits with the fused
kernels agree with the unfused torch ops (relative 2e-2).
"""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _ulp_close(a: torch.Tensor, b: torch.Tensor, ulps: int = 1) -> bool:
    """|a - b| <= ulps bf16 ulps of max(|a|, |b|) elementwise (bf16 inputs)."""
    a32, b32 = a.float(), b.float()
    mag = torch.maximum(a32.abs(), b32.abs())
    ulp = torch.where(mag > 0, torch.pow(2.0, torch.floor(torch.log2(mag)) - 7), torch.zeros_like(mag))
    return bool(((a32 - b32).abs() <= ulps * ulp + 1e-30).all())


@pytest.mark.parametrize("hidden", [896, 3584, 4096, 8192])
@pytest.mark.parametrize("rows", [1, 5, 32, 300])
def test_add_rms_norm(dev, hidden, rows):
    from minimal_inference_amd.dense import add_rms_norm

    g = torch.Generator(device=dev).manual_seed(hidden + rows)
    x = torch.randn(rows, hidden, device=dev, generator=g).to(torch.bfloat16)
    d = (torch.randn(rows, hidden, device=dev, generator=g) * 0.5).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(hidden, device=dev, generator=g)).to(torch.bfloat16)
    want_x = x + d
    x_run = x.clone()
    h = add_rms_norm(x_run, d, w, 1e-6)
    torch.cuda.synchronize()
    assert torch.equal(x_run, want_x)
    xf = want_x.float()
    ref = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6) * w.float()
    assert _ulp_close(h, ref.to(torch.bfloat16), 1)
    assert _ulp_close(h, F.rms_norm(want_x, (hidden,), w, 1e-6), 2)


def test_add_rms_norm_modes(dev):
    """No delta (norm only, x untouched); sum only (no norm); strided rows."""
    from minimal_inference_amd.dense import add_rms_norm

    x = torch.randn(7, 1024, device=dev).to(torch.bfloat16)
    w = torch.ones(1024, device=dev, dtype=torch.bfloat16)
    x0 = x.clone()
    h = add_rms_norm(x, None, w, 1e-5, write_x=False)
    torch.cuda.synchronize()
    assert torch.equal(x, x0)
    xf = x.float()
    assert _ulp_close(h, (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-5)).to(torch.bfloat16))
    d = torch.randn(7, 1024, device=dev).to(torch.bfloat16)
    assert add_rms_norm(x, d, w, 1e-5, norm=False) is None
    torch.cuda.synchronize()
    assert torch.equal(x, x0 + d)
    big = torch.randn(7, 2048, device=dev).to(torch.bfloat16)
    xv = big[:, 512:1536]                               # row stride 2048
    want = xv + d
    hv = add_rms_norm(xv, d, w, 1e-5)
    torch.cuda.synchronize()
    assert torch.equal(big[:, 512:1536], want)
    wf = want.float()
    assert _ulp_close(hv, (wf * torch.rsqrt(wf.pow(2).mean(-1, keepdim=True) + 1e-5)).to(torch.bfloat16))


@pytest.mark.parametrize("rows,inter", [(1, 4864), (32, 14336), (300, 18944), (5, 29568)])
def test_silu_mul(dev, rows, inter):
    from minimal_inference_amd.dense import silu_mul

    gu = (torch.randn(rows, 2 * inter, device=dev) * 3).to(torch.bfloat16)
    got = silu_mul(gu)
    g, u = gu.chunk(2, dim=-1)
    want = F.silu(g) * u
    torch.cuda.synchronize()
    assert got.shape == (rows, inter)
    assert _ulp_close(got, want, 1)
    assert (got == want).float().mean().item() > 0.99


def test_rejects_bad_shapes(dev):
    from minimal_inference_amd.dense import add_rms_norm, silu_mul

    with pytest.raises(ValueError):
        add_rms_norm(torch.zeros(2, 12, device=dev, dtype=torch.bfloat16), None,
                     torch.ones(12, device=dev, dtype=torch.bfloat16), 1e-6)     # hidden % 8
    with pytest.raises(ValueError):
        silu_mul(torch.zeros(2, 10, device=dev, dtype=torch.bfloat16))          # intermediate % 8
    with pytest.raises(ValueError):
        add_rms_norm(torch.zeros(2, 16, device=dev, dtype=torch.float32), None,
                     torch.ones(16, device=dev, dtype=torch.bfloat16), 1e-6)     # dtype


def test_model_prefill_logits_fused_vs_unfused(dev):
    from minimal_inference_amd.engine import Request, Scheduler
    from minimal_inference_amd.model import PRESETS, Model

    cfg = PRESETS["qwen2.5-0.5b"]
    cfg = type(cfg)(**{**cfg.__dict__, "num_hidden_layers": 6})
    logits = []
    for fused in (True, False):
        model = Model(cfg, dev, seed=5, max_positions=512, fused_dense=fused)
        sch = Scheduler(model, max_batch_size=4, max_seq_len=256, use_graphs=False)
        g = torch.Generator().manual_seed(9)
        for i, n in enumerate([12, 77, 200]):
            sch.submit(Request(str(i), torch.randint(0, cfg.vocab_size, (n,), generator=g).tolist(), 1, 0.0))
        captured = {}
        orig = model.forward

        def spy(*a, **k):
            captured["l"] = orig(*a, **k)
            return captured["l"]

        model.forward = spy
        sch._prefill(sch._admit())
        logits.append(captured["l"].float())
    rel = (logits[0] - logits[1]).abs().max().item() / logits[1].abs().max().item()
    assert rel < 2e-2, rel


@pytest.mark.parametrize("rows", [1, 8, 15, 16, 17, 32])
@pytest.mark.parametrize("n,k", [
    (16, 64), (48, 192), (1152, 896), (896, 4864), (4096, 320),   # one tile per workgroup, few slabs, odd slab counts
    (4112, 4096), (8176, 128), (8208, 576),                       # either side of 256 and 512 tiles of 16 columns
    (32768, 256), (32800, 256), (151936, 896),                    # 2,048 tiles, past them with a partial last workgroup
    (512, 8192), (16, 18944),                                     # long rows
    (2048, 1984), (2048, 2048), (2064, 2048),                     # either side of half tiles
])
def test_few_row_linear(dev, rows, n, k):
    """mi_linear at the edges of its forms against an fp32 product of the same
    bf16 values; x rows and out rows strided, and the columns and rows around
    them untouched.

    Bound: rounding errors of a sum of k products in fp32 are independent enough to
    stay within 4 sqrt(k) 2^-24 sum |x w| of the exact one (the worst case, k in the
    place of 4 sqrt(k), is 27 at k = 18,944 and would hide a lost slab of 64 k, 8),
    and the result is rounded once to bf16 (2^-8 relative); the reference's own fp32
    error is of the first kind."""
    from minimal_inference_amd import _lib

    g = torch.Generator(device=dev).manual_seed(rows * 131 + n + k)
    big = torch.randn(rows, k + 64, device=dev, generator=g).to(torch.bfloat16)
    x = big[:, 32:32 + k]
    w = torch.randn(n, k, device=dev, generator=g).to(torch.bfloat16)
    for bias in (None, torch.randn(n, device=dev, generator=g).to(torch.bfloat16)):
        out = torch.full((rows + 1, n + 8), 7.0, device=dev, dtype=torch.bfloat16)
        _lib.call("mi_linear", x.data_ptr(), x.stride(0), w.data_ptr(), bias.data_ptr() if bias is not None else None,
                  out.data_ptr(), out.stride(0), rows, n, k, torch.cuda.current_stream().cuda_stream)
        b = 0.0 if bias is None else bias.float()
        ref = x.float() @ w.float().t() + b
        mag = x.float().abs() @ w.float().abs().t() + (0.0 if bias is None else bias.float().abs())
        err = (out[:rows, :n].float() - ref).abs()
        assert bool((err <= 2 ** -8 * ref.abs() + 2 * 4 * k ** 0.5 * 2 ** -24 * mag).all())
        assert bool((out[rows] == 7.0).all()) and bool((out[:, n:] == 7.0).all())
        again = torch.empty_like(out)
        _lib.call("mi_linear", x.data_ptr(), x.stride(0), w.data_ptr(), bias.data_ptr() if bias is not None else None,
                  again.data_ptr(), again.stride(0), rows, n, k, torch.cuda.current_stream().cuda_stream)
        assert torch.equal(again[:rows, :n], out[:rows, :n])


@pytest.mark.parametrize("rows", [1, 16, 17, 32])
@pytest.mark.parametrize("n,k", [
    (16, 64), (48, 192), (896, 4864), (4096, 320), (4112, 4096), (8192, 576), (8208, 576), (32768, 256), (32784, 320),
    (512, 8192), (16, 18944), (16, 18880), (2048, 1984), (2048, 2112), (4608, 9024),
])
def test_few_row_linear_of_whole_numbers(dev, rows, n, k):
    """Whole numbers up to 8: every sum is exact in fp32 in any order, so the result
    is the exact one's bf16, and a part of k that is lost or taken twice moves it."""
    from minimal_inference_amd import _lib

    g = torch.Generator(device=dev).manual_seed(rows * 131 + n + k)
    x = torch.randint(-8, 9, (rows, k), device=dev, generator=g).to(torch.bfloat16)
    w = torch.randint(-8, 9, (n, k), device=dev, generator=g).to(torch.bfloat16)
    out = torch.empty(rows, n, device=dev, dtype=torch.bfloat16)
    _lib.call("mi_linear", x.data_ptr(), k, w.data_ptr(), None, out.data_ptr(), n, rows, n, k,
              torch.cuda.current_stream().cuda_stream)
    assert 64 * k < 2 ** 24
    assert torch.equal(out, (x.float() @ w.float().t()).to(torch.bfloat16))


def test_few_row_linear_routes(dev):
    """dense.linear: the kernel and torch's F.linear agree to bf16 rounding where
    the kernel takes the call, and the calls it does not take (more rows, odd
    widths, other types and layouts, gradients) are F.linear's, bit for bit."""
    from minimal_inference_amd.dense import linear

    x = torch.randn(8, 512, device=dev).to(torch.bfloat16)
    w = torch.randn(256, 512, device=dev).to(torch.bfloat16)
    b = torch.randn(256, device=dev).to(torch.bfloat16)
    assert _ulp_close(linear(x, w, b), F.linear(x.float(), w.float(), b.float()).to(torch.bfloat16), 1)
    assert linear(x[:0], w).shape == (0, 256)
    for xx, ww in [(x.repeat(5, 1), w), (x[:, :480], w[:, :480]), (x[:, :480], w[:, :480].contiguous()),
                   (x, w[:250]), (x.float(), w.float()), (x.t().contiguous().t(), w)]:
        assert torch.equal(linear(xx, ww), F.linear(xx, ww))
    wg = w.clone().requires_grad_()
    linear(x, wg).float().sum().backward()
    assert wg.grad is not None
    with pytest.raises(ValueError):
        from minimal_inference_amd import _lib
        _lib.call("mi_linear", x.data_ptr(), 512, w.data_ptr(), None, b.data_ptr(), 256, 33, 256, 512, 0)


def test_silu_mul_every_gate(dev):
    """Every bf16 gate (zeros, subnormals, infinities, NaNs and those whose
    exponential is past the end of fp32) times one: the bits of the fp32 formula
    with an IEEE division; and more rows than the grid's second axis has."""
    from minimal_inference_amd.dense import silu_mul

    gate = torch.arange(-32768, 32768, device=dev, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    out = silu_mul(torch.cat([gate, torch.ones_like(gate)])[None])[0]
    ref = (gate.float() / (1 + torch.exp(-gate.float()))).to(torch.bfloat16)
    assert torch.equal(out.isnan(), ref.isnan())
    assert torch.equal(out.nan_to_num(7.0).view(torch.int16), ref.nan_to_num(7.0).view(torch.int16))
    gu = torch.randn(65535 + 70, 48, device=dev, generator=torch.Generator(device=dev).manual_seed(3)).to(torch.bfloat16)
    assert _ulp_close(silu_mul(gu), F.silu(gu[:, :24]) * gu[:, 24:], 1)


@pytest.mark.parametrize("inter,k", [(16, 64), (48, 896), (4096, 128), (4112, 64), (4864, 896), (8208, 64), (14336, 256)])
@pytest.mark.parametrize("rows", [1, 16, 17, 32])
def test_few_row_linear_silu(dev, rows, inter, k):
    """mi_linear_silu at the edges of its forms (one and two blocks of rows, one
    and two pairs of tiles to a workgroup, a last workgroup half empty): the bits
    of the two separate kernels; nothing written around the rows."""
    from minimal_inference_amd import _lib
    from minimal_inference_amd.dense import silu_mul

    g = torch.Generator(device=dev).manual_seed(rows * 131 + inter + k)
    big = torch.randn(rows, k + 64, device=dev, generator=g).to(torch.bfloat16)
    x = big[:, 32:32 + k]
    w = torch.randn(2 * inter, k, device=dev, generator=g).to(torch.bfloat16)
    gu = torch.empty(rows, 2 * inter, device=dev, dtype=torch.bfloat16)
    stream = torch.cuda.current_stream().cuda_stream
    _lib.call("mi_linear", x.data_ptr(), x.stride(0), w.data_ptr(), None, gu.data_ptr(), 2 * inter, rows, 2 * inter, k,
              stream)
    out = torch.full((rows + 1, inter + 8), 7.0, device=dev, dtype=torch.bfloat16)
    _lib.call("mi_linear_silu", x.data_ptr(), x.stride(0), w.data_ptr(), out.data_ptr(), out.stride(0), rows, inter, k,
              stream)
    assert torch.equal(out[:rows, :inter], silu_mul(gu))
    assert bool((out[rows] == 7.0).all()) and bool((out[:, inter:] == 7.0).all())


def test_few_row_linear_silu_routes(dev):
    """dense.linear_silu is silu_mul(linear(..)), bit for bit, where the one launch
    takes the call and where it does not (more rows, narrow halves, strided
    weights), and refuses what silu_mul refuses."""
    from minimal_inference_amd.dense import linear, linear_silu, silu_mul

    x = torch.randn(8, 512, device=dev).to(torch.bfloat16)
    w = torch.randn(256, 512, device=dev).to(torch.bfloat16)
    for xx, ww in [(x, w), (x.repeat(5, 1), w), (x, w[:240]), (x[:, :480], w[:, :480]), (x[:0], w)]:
        assert torch.equal(linear_silu(xx, ww), silu_mul(linear(xx, ww)))
    for xx, ww in [(x, w[:255]), (x.float(), w.float())]:
        with pytest.raises((ValueError, TypeError)):
            linear_silu(xx, ww)


def test_few_row_linear_leaves_what_the_kernel_refuses_to_torch(dev):
    """Rows whose stride spans more than mi_linear's 2^29 elements, and weights of
    no rows, no columns or one axis, are F.linear's."""
    from minimal_inference_amd.dense import _takes, linear

    # (not multiplied: how the library takes rows this far apart is its own matter)
    step, k = (1 << 28) + 8, 512
    far = torch.zeros(step + k, device=dev, dtype=torch.bfloat16)
    x = far.as_strided((2, k), (step, 1))
    w = torch.randn(256, k, device=dev).to(torch.bfloat16)
    assert not _takes(x, w, None) and _takes(far.as_strided((2, k), (step - 8, 1)), w, None)
    x.copy_(torch.randn(2, k, device=dev))
    near = x.contiguous()
    assert torch.equal(linear(near, w[:0]), F.linear(near, w[:0]))
    assert torch.equal(linear(near, w[0]), F.linear(near, w[0]))
    for ww in (w[:, :0], torch.empty(256, 0, device=dev, dtype=torch.bfloat16)):
        assert torch.equal(linear(near[:, :0], ww), torch.zeros(2, 256, device=dev, dtype=torch.bfloat16))


def test_few_row_linear_under_torchs_modes(dev):
    """What torch does around F.linear happens around dense.linear too: autocast,
    forward-mode tangents, function transforms, dispatch and function modes and
    tensor subclasses all get F.linear's call."""
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from minimal_inference_amd.dense import _takes, linear

    x = torch.randn(8, 512, device=dev).to(torch.bfloat16)
    w = torch.randn(256, 512, device=dev).to(torch.bfloat16)
    assert _takes(x, w, None)
    with torch.autocast("cuda", dtype=torch.float16):
        assert torch.equal(linear(x, w), F.linear(x, w)) and linear(x, w).dtype == torch.float16
    with forward_ad.dual_level():
        primal, tangent = forward_ad.unpack_dual(linear(x, forward_ad.make_dual(w, torch.ones_like(w))))
        assert torch.equal(primal, F.linear(x, w)) and torch.equal(tangent, F.linear(x, torch.ones_like(w)))

    def rows(xx):  # (the product itself would be a batched one)
        assert not _takes(xx, w, None)
        return xx

    torch.vmap(rows)(x.view(2, 4, 512))

    class Seen(TorchDispatchMode):
        ops = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.ops += 1
            return func(*args, **(kwargs or {}))

    class Called(TorchFunctionMode):
        linears = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.linears += func is F.linear
            return func(*args, **(kwargs or {}))

    class Named(torch.Tensor):
        pass

    with Seen() as seen:
        linear(x, w)
    with Called() as called:
        linear(x, w)
    assert seen.ops >= 1 and called.linears == 1
    assert isinstance(linear(x, w.as_subclass(Named)), Named)
    assert not _takes(x.as_subclass(Named), w, None) and not _takes(x, w, w[:, 0].contiguous().as_subclass(Named))
    assert _takes(x, torch.nn.Parameter(w, requires_grad=False), None)


@pytest.mark.parametrize("rows,inter", [
    *[(rows, inter) for inter in (8, 16, 40, 1000, 2040, 2048, 2056, 2816, 4096, 4104, 4864) for rows in (1, 3, 31, 257)],
    (65535 + 70, 1032), (2 * 65535 + 3, 1024)])
def test_silu_mul_widths(dev, rows, inter):
    """The shapes of a workgroup (many rows, one, half of one, part of one), rows that
    do not fill the last, and more workgroups of rows than the grid's second axis
    has: the bits of the fp32 formula, nothing written around them."""
    from minimal_inference_amd.dense import silu_mul

    g = torch.Generator(device=dev).manual_seed(rows * 131 + inter)
    gu = (3 * torch.randn(rows, 2 * inter, device=dev, generator=g)).to(torch.bfloat16)
    out = torch.full((rows + 1, inter + 8), 7.0, device=dev, dtype=torch.bfloat16)
    silu_mul(gu, out=out[:rows, :inter])
    gate, up = gu[:, :inter].float(), gu[:, inter:].float()
    ref = ((gate / (1 + torch.exp(-gate))).to(torch.bfloat16).float() * up).to(torch.bfloat16)
    assert torch.equal(out[:rows, :inter], ref)
    assert bool((out[rows] == 7.0).all()) and bool((out[:, inter:] == 7.0).all())
