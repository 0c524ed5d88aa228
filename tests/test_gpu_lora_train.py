"""The training form of the NF4 + LoRA linear on the GPU against
float64 torch on the same rounding points: grpo_nf4_dequant_t bit for bit with
grpo_nf4_dequant, grpo_nf4_lora_train_forward and _backward (csrc/lora_train.hip, csrc/gemm16.hip).

Tolerances: every result is a float32 sum of exact products, rounded once to the
16-bit type.  Against the float64 sum it differs by that rounding, at most the unit
roundoff u (2^-8 in bf16, 2^-11 in float16) of the value, and by an intermediate of
its size that falls to the other neighbour, one ulp or at most 2 u (those inside a sum
average out): 3 u of max|result|."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}  # unit roundoff


def _close(got, want, dt, what):
    err = float((got.double() - want).abs().max() / want.abs().max())
    print(f"{what}: {err:.2e}", flush=True)
    assert err <= 3 * U[dt], what


def _inputs(dev, m, n, k, r, dt, seed):
    from grpo_mi355x.core.nf4 import quantize_nf4

    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s, sd=1.0: (torch.randn(*s, generator=g) * sd).to(dt).to(dev)
    packed, st = quantize_nf4((torch.randn(n, k, generator=g) * 0.02).to(dev),
                              64 if k % 64 == 0 else 32)
    return (rnd(m, k), rnd(m, n, sd=0.1), (packed.view(-1), st.absmax, st.code, st.blocksize),
            rnd(r, k, sd=0.05), rnd(n, r, sd=0.05), rnd(n))


# M: one row to past each tile (64, 128, 256) and each row slicing of the adapters'
# gradients; N, K: column tiles with remainders, 1 to 48 stages of 32 of either
# product; ranks below, at and past a tile of 16
@pytest.mark.parametrize("m,n,k,r", [(1, 32, 32, 1), (16, 128, 64, 16), (33, 160, 544, 8),
                                     (127, 256, 1536, 17), (300, 1536, 96, 32),
                                     (1050, 288, 1024, 16), (1300, 4096, 512, 5),
                                     (8200, 1536, 512, 16), (5000, 4128, 256, 16),
                                     (1050, 1024, 288, 16), (8200, 512, 1536, 16)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_training_linear(dev, m, n, k, r, dt):
    from grpo_mi355x.kernels import ops

    x, g, wq, a, b, bias = _inputs(dev, m, n, k, r, dt, m + n + k + r)
    print(f"nf4_lora_train M={m} N={n} K={k} r={r} {dt}", flush=True)
    w = ops.nf4_dequant(*wq[:3], n * k, wq[3], dtype=dt).view(n, k).double()
    s = 1.7  # not a power of two: the rounded scaling matters
    sd = float(torch.tensor(s, dtype=dt))
    rt = lambda t: t.to(dt).double()
    sg = rt(g.double() * sd)
    gi, xa = rt(sg @ b.double()), rt(x.double() @ a.double().t())
    gx, ga, gb = ops.nf4_lora_train_backward(x, g, *wq, a, b, s)
    _close(ga, gi.t() @ x.double(), dt, "grad_A")
    _close(gb, sg.t() @ xa, dt, "grad_B")
    _close(gx, rt(g.double() @ w) + rt(gi @ a.double()), dt, "grad_x")
    # each result alone is the same
    for i in range(3):
        only = ops.nf4_lora_train_backward(x, g, *wq, a, b, s, *(j == i for j in range(3)))
        assert [o is not None for o in only] == [j == i for j in range(3)]
        assert torch.equal(only[i], (gx, ga, gb)[i])
    u = rt(rt(xa @ b.double().t()) * sd)
    acc = rt(x.double() @ w.t())
    for bi in (None, bias):
        base = acc if bi is None else rt(acc + bi.double())
        _close(ops.nf4_lora_train_forward(x, *wq, a, b, s, bi), base + u, dt, "y")


def test_training_linear_reaches_every_tile():
    """The cases above run each of the GEMM's four tiles in either direction."""
    from grpo_mi355x import _lib

    def tile(m, n):
        a, b = ctypes.c_int(0), ctypes.c_int(0)
        _lib.check(_lib.library().grpo_gemm16_tile(m, n, ctypes.byref(a), ctypes.byref(b)), "tile")
        return a.value, b.value

    (shapes,) = [m.args[1] for m in test_training_linear.pytestmark if m.args[0] == "m,n,k,r"]
    tiles = {(256, 256), (128, 128), (64, 128), (64, 64)}
    assert {tile(m, n) for m, n, _, _ in shapes} == tiles  # y: [M, N]
    assert {tile(m, k) for m, _, k, _ in shapes} == tiles  # grad_x: [M, K]


def test_rows_past_the_end_add_nothing(dev):
    """Rows after the last (the tail of a 32-row step) repeat no infinity: an inf in
    the last row reaches its own results only."""
    from grpo_mi355x.kernels import ops

    x, g, wq, a, b, _ = _inputs(dev, 37, 128, 128, 16, torch.bfloat16, 3)
    g[-1, 5] = float("inf")
    gx, ga, gb = ops.nf4_lora_train_backward(x, g, *wq, a, b, 1.0)
    assert torch.isfinite(gb[torch.arange(128) != 5]).all()
    assert not torch.isfinite(gb[5]).any()
    assert torch.isfinite(gx[:-1]).all()


@pytest.mark.parametrize("how", ["misaligned", "create_graph", "batched"])
def test_backward_of_what_the_kernels_do_not_take(dev, how):
    """grad_out rows off their alignment, a differentiable and a batched backward
    give the gradients of the kernels' path (one rounding of each product)."""
    from grpo_mi355x.core.nf4 import Linear4bitNF4
    from grpo_mi355x.kernels import lora_fused_forward

    m, n, k, r = 1100, 256, 128, 16
    gen = torch.Generator().manual_seed(1)
    rnd = lambda *s, sd: (torch.randn(*s, generator=gen) * sd).bfloat16().to(dev)
    base = Linear4bitNF4.from_weight(rnd(n, k, sd=0.02).float())
    x, g = rnd(1, m, k, sd=1.0).requires_grad_(), rnd(1, m, n, sd=0.1)
    a, b = rnd(r, k, sd=0.05).requires_grad_(), rnd(n, r, sd=0.05).requires_grad_()
    y = lora_fused_forward(x, base_layer=base, lora_A=a, lora_B=b, scaling=2.0)
    grads = lambda go, **kw: torch.autograd.grad(y, (x, a, b), go, retain_graph=True, **kw)
    want = grads(g)
    if how == "misaligned":
        got = grads(torch.cat([g.new_zeros(4), g.reshape(-1)])[4:].view(1, m, n))
    elif how == "create_graph":
        got = grads(g, create_graph=True)
        assert all(t.requires_grad for t in got)
    else:
        got = [t[1] for t in grads(torch.stack([g * 0, g]), is_grads_batched=True)]
    for u, v in zip(got, want):
        _close(u.detach(), v.double(), torch.bfloat16, how)


@pytest.mark.parametrize("m", [1, 33, 2048, 2049])
def test_linear4bit_weight_layout_with_and_without_gradient(dev, m):
    """Linear4bitNF4 keeps the weight transposed where x's gradient is asked for (up to
    2048 rows): the same output and gradient as over the row-major weight, up to the
    order of the float32 sums."""
    from grpo_mi355x.core.nf4 import Linear4bitNF4

    torch.manual_seed(m)
    lin = Linear4bitNF4.from_weight(torch.randn(2048, 1024, device=dev) * 0.02)
    x = torch.randn(1, m, 1024, device=dev).bfloat16().requires_grad_()
    g = torch.randn(1, m, 2048, device=dev).bfloat16()
    w = lin.dequantize()
    used = lin._dequantized_for(x, torch.bfloat16)
    assert torch.equal(used, w) and used.is_contiguous() == (m > 2048)
    assert lin._dequantized_for(x.detach(), torch.bfloat16).is_contiguous()
    y = lin(x)
    y.backward(g)
    _close(y.detach(), torch.nn.functional.linear(x.detach().double(), w.double()),
           torch.bfloat16, "y")
    _close(x.grad, g.double() @ w.double(), torch.bfloat16, "grad_x")


@pytest.mark.parametrize("n,k,bs", [
    (1, 8, 8), (3, 24, 24), (65, 128, 64), (129, 1536, 4096),
    # one run of eight per thread up to 2^24 values, four beyond
    (4096, 4096, 64), (4099, 4104, 64), (4097, 4104, 24)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_dequant_runs_of_eight(dev, n, k, bs, dt):
    """nf4_dequant's vector path over odd run counts and blocksizes, bit for bit with
    the codebook product rounded by torch."""
    from grpo_mi355x.core.nf4 import nf4_code
    from grpo_mi355x.kernels import ops

    torch.manual_seed(n)
    packed = torch.randint(0, 256, (n * k // 2,), dtype=torch.uint8, device=dev)
    absmax = torch.rand(-(-n * k // bs), device=dev)
    q = torch.stack([packed >> 4, packed & 15], 1).view(-1).long()
    want = (nf4_code(dev)[q] * absmax.repeat_interleave(bs)[:n * k]).to(dt)
    got = ops.nf4_dequant(packed, absmax, nf4_code(dev), n * k, bs, dtype=dt)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_no_grad_call_is_the_recorded_one(dev):
    """Without grad mode the autograd function is passed by: the same output, and a
    forward-mode level, a transform or grad mode still goes through it; arguments
    the kernels must not see stay refused."""
    from grpo_mi355x.core.lora import ManualLoRALayer
    from grpo_mi355x.core.nf4 import Linear4bitNF4
    from grpo_mi355x.kernels import lora_forward as L, lora_fused_forward

    torch.manual_seed(0)
    base = Linear4bitNF4.from_weight(torch.randn(256, 512, device=dev) * 0.02,
                                     torch.randn(256, device=dev))
    layer = ManualLoRALayer(base).to(dev).bfloat16()
    torch.nn.init.normal_(layer.lora_B.weight, std=0.05)
    called, apply = [], L.FusedLoRAFunction.apply
    for m in (8, 100, 600):
        x = torch.randn(1, m, 512, device=dev).bfloat16()
        want = lora_fused_forward(x, lora_layer=layer)
        assert want.grad_fn is not None
        with torch.no_grad():
            got = lora_fused_forward(x, lora_layer=layer)
        assert got.grad_fn is None and torch.equal(got, want.detach())
    L.FusedLoRAFunction.apply = staticmethod(lambda *a: called.append(1) or apply(*a))
    try:
        with torch.no_grad():
            lora_fused_forward(x, lora_layer=layer)
            assert not called
            with torch.autograd.forward_ad.dual_level():
                lora_fused_forward(x, lora_layer=layer)
            assert len(called) == 1
    finally:
        L.FusedLoRAFunction.apply = apply
    with torch.no_grad():
        for bad in (torch.zeros(255, device=dev), torch.zeros(256)):
            base.bias = torch.nn.Parameter(bad, requires_grad=False)
            with pytest.raises(ValueError):
                lora_fused_forward(x, lora_layer=layer)
        base.bias = None
        full, base.weight.quant_state.absmax = base.weight.quant_state.absmax, \
            base.weight.quant_state.absmax[:-1]
        with pytest.raises(ValueError):
            lora_fused_forward(x, lora_layer=layer)
        base.weight.quant_state.absmax = full
        # vmap: no storage to hand to a kernel; the layer's torch branch serves it
        y = torch.vmap(lambda t: layer(t))(torch.stack([x, 2 * x]))
        assert y.shape == (2, 1, 600, 256)


def test_transposed_dequant_of_strided_scales(dev):
    """The weight kept transposed for a gradient holds the values of dequantize() also
    for strided absmax and codebook, and what dequantize() refuses stays refused."""
    from grpo_mi355x.core.nf4 import Linear4bitNF4

    torch.manual_seed(3)
    layer = Linear4bitNF4.from_weight(torch.randn(2048, 1024, device=dev) * 0.02)
    x = torch.randn(1, 40, 1024, device=dev).bfloat16().requires_grad_()
    qs, want = layer.weight.quant_state, layer.dequantize()
    every2 = lambda t: torch.stack([t, t + 1], 1).view(-1)[::2]
    qs.absmax, qs.code = every2(qs.absmax), every2(qs.code)
    w = layer._dequantized_for(x, torch.bfloat16)
    assert not w.is_contiguous() and torch.equal(w, want)  # stored [in, out]
    qs.code = qs.code.double()
    with pytest.raises(ValueError):
        layer(x)


@pytest.mark.parametrize("m,n,k,r,dt", [(1030, 96, 4224, 16, torch.bfloat16),
                                        (1100, 64, 4128, 32, torch.float16)])
def test_forward_over_library_products_is_the_training_forward(dev, m, n, k, r, dt):
    """A long K over few tiles runs the dequantized weight + library products: the same
    rounding points as the training kernels."""
    from grpo_mi355x.core.nf4 import Linear4bitNF4
    from grpo_mi355x.kernels import lora_forward as L, lora_fused_forward, ops

    gen = torch.Generator().manual_seed(n)
    rnd = lambda *s, sd: (torch.randn(*s, generator=gen) * sd).to(dt).to(dev)
    base = Linear4bitNF4.from_weight(rnd(n, k, sd=0.02).float(), rnd(n, sd=1.0))
    x, a, b = rnd(1, m, k, sd=1.0), rnd(r, k, sd=0.05), rnd(n, r, sd=0.05)
    qs = base.weight.quant_state
    assert not L.train_forward_pays(m, n, k, r, qs.blocksize, dt)
    got = lora_fused_forward(x, base_layer=base, lora_A=a, lora_B=b, scaling=1.7)
    want = ops.nf4_lora_train_forward(x[0], base.weight.data.view(-1), qs.absmax, qs.code,
                                      qs.blocksize, a, b, 1.7, base.bias.to(dt))
    _close(got[0], want.double(), dt, "y")
