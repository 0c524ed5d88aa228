"""The LoRA side of the training step on the GPU (csrc/lora_train.hip) against
float64 torch on the same rounding points: grpo_nf4_dequant_t bit for bit with
grpo_nf4_dequant, grpo_lora_backward and grpo_lora_forward_add.

Tolerances: every result is a float32 sum of exact products, rounded once to the
16-bit type.  Against the float64 sum it differs by that rounding (half an ulp:
2^-9 of the value in bf16, 2^-12 in float16) plus the rounding of the 16-bit
intermediates, which can each fall to the other neighbour (one ulp of a term,
averaged over the sum); 2.5 ulp of max|result| covers both."""

import pytest
import torch

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _close(got, want, dt, what):
    err = float((got.double() - want).abs().max() / want.abs().max())
    print(f"{what}: {err:.2e}", flush=True)
    assert err <= 2.5 * ULP[dt], what


def _inputs(dev, m, n, k, r, dt, seed):
    g = torch.Generator().manual_seed(seed)
    rnd = lambda *s, sd=1.0: (torch.randn(*s, generator=g) * sd).to(dt).to(dev)
    return (rnd(m, k), rnd(m, n, sd=0.1), rnd(r, k, sd=0.05), rnd(n, r, sd=0.05),
            rnd(m, k), rnd(m, n), rnd(n))


@pytest.mark.parametrize("n,k", [(8, 32), (64, 128), (72, 160), (1536, 256), (200, 1536)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_dequant_t_is_the_transposed_dequant(dev, n, k, dt):
    from grpo_mi355x.core.nf4 import quantize_nf4
    from grpo_mi355x.kernels import ops

    torch.manual_seed(n + k)
    packed, st = quantize_nf4(torch.randn(n, k, device=dev) * 0.02, 32 if k % 64 else 64)
    args = (packed.view(-1), st.absmax, st.code)
    want = ops.nf4_dequant(*args, n * k, st.blocksize, dtype=dt).view(n, k)
    got = ops.nf4_dequant_t(*args, n, k, st.blocksize, dtype=dt)
    assert torch.equal(got.view(torch.int16), want.t().contiguous().view(torch.int16))


@pytest.mark.parametrize("m,n,k,r", [(1, 8, 8, 1), (16, 128, 64, 16), (33, 136, 520, 8),
                                     (127, 256, 1536, 17), (300, 1536, 72, 32),
                                     (1050, 264, 1000, 16), (8200, 1536, 512, 16)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_lora_backward_and_forward_add(dev, m, n, k, r, dt):
    from grpo_mi355x.kernels import ops

    x, g, a, b, gx, y, bias = _inputs(dev, m, n, k, r, dt, m + n + k + r)
    s = 1.7  # not a power of two: the rounded scaling matters
    sd = float(torch.tensor(s, dtype=dt))
    rt = lambda t: t.to(dt).double()
    sg = rt(g.double() * sd)
    gi, xa = rt(sg @ b.double()), rt(x.double() @ a.double().t())
    ga, gb = ops.lora_backward(x, g, a, b, s, grad_x=(got := gx.clone()))
    _close(ga, gi.t() @ x.double(), dt, "grad_A")
    _close(gb, sg.t() @ xa, dt, "grad_B")
    _close(got, gx.double() + rt(gi @ a.double()), dt, "grad_x")
    # each result alone is the same
    assert torch.equal(ops.lora_backward(x, g, a, b, s, want_b=False)[0], ga)
    assert torch.equal(ops.lora_backward(x, g, a, b, s, want_a=False)[1], gb)
    alone = gx.clone()
    ops.lora_backward(x, g, a, b, s, grad_x=alone, want_a=False, want_b=False)
    assert torch.equal(alone, got)
    u = rt(rt(xa @ b.double().t()) * sd)
    for bi in (None, bias):
        base = y.double() if bi is None else rt(y.double() + bi.double())
        _close(ops.lora_forward_add(y.clone(), x, a, b, s, bi), base + u, dt, "y")


def test_rows_past_the_end_add_nothing(dev):
    """Rows after the last (the tail of a 32-row step) repeat no infinity: an inf in
    the last row reaches its own results only."""
    from grpo_mi355x.kernels import ops

    x, g, a, b, _, _, _ = _inputs(dev, 37, 128, 128, 16, torch.bfloat16, 3)
    g[-1, 5] = float("inf")
    ga, gb = ops.lora_backward(x, g, a, b, 1.0)
    assert torch.isfinite(gb[torch.arange(128) != 5]).all()
    assert not torch.isfinite(gb[5]).any()
