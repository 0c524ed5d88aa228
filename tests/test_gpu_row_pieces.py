"""The 16-byte forms of embedding, add + RMSNorm and RoPE + append against their
column-wise forms, which the same call takes for rows that are not 16-byte aligned.

Copies and RoPE are equal bit for bit; the norm's sum of squares runs in another order
(float32, relative error below 1e-5), so a result may fall to the neighbouring bf16 value."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _off(t):
    """A copy of t that starts 2 bytes past a 16-byte boundary."""
    buf = torch.zeros(t.numel() + 1, dtype=t.dtype, device=t.device)
    return buf[1:].view(t.shape).copy_(t)


def _lib():
    from grpo_mi355x import _lib

    return _lib.device_library(), _lib.check


# widths: one piece, a partial and a whole pass of 2048, two passes, one past them (column-wise)
@pytest.mark.parametrize("m,h", [(1, 8), (3, 1536), (511, 2048), (5, 2056), (64, 3584),
                                 (2, 4096), (2, 4104), (3, 1540)])
@pytest.mark.parametrize("residual", [True, False])
def test_add_rmsnorm_pieces(dev, m, h, residual):
    lib, check = _lib()
    g = torch.Generator().manual_seed(m + h)
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)
    x, r, w = rnd(m, h), rnd(m, h), rnd(h)
    got = []
    for f in (lambda t: t.clone(), _off):
        a, b, y = f(x), f(r), f(torch.zeros_like(x))
        bp = b.data_ptr() if residual else None
        check(lib.grpo_add_rmsnorm(a.data_ptr(), bp, bp, w.data_ptr(), y.data_ptr(), m, h, 1e-6,
                                   torch.cuda.current_stream().cuda_stream), "norm")
        got.append((y.float(), b))
    assert torch.equal(got[0][1], got[1][1])
    hh = (x + r if residual else x).double()
    want = hh * torch.rsqrt(hh.pow(2).mean(1, keepdim=True) + 1e-6) * w.double()
    for y, _ in got:  # two roundings to bf16, at most 2^-8 each, and the sum's error
        assert float(((y - want).abs() / want.abs().clamp(min=1e-6)).max()) <= 2.02 * 2.0 ** -8
    assert float(((got[0][0] - got[1][0]).abs() / want.abs().clamp(min=1e-6)).max()) <= 2.0 ** -6
    assert float((got[0][0] == got[1][0]).float().mean()) >= 0.99


@pytest.mark.parametrize("h", [8, 1536, 3584, 1540])
def test_embedding_pieces(dev, h):
    lib, check = _lib()
    table = torch.randn(50, h, device=dev).bfloat16()
    ids = torch.tensor([0, 49, -1, 50, 7], device=dev)
    for f in (lambda t: t.clone(), _off):
        t, out = f(table), f(torch.ones(5, h, dtype=torch.bfloat16, device=dev))
        check(lib.grpo_embedding(ids.data_ptr(), t.data_ptr(), 50, h, out.data_ptr(), 5,
                                 torch.cuda.current_stream().cuda_stream), "embedding")
        assert torch.equal(out[[0, 1, 4]], table[[0, 49, 7]]) and not out[2:4].any()


@pytest.mark.parametrize("hq,hkv,d,pad", [(12, 2, 128, 0), (28, 4, 128, 8), (1, 1, 16, 0),
                                          (32, 8, 128, 0), (2, 1, 24, 0), (12, 2, 128, 4),
                                          (2, 1, 128, 0), (6, 5, 32, 8)])
def test_rope_append_pieces(dev, hq, hkv, d, pad):
    lib, check = _lib()
    rows, bs, blocks, cap = 37, 16, 24, 4
    g = torch.Generator().manual_seed(hq + d)
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)
    qkv, cos, sin = rnd(rows, (hq + 2 * hkv) * d + pad), rnd(50, d), rnd(50, d)
    pos = torch.arange(rows, dtype=torch.int32) * 2 - 3  # negative, in range, past the tables
    bt = torch.randint(-1, blocks + 1, (rows, cap), generator=g).int()
    # one row per slot, so that the result does not depend on the order of the rows
    used = set()
    for i in range(rows):
        p = int(pos[i])
        if 0 <= p < cap * bs and (int(bt[i, p // bs]), p % bs) in used:
            bt[i, p // bs] = -1
        if 0 <= p < cap * bs:
            used.add((int(bt[i, p // bs]), p % bs))
    pos, bt = pos.to(dev), bt.to(dev)
    got = []
    for f in (lambda t: t.clone(), _off):
        a = f(qkv)
        q, k, v = (f(torch.ones(*s, dtype=torch.bfloat16, device=dev)) for s in (
            (rows, hq, d), (blocks, hkv, bs, d), (blocks, hkv, bs, d)))
        check(lib.grpo_rope_append(
            a.data_ptr(), a.shape[1], hq, hkv, d, cos.data_ptr(), sin.data_ptr(), 50,
            pos.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), blocks, bt.data_ptr(), cap,
            bs, cap, rows, torch.cuda.current_stream().cuda_stream), "rope")
        got.append((q, k, v))
    for x, y in zip(*got):
        assert torch.equal(x, y)
