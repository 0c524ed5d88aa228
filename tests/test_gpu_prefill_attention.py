"""grpo_paged_attn_prefill against the decode attention of the same rows, which is
pinned against the oracle (tests/test_gpu_attention.py), and against float64.

Both kernels hold float32 scores, sums and P (as two bf16 terms) and round once to
bf16; they differ in the order of the sums, so a result can fall to the other
neighbouring bf16 value: within one ulp (2^-7 of the value at most), most of them equal."""

import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(dev, M, Hq, Hkv, lens, max_blocks, seed, holes=()):
    from grpo_mi355x import _lib
    from grpo_mi355x.kernels import ops

    lib = _lib.device_library()
    g = torch.Generator().manual_seed(seed)
    nb = max_blocks + 3
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16().to(dev)
    q, k, v = rnd(M, Hq, 128), rnd(nb, Hkv, 16, 128), rnd(nb, Hkv, 16, 128)
    table = torch.randperm(nb, generator=g)[:max_blocks].int()
    if holes:  # ids out of range, and a block 0 that must not leak through them
        table[table == 0] = nb - 1
        for i, b in enumerate(holes):
            table[b] = (-1, nb)[i % 2]
        k[0], v[0] = float("nan"), float("nan")
    table = table.to(dev)
    ln = torch.tensor(lens, dtype=torch.int32, device=dev)
    out = torch.full((M, Hq, 128), 7.0, dtype=torch.bfloat16, device=dev)
    print(f"prefill attention M={M} Hq={Hq} Hkv={Hkv} max_blocks={max_blocks}", flush=True)
    _lib.check(lib.grpo_paged_attn_prefill(
        q.data_ptr(), Hq * 128, 128, k.data_ptr(), v.data_ptr(), nb, table.data_ptr(),
        ln.data_ptr(), out.data_ptr(), M, Hq, Hkv, 128, 16, max_blocks, 1 / math.sqrt(128),
        _lib.stream_handle(dev)), "prefill")
    want = ops.paged_attention_decode(q, k, v, table.expand(M, max_blocks).contiguous(), ln,
                                      1 / math.sqrt(128), out_dtype=torch.float32)
    ops.attention_handover_check(dev)
    return out.float(), want, (q, k, v, table)


def _form(M, Hq, Hkv):
    """(heads per workgroup, parts of a step) that the launcher picks."""
    from grpo_mi355x import _lib

    h, p = ctypes.c_int(0), ctypes.c_int(0)
    _lib.check(_lib.library().grpo_paged_attn_prefill_plan(M, Hq, Hkv, ctypes.byref(h),
                                                           ctypes.byref(p)), "plan")
    return h.value, p.value


# rows: within, at and past a 16-row tile; contexts: within a block, at and past the 32-token
# parts, the 128-token steps, the ring of two, the 64-block table windows, empty and clamped ones
@pytest.mark.parametrize("M,Hq,Hkv,first,max_blocks", [
    (1, 1, 1, 1, 1), (17, 12, 2, 1, 2), (16, 4, 4, 17, 3), (40, 7, 1, 60, 8), (64, 28, 4, 129, 12),
    (33, 10, 2, 200, 16), (70, 8, 1, 1, 6), (512, 12, 2, 1, 32), (100, 16, 8, 4000, 260),
    (16, 2, 1, 1009, 64), (16, 2, 1, 1020, 70), (16, 2, 1, 2040, 130),
    # a longest row that ends with a step, which fetches nothing after it: the first,
    # the second, the first of the second table window
    (16, 2, 1, 113, 8), (16, 2, 1, 241, 16), (16, 12, 2, 1137, 72)])
def test_prefill_attention(dev, M, Hq, Hkv, first, max_blocks):
    lens = [first + i for i in range(M)]
    if M > 20:
        lens[3], lens[5], lens[-1] = 0, -4, 16 * max_blocks + 50
    got, want, _ = _run(dev, M, Hq, Hkv, lens, max_blocks, M + Hq)
    assert float(((got - want).abs() / want.abs().clamp(min=1e-3)).max()) <= 2.0 ** -7
    assert float((got == want.bfloat16().float()).float().mean()) >= 0.97
    if M > 20:
        assert not got[3].any() and not got[5].any()


# More workgroups than CUs: two parts of 32 tokens per 64-token step (a 64-block table window
# is 16 of them), one, two and four heads per workgroup, the last with and without an idle
# wave; contexts from one step to several windows, one that ends with a step and a window
@pytest.mark.parametrize("M,Hq,Hkv,form", [(528, 8, 8, (1, 2)), (528, 16, 8, (2, 2)),
                                           (512, 28, 4, (4, 2)), (530, 32, 8, (4, 2)),
                                           (520, 6, 2, None), (1300, 6, 2, (4, 2))])
@pytest.mark.parametrize("first,max_blocks", [(1, 40), (1000, 128), (2040, 210)])
def test_prefill_attention_in_two_parts(dev, M, Hq, Hkv, form, first, max_blocks):
    assert _form(M, Hq, Hkv) == (form or (2, 4))
    lens = [first + i // 2 for i in range(M)]
    lens[3], lens[5], lens[-1] = 0, -4, 16 * max_blocks + 50
    lens[96:112] = [1024] * 16
    got, want, _ = _run(dev, M, Hq, Hkv, lens, max_blocks, M + Hq)
    assert float(((got - want).abs() / want.abs().clamp(min=1e-3)).max()) <= 2.0 ** -7
    assert float((got == want.bfloat16().float()).float().mean()) >= 0.97
    assert not got[3].any() and not got[5].any()


@pytest.mark.parametrize("M,Hq,Hkv", [(50, 6, 1), (528, 8, 8), (528, 16, 8), (512, 28, 4)])
@pytest.mark.parametrize("first,max_blocks,holes", [
    (20, 12, (1, 6)), (1000, 80, (0, 62, 63, 64, 65, 66)), (1, 3, (0, 1, 2))])
def test_prefill_attention_skips_invalid_blocks(dev, first, max_blocks, holes, M, Hq, Hkv):
    got, want, _ = _run(dev, M, Hq, Hkv, [first + 3 * (i % 50) for i in range(M)], max_blocks, 5,
                        holes)
    assert torch.isfinite(got).all()
    assert float(((got - want).abs() / want.abs().clamp(min=1e-3)).max()) <= 2.0 ** -7


def test_prefill_attention_against_float64(dev):
    got, _, (q, k, v, table) = _run(dev, 96, 12, 2, [100 + i for i in range(96)], 13, 9)
    kk, vv = (t[table.long()].transpose(1, 2).reshape(-1, 2, 128).double().repeat_interleave(6, 1)
              for t in (k, v))
    s = torch.einsum("mhd,thd->mht", q.double(), kk) / math.sqrt(128)
    on = torch.arange(kk.shape[0], device=dev) < torch.arange(100, 196, device=dev)[:, None]
    p = torch.softmax(s.masked_fill(~on[:, None], -math.inf), -1)
    want = torch.einsum("mht,thd->mhd", p, vv)
    # one rounding to bf16, 2^-8 of the value at most, with a little for the float32 sums
    assert float(((got - want).abs() / want.abs().clamp(min=1e-2)).max()) <= 1.05 * 2.0 ** -8


# lens of a chunk that starts inside a block, of rows in no order, of idle rows; four parts and two
@pytest.mark.parametrize("M,Hq,Hkv,lens", [
    (40, 6, 1, lambda i: 101 + i), (33, 4, 4, lambda i: (37 * i) % 250),
    (600, 14, 2, lambda i: 3 * i % 700), (530, 8, 8, lambda i: 90 + i % 50)])
def test_prefill_attention_takes_nothing_from_tokens_past_a_context(dev, M, Hq, Hkv, lens):
    """Infinite and NaN values of tokens that a row does not attend (later tokens of the
    chunk, slots not written yet) do not reach it; of those it attends, they do."""
    from grpo_mi355x import _lib

    lib = _lib.device_library()
    g = torch.Generator().manual_seed(M)
    n = [lens(i) for i in range(M)]
    top = max(n)
    max_blocks = -(-top // 16)
    rnd = lambda *s: torch.randn(*s, generator=g).bfloat16()
    q, k, v = rnd(M, Hq, 128), rnd(max_blocks, Hkv, 16, 128), rnd(max_blocks, Hkv, 16, 128)
    at = lambda c, t: c[t // 16, :, t % 16]  # table: the identity
    for i, t in enumerate(t for t in (70, 112, 113, 127, 128, 200, top - 1) if t < top):
        at(v, t)[:, 5 * i] = (float("inf"), float("-inf"), float("nan"))[i % 3]
    at(k, min(top - 1, 130))[:] = float("nan")
    for t in range(top, 16 * max_blocks):  # never written
        at(k, t)[:], at(v, t)[:] = float("nan"), float("nan")
    table, ln = torch.arange(max_blocks, dtype=torch.int32), torch.tensor(n, dtype=torch.int32)
    d = [t.to(dev) for t in (q, k, v, table, ln)]
    out = torch.empty(M, Hq, 128, dtype=torch.bfloat16, device=dev)
    print(f"prefill attention, values not finite, M={M} Hq={Hq} Hkv={Hkv}", flush=True)
    _lib.check(lib.grpo_paged_attn_prefill(
        d[0].data_ptr(), Hq * 128, 128, d[1].data_ptr(), d[2].data_ptr(), max_blocks,
        d[3].data_ptr(), d[4].data_ptr(), out.data_ptr(), M, Hq, Hkv, 128, 16, max_blocks,
        1 / math.sqrt(128), _lib.stream_handle(dev)), "prefill")
    got = out.float().cpu()
    kk, vv = (c.transpose(1, 2).reshape(-1, Hkv, 128).double().repeat_interleave(Hq // Hkv, 1)
              for c in (k, v))
    for m in range(M):
        if n[m] == 0:
            assert not got[m].any()
            continue
        s = torch.einsum("hd,thd->ht", q[m].double(), kk[:n[m]]) / math.sqrt(128)
        want = torch.einsum("ht,thd->hd", torch.softmax(s, -1), vv[:n[m]])
        on = torch.isfinite(want)
        assert torch.equal(torch.isfinite(got[m]), on), (m, n[m])
        assert ((got[m] - want).abs()[on] <= 1.05 * 2.0 ** -8 * want.abs()[on].clamp(min=1e-2)).all()
