"""Loading rows into an engine's device state (grpo_decode_start,
grpo_prefill_rows) against the same state built with torch, exactly."""

import pytest
import torch

pytestmark = pytest.mark.gpu


class _State:
    """The attributes DecodeEngine.start writes."""

    def __init__(self, lib, dev, B, max_blocks):
        i32 = dict(dtype=torch.int32, device=dev)
        self.lib, self.device, self.B, self.max_blocks = lib, dev, B, max_blocks
        for name in ("pos", "append_pos", "attn_len", "count", "limit"):
            setattr(self, name, torch.full((B,), 77, **i32))
        self.tokens = torch.full((B,), 77, dtype=torch.int64, device=dev)
        self.active = torch.zeros(B, dtype=torch.bool, device=dev)
        self.eos = torch.zeros(1, dtype=torch.int64, device=dev)
        self.pad = torch.zeros(1, dtype=torch.int64, device=dev)
        self.block_tables = torch.full((B, max_blocks), 77, **i32)
        self.generated, self.graph, self.graph_multi = None, object(), {1: 2}

    def step(self):
        self.seen = getattr(self, "seen", []) + [[t.clone() for t in (
            self.tokens, self.append_pos, self.attn_len, self.block_tables)]]


@pytest.mark.parametrize("B,max_blocks,w,cols,kind", [
    (1, 1, 1, 1, torch.int64), (8, 300, 257, 512, torch.int64), (64, 256, 256, 300, torch.int32),
    (5, 7, 0, 3, torch.float32)])
def test_decode_start(dev, B, max_blocks, w, cols, kind):
    from grpo_mi355x import _lib
    from grpo_mi355x.rollout.decode import DecodeEngine

    torch.manual_seed(B)
    s = _State(_lib.device_library(), dev, B, max_blocks)
    tok = torch.randint(0, 1 << 40, (B, 1))
    pos, lim = torch.randint(0, 5000, (B,)).to(kind), torch.randint(-1, 3, (B,)).to(kind)
    bt = torch.randint(0, 1 << 20, (B, w), dtype=torch.int32)
    DecodeEngine.start(s, tok.to(dev), pos.to(dev), bt.to(dev), lim.to(dev), cols, 5, 9)
    on = lim > 0
    assert s.graph is None and s.graph_multi == {} and s._pos_hi is None
    assert torch.equal(s.tokens.cpu(), tok.view(B)) and int(s.eos) == 5 and int(s.pad) == 9
    assert torch.equal(s.pos.cpu(), pos.int()) and torch.equal(s.limit.cpu(), lim.int())
    assert not s.count.any() and torch.equal(s.active.cpu(), on)
    assert torch.equal(s.append_pos.cpu(), torch.where(on, pos.int(), -1))
    assert torch.equal(s.attn_len.cpu(), torch.where(on, pos.int() + 1, 0))
    assert torch.equal(s.block_tables[:, :w].cpu(), bt) and (s.block_tables[:, w:] == -1).all()
    assert s.generated.shape == (B, cols) and (s.generated == 9).all()
    # host tensors, one shared table row, no eos, nothing recorded
    s.generated.fill_(3)
    s.graph = keep = object()
    if w:
        DecodeEngine.start(s, tok, pos, bt[:1], lim, cols + 1, record=False)
        assert torch.equal(s.block_tables[:, :w].cpu(), bt[:1].expand(B, w))
        assert int(s.eos) == -1 and (s.generated == 3).all() and s.graph is keep
    with pytest.raises((ValueError, RuntimeError)):
        DecodeEngine.start(s, tok, pos, torch.zeros(B, max_blocks + 1, dtype=torch.int32), lim, 4)
    with pytest.raises(RuntimeError):
        DecodeEngine.start(s, tok.repeat(2, 1), pos, bt, lim, 4)


@pytest.mark.parametrize("B,n,w", [(16, 1, 1), (64, 64, 4), (64, 150, 10), (512, 511, 33)])
def test_prefill_chunks(dev, B, n, w):
    from grpo_mi355x import _lib
    from grpo_mi355x.rollout.decode import _run_chunks

    s = _State(_lib.device_library(), dev, B, 40)
    prompt, table = torch.randint(0, 1000, (n + 3,)), torch.randint(0, 99, (1, w)).int()
    _run_chunks(s, table.to(dev), prompt.to(dev), n)
    assert len(s.seen) == -(-n // B)
    row = torch.arange(B)
    for c, (tok, ap, al, bt) in enumerate(s.seen):
        at = c * B + row
        on = at < n
        want = torch.where(on, prompt[at.clamp(max=n - 1)], 0)
        assert torch.equal(tok.cpu(), want)
        assert torch.equal(ap.cpu(), torch.where(on, at, -1).int())
        assert torch.equal(al.cpu(), torch.where(on, at + 1, 0).int())
        assert torch.equal(bt[:, :w].cpu(), table.expand(B, w)) and (bt[:, w:] == -1).all()
    with pytest.raises(RuntimeError):
        _run_chunks(s, table, prompt, n + 4)
