"""Causal attention of whole prompts (arcq_attention_prefill) against 64-bit softmax(q k^T / sqrt(d)) v on the CPU
(model/qLlamaLayer.py:340-370)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def operands(batch, seq, heads, kv_heads, gain=2.0, seed=1):
    g = torch.Generator().manual_seed(seed + seq + heads)
    t = batch * seq
    q = (torch.randn(t, heads, 128, generator=g) * gain).to(torch.bfloat16)
    k = torch.randn(t, kv_heads, 128, generator=g).to(torch.bfloat16)
    qkv = torch.randn(t, (heads + 2 * kv_heads) * 128, generator=g).to(torch.bfloat16)
    return q, k, qkv


def reference(q, k, v, seq):
    t, heads, d = q.shape
    q, k, v = (x.double().view(t // seq, seq, -1, d).transpose(1, 2) for x in (q, k, v))
    k, v = (x.repeat_interleave(heads // x.shape[1], 1) for x in (k, v))
    s = (q @ k.transpose(-1, -2)) / math.sqrt(d)
    s = s.masked_fill(torch.ones(seq, seq, dtype=torch.bool).triu(1), float("-inf"))
    return (torch.softmax(s, -1) @ v).transpose(1, 2).reshape(t, heads * d)


@pytest.mark.parametrize("batch,seq,heads,kv_heads", [(1, 1, 1, 1), (3, 2, 4, 4), (2, 31, 8, 2), (1, 32, 7, 1), (2, 33, 4, 2), (1, 63, 4, 1), (1, 64, 2, 2),
                                                      (5, 65, 4, 2), (1, 127, 8, 8), (2, 128, 6, 2), (3, 129, 8, 1), (1, 257, 28, 4), (2, 500, 8, 2)])
def test_attention_prefill(batch, seq, heads, kv_heads):
    """Queries and keys ending inside a tile and at its edge, every kind of grouping, V as a strided slice.  What is left of the
    rounding: the output's to bf16 (2^-9 at most, 1.66e-3 in norm) and the weights' (2^-9 each, partly cancelled by their sum)."""
    from arcquant_amd import kv_cache
    q, k, qkv = operands(batch, seq, heads, kv_heads)
    v = qkv[:, (heads + kv_heads) * 128:]
    got = kv_cache.attention_prefill(q.cuda(), k.cuda(), qkv.cuda()[:, (heads + kv_heads) * 128:], seq).cpu().double()
    want = reference(q, k, v, seq)
    assert float((got - want).norm() / want.norm()) < 2.3e-3
    # a weight's error of 2^-9 of itself moves the result by 2^-9 of the weighted magnitudes, which abs() bounds; and the output's own
    bound = reference(q, k, v.abs(), seq) * 2 ** -8 + want.abs() * 2 ** -8 + 1e-30
    assert bool(((got - want).abs() <= bound).all())
    first = got.view(batch, seq, heads, 128)[:, 0]                  # the first token sees itself alone: its V, unchanged
    assert torch.equal(first, v.double().view(batch, seq, kv_heads, 128)[:, 0].repeat_interleave(heads // kv_heads, 1))


def test_attention_prefill_large_scores_and_order():
    """Scores of hundreds (one key takes all), equal scores (the mean), maxima that grow and fall along the keys"""
    from arcquant_amd import kv_cache
    seq, heads = 300, 2
    q, k, qkv = operands(1, seq, heads, heads, gain=40.0)
    for scale in (torch.zeros(seq, 1, 1), torch.linspace(0, 1, seq).view(-1, 1, 1), torch.linspace(1, 0, seq).view(-1, 1, 1)):
        ks = (k.float() * scale).to(torch.bfloat16)
        got = kv_cache.attention_prefill(q.cuda(), ks.cuda(), qkv.cuda()[:, 2 * heads * 128:], seq).cpu().double()
        want = reference(q, ks, qkv[:, 2 * heads * 128:], seq)
        assert float((got - want).norm() / want.norm()) < 2.3e-3


def test_attention_prefill_minus_infinite_scores():
    """An infinity among the keys that makes a query's scores -inf: no weight for that key, also where it is all that a query has seen
    in its first tile of 64 keys; no other query of the wave is touched, and a query that sees nothing else is NaN"""
    from arcquant_amd import kv_cache
    seq, heads, hidden = 200, 2, 70
    q, k, qkv = operands(1, seq, heads, heads)
    q[..., 5] = torch.where(torch.arange(seq).view(-1, 1) % 2 == 0, 1.0, -1.0)      # even queries see -inf, odd ones +inf
    for first in (0, 3):
        kk = k.clone()
        kk[first:hidden, :, 5] = float("-inf")
        got = kv_cache.attention_prefill(q.cuda(), kk.cuda(), qkv.cuda()[:, 2 * heads * 128:], seq).cpu().double().view(seq, -1)
        want = reference(q, kk, qkv[:, 2 * heads * 128:], seq).view(seq, -1)        # (NaN where the kernel documents it)
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        ok = ~torch.isnan(want).any(1)
        assert int(ok.sum()) == (65 if first == 0 else 65 + 3 + 33) and bool(ok[198]) and not bool(ok[199])
        assert float((got[ok] - want[ok]).norm() / want[ok].norm()) < 2.3e-3


def test_attention_prefill_refuses():
    """what the kernel does not take is left to torch, and refused by the entry point"""
    from arcquant_amd import _lib, kv_cache
    q, k, qkv = operands(1, 8, 4, 2)
    v = qkv[:, 6 * 128:]
    q, k, v = q.cuda(), k.cuda(), v.cuda()
    assert kv_cache.attention_prefill(q.half(), k, v, 8) is None
    assert kv_cache.attention_prefill(q[:, :3].contiguous(), k, v, 8) is None       # 3 heads over 2
    assert kv_cache.attention_prefill(q.transpose(0, 1).contiguous().transpose(0, 1), k, v, 8) is None
    ok, f = 0x1000, _lib.lib().arcq_attention_prefill
    good = dict(q=ok, ldq=512, k=ok, ldk=256, v=ok, ldv=256, b=0, s=8, h=4, g=2, d=128, c=0.1, o=ok, ldo=512)
    call = lambda **kw: f(*{**good, **kw}.values(), None)
    assert call() == 0 and call(b=1, s=0) == 0
    assert call(d=64) == 2 and call(h=3) == 2 and call(ldq=511) == 2 and call(ldv=260) == 2 and call(ldk=128) == 2 and call(g=0) == 2
    for c in (0.0, -0.1, float("inf"), float("-inf"), float("nan"), 3e38):             # 3e38 log2 e is not finite
        assert call(c=c) == 2
    assert call(b=1, q=None) == 1 and call(b=1, v=0x1008) == 4 and call(b=1, s=1 << 23, ldk=512) == 2


@pytest.mark.parametrize("batch,seq,heads,kv_heads,positions", [(1, 1, 1, 1, 1), (3, 2, 4, 4, 8), (2, 33, 4, 2, 33), (1, 127, 8, 8, 100), (2, 128, 6, 2, 128),
                                                                (3, 129, 8, 1, 4096), (1, 257, 28, 4, 300)])
def test_attention_prefill_rotates_queries(batch, seq, heads, kv_heads, positions):
    """Queries rotated by the attention itself, read from the projection's rows: the bits of the rotary pass followed by the attention,
    also behind the table's last position (which stands for every later one)"""
    from arcquant_amd import _lib, kv_cache
    _, _, qkv = operands(batch, seq, heads, kv_heads)
    qkv = torch.cat([qkv, qkv[:, :8]], 1).cuda()                    # rows that end behind the heads
    qkv[0, :2] = torch.tensor([float("nan"), 0.0])                  # what is not finite stays where it was
    tables = kv_cache.rope_tables(positions, 128, torch.bfloat16, "cuda")
    q, k = kv_cache.rope(qkv, seq, 0, heads, kv_heads, *tables)
    rows, v = qkv[:, :heads * 128], qkv[:, (heads + kv_heads) * 128:(heads + 2 * kv_heads) * 128]
    want = kv_cache.attention_prefill(q, k, v, seq)
    got = kv_cache.attention_prefill((rows, *tables), k, v, seq)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())
    assert kv_cache.attention_prefill((rows.half(), *tables), k, v, seq) is None
    assert kv_cache.attention_prefill((rows, tables[0][:, :32], tables[1]), k, v, seq) is None
    assert kv_cache.attention_prefill((rows[:, :64], *tables), k, v, seq) is None
    ok, f = 0x1000, _lib.lib().arcq_attention_prefill_rope
    args = lambda cos, n: (ok, 128, cos, ok, n, ok, 128, ok, 128, 1, 1, 1, 1, 128, 1.0, ok, 128, None)
    null, shape, align = (f(*args(*a)) for a in ((None, 1), (ok, 0), (ok + 2, 1)))
    assert len({null, shape, align}) == 3 and 0 not in (null, shape, align)      # refused ahead of any launch
