"""The kernels around the products of a pass over prompts, against float64 on the CPU: sizes at the edges of the 16-query
fragments, 64-key tiles and 64 / 128-query workgroups, grouped heads, caches longer than the prompt, strided operands."""
import math

import pytest
import torch

from ternaryllm_amd import ops
from ternaryllm_amd.attention import apply_rope, rope_tables

pytestmark = pytest.mark.gpu


def reference(q, k, v):
    """q [B, S, heads, hd], k, v [B, kv_heads, L, hd] on the CPU; float64."""
    q, k, v = q.double().transpose(1, 2), k.double(), v.double()
    k, v = (t.repeat_interleave(q.shape[1] // k.shape[1], dim=1) for t in (k, v))
    S, L = q.shape[2], k.shape[2]
    scores = (q @ k.transpose(2, 3)) / math.sqrt(q.shape[3])
    scores = scores.masked_fill(~torch.ones((S, L), dtype=torch.bool).tril(L - S), float("-inf"))
    return (torch.softmax(scores, -1) @ v).transpose(1, 2).reshape(q.shape[0], S, -1)


@pytest.mark.parametrize("B,heads,kv_heads,hd,S,L", [
    (1, 1, 1, 128, 1, 1), (2, 3, 1, 128, 15, 15), (1, 4, 2, 64, 16, 17), (2, 2, 2, 128, 63, 63), (1, 2, 2, 64, 64, 64), (1, 2, 1, 128, 65, 129),
    (2, 8, 8, 64, 127, 127), (1, 8, 4, 128, 129, 200), (3, 5, 5, 128, 200, 200), (1, 2, 2, 128, 1, 300), (1, 2, 2, 64, 3, 131),
    (4, 64, 32, 128, 130, 130), (4, 64, 64, 64, 257, 260), (1, 2, 2, 128, 700, 700)])
@pytest.mark.parametrize("rotate", [False, True])
def test_attention(B, heads, kv_heads, hd, S, L, rotate):
    g = torch.Generator().manual_seed(S * 1000 + L)
    qkv = torch.randn((B, S, heads + 2, hd), generator=g).half()    # queries as a view among other heads
    k, v = (torch.randn((B, kv_heads, L + 9, hd), generator=g).half() for _ in range(2))
    q, kc, vc = qkv.cuda()[:, :, 1:-1], k.cuda()[:, :, :L], v.cuda()[:, :, :L]
    rotated, tables = qkv[:, :, 1:-1], None
    if rotate:
        cos, sin = rope_tables(torch.arange(S), hd, 10000.0, torch.float16, "cpu")
        tables = cos.cuda(), sin.cuda()
        rotated = apply_rope(rotated.transpose(1, 2).float(), cos.float(), sin.float()).half().transpose(1, 2)
    out = ops.prefill_attention(q, kc, vc, tables).cpu().double()
    want = reference(rotated, k[:, :, :L], v[:, :, :L])
    # probabilities and the result are each rounded to 11 bits: 2 * 2^-11 of the largest value, and half as much again
    # for a rotated query that rounds to its other neighbour
    assert (out - want).abs().max() <= 1.5 * 2.0 ** -10 * v.abs().max()


# heads of 128 where workgroups own 128 queries (768 of them are three for each of 256 compute units): a last workgroup with two queries
# and one with nine, more keys than queries, grouped heads
@pytest.mark.parametrize("B,heads,kv_heads,hd,S,L", [(6, 64, 32, 128, 130, 130), (6, 64, 16, 128, 137, 200), (13, 60, 60, 128, 64, 131)])
@pytest.mark.parametrize("rotate", [False, True])
def test_attention_of_tall_workgroups(B, heads, kv_heads, hd, S, L, rotate):
    test_attention(B, heads, kv_heads, hd, S, L, rotate)


def test_attention_values_that_are_not_finite():
    """A row past the end of the keys and a key of -inf scores weigh nothing; NaN reaches the queries that see it, and only
    those outside its tile of keys are sure not to."""
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn((1, 70, 2, 64), generator=g).half(), torch.randn((1, 2, 80, 64), generator=g).half(), torch.randn((1, 2, 80, 64), generator=g).half())
    k[:, :, 70:], v[:, :, 70:] = float("nan"), float("inf")
    q[..., 0] = q[..., 0].abs() + 0.5
    k[:, :, :64, 0] = float("-inf")                                  # a whole tile of keys without weight, for queries 64 on
    out = ops.prefill_attention(q.cuda(), k.cuda()[:, :, :70], v.cuda()[:, :, :70]).cpu().double()
    want = reference(q, k[:, :, :70], v[:, :, :70])
    assert torch.isnan(out[:, :64]).all() and torch.isnan(want[:, :64]).all()
    assert (out[:, 64:] - want[:, 64:]).abs().max() <= 1.5 * 2.0 ** -10 * v[:, :, :70].abs().max()


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,S,heads,hd,per_row", [(1, 1, 1, 16, False), (2, 37, 3, 64, True), (3, 65, 5, 128, False)])
def test_rope_rows(dtype, B, S, heads, hd, per_row):
    g = torch.Generator().manual_seed(3)
    qkv = torch.randn((B, S, 3, heads, hd), generator=g).to(dtype)
    tables = [torch.randn((B, S, hd) if per_row else (S, hd), generator=g).to(dtype) for _ in range(2)]
    kc, vc = torch.zeros((2, B, heads, S + 5, hd), dtype=dtype, device="cuda").unbind(0)
    dev = qkv.cuda()
    ops.rope_rows(dev[:, :, 1], [t.cuda() for t in tables], kc[:, :, :S], dev[:, :, 2], vc[:, :, :S])
    want = apply_rope(qkv[:, :, 1].transpose(1, 2).double(), *[t.double() for t in tables])
    # one rounding of x * cos in fp32, of the sum, and of the result
    eps = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -23
    bound = 2 * eps * (qkv.double().abs().max() * sum(t.double().abs().max() for t in tables))
    assert (kc[:, :, :S].cpu().double() - want).abs().max() <= bound
    assert torch.equal(vc[:, :, :S].cpu(), qkv[:, :, 2].transpose(1, 2))
    assert not kc[:, :, S:].any() and not vc[:, :, S:].any()


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_rope_table(dtype):
    cos, sin = ops.rope_table(5, 300, 128, 10000.0, dtype, torch.device("cuda:0"))
    want = rope_tables(torch.arange(5, 305).double(), 128, 10000.0, torch.float64, "cpu")
    # the angle is up to 305, rounded to fp32 after a power and a product of a few units in the last place each
    bound = 305 * 8 * 2.0 ** -24 + (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -22)
    for got, t in zip((cos, sin), want):
        assert (got.cpu().double() - t).abs().max() <= bound


def test_misaligned_and_odd_operands_are_refused():
    q = torch.zeros((1, 4, 2, 64), dtype=torch.float16, device="cuda")
    k = torch.zeros((1, 2, 4, 64), dtype=torch.float16, device="cuda")
    odd = torch.zeros(1 * 2 * 4 * 64 + 1, dtype=torch.float16, device="cuda")[1:].view(1, 2, 4, 64)
    assert not ops.in_pieces(odd) and ops.in_pieces(k)
    with pytest.raises((ValueError, RuntimeError)):
        ops.prefill_attention(q, odd, k)
    with pytest.raises((ValueError, RuntimeError)):
        ops.prefill_attention(q, k[:, :, :3], k[:, :, :3])   # fewer keys than queries
    with pytest.raises((ValueError, RuntimeError)):
        ops.prefill_attention(q.float(), k.float(), k.float())
