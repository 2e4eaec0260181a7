"""fp32 attention on operands that three bfloat16 pieces do not hold, which beyond 32 positions run on the float instructions: magnitudes
far from 1, infinities, the largest float, exponentials far below the largest."""
import math

import pytest
import torch

import test_gpu_head_exponents as layers
from test_gpu_attention_f32 import _reference

pytestmark = pytest.mark.gpu


# The floats are powers of two apart from those of an ordinary head: Q and K by the factors' product, V by its own.  Below 2^-110
# a float is more than its three pieces, and from 3.4e38 on its first one is infinite; the last head always is an ordinary one.
@pytest.mark.parametrize("q_by,k_by,v_by", [(0, 0, -110), (0, 0, -118), (0, 0, -124), (-120, 120, 0), (120, -120, 0),
                                            (-116, 116, -116), (0, 0, 116)])
@pytest.mark.parametrize("S", [33, 63, 64, 65, 97, 379, 1023, 1024])
@pytest.mark.parametrize("holes", [False, True])
@pytest.mark.parametrize("form", ["plain", "causal"])
def test_powers_of_two(S, holes, form, q_by, k_by, v_by):
    from effective_transformer_amd import kernel_ops as k
    B, heads, d = 3, 2, 64
    H = heads * d
    gen = torch.Generator().manual_seed(S * 4 + holes * 2 + (form == "causal"))
    lens = torch.tensor([S, max(1, S // 2 + 1), 1])
    valid = torch.arange(S)[None] < lens[:, None]
    if holes:
        valid &= torch.rand(B, S, generator=gen) < 0.8
        valid[:, 0] = True
    b_idx, w_idx = (t.int() for t in valid.nonzero(as_tuple=True))
    T = len(b_idx)
    attr = valid[:, None, :].expand(B, S, S).float()
    if form == "causal":
        attr = attr * torch.tril(torch.ones(S, S))
    attr = attr.contiguous()
    qkv = torch.randn(T, 3 * H, generator=gen)
    qkv[:, :H] *= 3.0
    for part, by in enumerate((q_by, k_by, v_by)):
        qkv[:, part * H:part * H + d] *= 2.0 ** by
    dev = [t.cuda() for t in (qkv, attr, b_idx, w_idx)]
    x = dev[0]
    got = k.attention(x[:, :H], x[:, H:2 * H], x[:, 2 * H:], 1, 3 * H, dev[1], torch.tensor([T], dtype=torch.int32).cuda(), B, S, heads,
                      d, dev[2], dev[3])[:T].double().cpu()
    for b in range(B):
        rows = (b_idx == b).nonzero()[:, 0]
        at = w_idx[rows].long()
        for h in range(heads):
            col = slice(h * d, (h + 1) * d)
            # keys without a token have zero rows and are in the mask like the others
            full = torch.zeros(2, S, d)
            full[0, at], full[1, at] = qkv[rows, H:2 * H][:, col], qkv[rows, 2 * H:][:, col]
            want, bound = _reference(qkv[rows, :H][:, col], full[0], full[1], attr[b][at])
            # (a sum of up to S floats may end half a step of the smallest ones off at each of them)
            over = ((got[rows][:, col] - want).abs() / (bound + S * 2.0 ** -150)).max().item()
            assert over < 1.0, "sequence %d head %d: %g of the bound" % (b, h, over)


def _one_head(q, k, v, attr, S):
    """Attention of one head over one sequence without holes, from packed rows."""
    from effective_transformer_amd import kernel_ops as ops
    n = len(q)
    x = torch.cat([q, k, v], dim=1).cuda()
    at = torch.arange(n, dtype=torch.int32).cuda()
    return ops.attention(x[:, :64], x[:, 64:128], x[:, 128:], 1, 192, attr[None].cuda(), torch.tensor([n], dtype=torch.int32).cuda(), 1, S, 1,
                         64, torch.zeros_like(at), at)[:n].double().cpu()


@pytest.mark.parametrize("S", [20, 33, 100, 379, 1024])
@pytest.mark.parametrize("form", ["plain", "causal"])
def test_infinities_and_the_largest_floats(S, form):
    """What the float instructions make of them: an infinity of V is the result of the queries that see it and of its feature alone,
    a key whose score is -infinity weighs nothing, a float of 3.4e38 stays one."""
    gen = torch.Generator().manual_seed(S)
    n = S - 1
    q, k, v = (torch.randn(n, 64, generator=gen) for _ in range(3))
    q[:, 0] = q[:, 0].abs() + 0.1
    attr = torch.zeros(S, S)
    attr[:, :n] = 1
    if form == "causal":
        attr = attr * torch.tril(torch.ones(S, S))
    seen = attr[:n, :n].bool()
    want, bound = _reference(q, k, v, attr[:n, :n])

    hidden = k.clone()
    hidden[n // 3, 0] = float("-inf")                 # as if that key were masked for everybody
    mask = attr[:n, :n].clone()
    mask[:, n // 3] = 0
    low, low_bound = _reference(q, k, v, mask)
    rows = mask.sum(dim=1) > 0
    got = _one_head(q, hidden, v, attr, S)
    assert ((got - low).abs() <= low_bound)[rows].all()

    high = v.clone()
    high[n // 2, 5] = float("inf")
    got = _one_head(q, k, high, attr, S)
    others = torch.arange(64) != 5
    assert ((got - want).abs() <= bound)[:, others].all()
    assert (got[seen[:, n // 2], 5] == float("inf")).all()

    top = torch.finfo(torch.float32).max
    alone = torch.zeros(S, S)
    alone[:, 0] = 1
    got = _one_head(q[:1], k[:1], torch.full((1, 64), top), alone, S)
    score = (q[0] @ k[0]).double().item() / 8
    share = 1 / (1 + 1e-6 * math.exp(-min(score, 0)) if S < 1024 else 1 + 1e-6)
    assert ((got / (top * share) - 1).abs() < 2.0 ** -20).all()


@pytest.mark.parametrize("S", [33, 100, 1024])
def test_weights_far_below_the_largest(S):
    """The result of a feature that only keys of little weight have: their exponentials down to 2^-125 of the largest keep the
    floats' bits (the exponent of 125 is held to 2^-18, the score of 87 to 2^-18)."""
    n = 32
    q, k, v = torch.zeros(n, 64), torch.zeros(n, 64), torch.zeros(n, 64)
    q[:, 0] = 8.0
    k[1:, 0] = -torch.linspace(50.0, 86.5, n - 1)
    v[torch.arange(1, n), torch.arange(1, n)] = 1.2345
    attr = torch.zeros(S, S)
    attr[:, :n] = 1
    got = _one_head(q, k, v, attr, S)[:, 1:n]
    e = k[1:, 0].double().exp()
    want = 1.2345 * e / (1 + e.sum() + 1e-6)
    assert ((got / want - 1).abs() < 2.0 ** -16).all(), ((got / want - 1).abs().max().item())


def test_other_sequences_keep_their_bits():
    """A sequence that needs the float instructions changes nothing for its neighbours."""
    from effective_transformer_amd import kernel_ops as k
    B, S, H = 5, 130, 128
    gen = torch.Generator().manual_seed(3)
    x = torch.randn(B * S, 3 * H, generator=gen)
    b_idx = torch.arange(B, dtype=torch.int32).repeat_interleave(S).cuda()
    w_idx = torch.arange(S, dtype=torch.int32).repeat(B).cuda()
    attr = torch.ones(B, S, S).cuda()

    def run(t):
        t = t.cuda()
        return k.attention(t[:, :H], t[:, H:2 * H], t[:, 2 * H:], 1, 3 * H, attr, torch.tensor([B * S], dtype=torch.int32).cuda(), B, S, 2,
                           64, b_idx, w_idx).cpu().view(B, S, 2, 64)
    plain = run(x)
    odd = x.clone()
    odd[2 * S + 7, 2 * H + 64 + 3] = 2.0 ** -120 * 1.2345     # sequence 2, head 1
    got = run(odd)
    keep = torch.ones(B, 2, dtype=torch.bool)
    keep[2, 1] = False
    at = keep[:, None, :].expand(B, S, 2)
    assert torch.equal(got[at], plain[at])
    assert not torch.equal(got[2, :, 1], plain[2, :, 1])


@pytest.mark.parametrize("heads,S,B", [(8, 40, 3), (12, 65, 70)])
def test_layers_whose_context_leaves_as_pair_rows(heads, S, B):
    """A head whose Q is 2^70 and K 2^-70 of the others': its blocks run on the float instructions and store pair rows.  The bound is
    that of layers on ordinary heads: an error of 2^-22 per product of the layer's four, each of a row's size after the norms."""
    w = layers._layer(heads, 64, heads)
    x = torch.randn(B, S, heads * 64, generator=torch.Generator().manual_seed(B))
    col = slice(64, 128)
    for i, by in ((0, 2.0 ** 70), (2, 2.0 ** -70)):
        w[i][:, col] *= by
        w[i + 1][col] *= by
    got = layers._run(x, w, heads, 64)[B - 1].double()
    want = layers._reference(x[B - 1:], w, heads, 64)[0]
    assert ((got - want).norm(dim=1) / want.norm(dim=1)).max() < 8 * 2.0 ** -22
