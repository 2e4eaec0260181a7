"""fp32 layers whose context rows have an exponent per head: the output product at the edges of its tiles and heads."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(heads, d, seed):
    H = heads * d
    gen = torch.Generator().manual_seed(seed)

    def kernel(k, n):
        return torch.randn(k, n, generator=gen) * k ** -0.5
    w = []
    for _ in range(4):
        w += [kernel(H, H), torch.randn(H, generator=gen) * 0.1]
    w += [torch.randn(H, generator=gen) * 0.1, torch.ones(H)]
    w += [kernel(H, 4 * H), torch.randn(4 * H, generator=gen) * 0.1, kernel(4 * H, H), torch.randn(H, generator=gen) * 0.1]
    return w + [torch.randn(H, generator=gen) * 0.1, torch.ones(H)]


def _spread_heads(w, heads, d):
    """Heads of V from 2^-6 to 2^6 of the others', taken back by their rows of the output kernel (whose columns have one exponent:
    values 2^-16 of a column's largest would lose bits)."""
    by = 2.0 ** ((torch.arange(heads) * 7) % 13 - 6).repeat_interleave(d)
    w[4], w[5], w[6] = w[4] * by, w[5] * by, w[6] / by[:, None]
    return w


def _reference(x, w, heads, d):
    """The layer in float64; all positions of x hold tokens."""
    x, w = x.double(), [t.double() for t in w]
    B, S, H = x.shape
    q, k, v = ((x @ w[2 * i] + w[2 * i + 1]).view(B, S, heads, d).transpose(1, 2) for i in range(3))
    s = q @ k.transpose(-1, -2) * d ** -0.5
    top = s.amax(-1, keepdim=True).clamp(min=0)
    e = (s - top).exp()
    c = (e / (e.sum(-1, keepdim=True) + 1e-6)) @ v

    def norm(t, beta, gamma):
        return (t - t.mean(-1, keepdim=True)) / (t.var(-1, unbiased=False, keepdim=True) + 1e-6).sqrt() * gamma + beta
    a = norm(c.transpose(1, 2).reshape(B, S, H) @ w[6] + w[7] + x, w[8], w[9])
    u = a @ w[10] + w[11]
    u = 0.5 * u * (1 + torch.tanh(0.7978845608028654 * (u + 0.044715 * u ** 3)))
    return norm(u @ w[12] + w[13] + a, w[14], w[15])


def _run(x, w, heads, d):
    from effective_transformer_amd import ops
    B, S, _ = x.shape
    enc = ops.EffectiveTransformerEncoder(1, heads, d, [t.cuda() for t in w], torch.float32, "cuda")
    return enc(x.cuda(), torch.ones(B, S, dtype=torch.int32).cuda(), torch.ones(B, S, S).cuda()).cpu()


# batches whose rows take the tiles of 32 to 256 rows, one and several to a workgroup, with remainders; 8 to 32 heads
@pytest.mark.parametrize("heads,S,B", [(8, 31, 1), (8, 40, 3), (8, 33, 41), (12, 31, 40), (12, 65, 70), (8, 65, 150), (8, 64, 420),
                                       (12, 40, 520), (16, 50, 130), (29, 33, 40), (31, 40, 110), (32, 40, 150)])
def test_rows_have_their_bits_in_every_batch(heads, S, B):
    """A sequence alone takes the smallest tiles; its rows must come out the same in a batch, and near float64: an error of 2^-22
    per product of the layer's four, each of a row's size after the norms."""
    w = _spread_heads(_layer(heads, 64, heads), heads, 64)
    x = torch.randn(B, S, heads * 64, generator=torch.Generator().manual_seed(B))
    got = _run(x, w, heads, 64)
    for b in sorted({0, B // 2, B - 1}):
        alone = _run(x[b:b + 1], w, heads, 64)
        assert torch.equal(alone[0], got[b]), "sequence %d" % b
    want = _reference(x[B - 1:], w, heads, 64)[0]
    err = (got[B - 1].double() - want).norm(dim=1) / want.norm(dim=1)
    assert err.max() < 8 * 2.0 ** -22, err.max().item()


def test_heads_of_another_size_have_rows_paired_as_a_whole():
    w = _layer(16, 48, 5)
    x = torch.randn(3, 37, 768, generator=torch.Generator().manual_seed(9))
    got, want = _run(x, w, 16, 48), _reference(x, w, 16, 48)
    assert ((got.double() - want).norm(dim=2) / want.norm(dim=2)).max() < 8 * 2.0 ** -22
