"""fp32 attention beyond 32 positions, whose products run on three bfloat16 pieces of every float, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _reference(q, k, v, mask):
    """One head in float64: the result, and per element the bound that the test allows.

    A float is the sum of its three pieces exactly; of the nine products of pieces three are left out, together at most
    2^-23 of the product of the two floats, and the others are added in float, 12 (scores) and 6 a stage (P.V) at a time.
    A score may so be off by 2^-21 of the sum of its products' magnitudes (and by its own rounding in the softmax, 2^-22 of
    it), a probability by as much again relatively, and the sum over the keys adds 2^-20 of the magnitudes it sums."""
    q, k, v, mask = (t.double() for t in (q, k, v, mask))
    s = q @ k.T * 0.125
    size = (q.abs() @ k.abs().T * 0.125).amax(dim=1, keepdim=True)
    s = s + (1 - mask) * -10000
    m = s.amax(dim=1, keepdim=True)
    if mask.shape[-1] < 1024:
        m = m.clamp(min=0)
    e = (s - m).exp()
    p = e / (e.sum(dim=1, keepdim=True) + 1e-6)
    # (the masked scores are as large as the bias, of which a float holds 2^-24)
    off = 2.0 ** -20 * size + 2.0 ** -22 * m.abs() + 2.0 ** -20
    return p @ v, 2 * off * (p @ v.abs())


@pytest.mark.parametrize("S", [33, 63, 64, 65, 97, 379, 1023, 1024])
@pytest.mark.parametrize("holes", [False, True])
@pytest.mark.parametrize("form", ["plain", "causal"])
def test_attention(S, holes, form):
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
    qkv[:, 2 * H:2 * H + d] *= 2.0 ** 40              # a head of V far above the other
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
            over = ((got[rows][:, col] - want).abs() / bound.clamp(min=1e-300)).max().item()
            assert over < 1.0, "sequence %d head %d: %g of the bound" % (b, h, over)
