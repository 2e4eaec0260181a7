"""Attention launches of many workgroups, where blocks of queries without tokens come last: every sequence as it comes out alone."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _valid(B, S, kind, gen):
    """[B, S]: tokens at the start of each sequence, or with holes; some sequences without any."""
    lens = torch.randint(0, S // 4, (B,), generator=gen)
    lens[0], lens[B // 2], lens[-1] = S, 0, 1
    lens[1::5] = torch.randint(S // 2, S + 1, (len(lens[1::5]),), generator=gen)
    at = torch.arange(S)[None]
    if kind == "dense":
        return at < lens[:, None]
    # as many tokens, far apart: the last ones' queries lie in blocks behind what the count of tokens fills
    step = (S // lens.clamp(min=1)).clamp(max=3)[:, None]
    return (at % step == 0) & (at // step < lens[:, None])


# grids above 1024 workgroups with up to 64 sequences, heads that the XCDs do not share evenly, one sequence more, and fewer
@pytest.mark.parametrize("B,heads,S", [(64, 12, 300), (63, 5, 513), (64, 16, 129), (17, 13, 1024), (40, 3, 1000), (65, 12, 300), (5, 3, 300)])
@pytest.mark.parametrize("kind", ["dense", "holes"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_sequences_alone_and_together(B, heads, S, kind, dtype):
    from effective_transformer_amd import kernel_ops as k
    gen = torch.Generator().manual_seed(B * S + heads)
    valid = _valid(B, S, kind, gen)
    d, H = 64, heads * 64
    b_idx, w_idx = (t.int() for t in valid.nonzero(as_tuple=True))
    T = len(b_idx)
    qkv = torch.randn(T, 3 * H, generator=gen).to(dtype).cuda()
    attr = valid[:, None, :].expand(B, S, S).to(dtype).contiguous().cuda()

    def run(x, mask, b, w):
        n = torch.tensor([len(b)], dtype=torch.int32).cuda()
        out = torch.full((mask.shape[0] * S, H), 7.0, dtype=dtype, device="cuda")
        return k.attention(x[:, :H], x[:, H:2 * H], x[:, 2 * H:], 1, 3 * H, mask, n, mask.shape[0], S, heads, d, b.cuda(), w.cuda(), dst=out)
    got = run(qkv, attr, b_idx, w_idx)
    assert (got[T:] == 7.0).all() and not (got[:T] == 7.0).all(dim=1).any()
    for b in sorted({0, 1, 2, B // 2 - 1, B - 2, B - 1}):
        rows = (b_idx == b).nonzero()[:, 0]
        if len(rows) == 0:
            continue
        alone = run(qkv[rows.cuda()].contiguous(), attr[b:b + 1], torch.zeros(len(rows), dtype=torch.int32), w_idx[rows])
        assert torch.equal(alone[:len(rows)], got[rows.cuda()]), "sequence %d" % b
