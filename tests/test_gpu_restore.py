"""The padded output from packed rows: by a search of the indices (the output op) and from the packed row of every position (the
encoder in one call), on both sides of every split, against the oracle and each other."""
import numpy as np
import pytest
import torch

from oracle import et_oracle as o

pytestmark = pytest.mark.gpu


def _mask(B, S, rng):
    """Ragged sequences with holes, empty ones among them."""
    mask = (np.arange(S)[None] < rng.randint(0, S + 1, size=B)[:, None]).astype(np.int32)
    mask[rng.randint(0, B, max(1, B // 8)), rng.randint(0, S, max(1, B // 8))] ^= 1
    mask[0, 0] = 1
    return mask


# positions that end inside a workgroup's window, 8 and 32 of them a workgroup, one chunk a row and rows of 2- and 4-byte pieces
@pytest.mark.parametrize("B,S,H", [(1, 1, 8), (3, 5, 6), (7, 9, 3), (1, 33, 768), (33, 31, 64), (127, 129, 64), (1024, 16, 24), (331, 51, 5)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_search(B, S, H, dtype):
    from effective_transformer_amd import kernel_ops as ko
    rng = np.random.RandomState(B + S + H)
    mask = _mask(B, S, rng)
    pos = np.flatnonzero(mask)
    T = len(pos)
    bi, wi = np.full(B * S, 10 ** 6, np.int32), np.full(B * S, 10 ** 6, np.int32)
    bi[:T], wi[:T] = pos // S, pos % S
    x = rng.randn(B * S, H).astype(np.float32 if dtype == torch.float32 else np.float16)
    got = ko.restore(torch.from_numpy(x).cuda(), torch.from_numpy(bi).cuda(), torch.from_numpy(wi).cuda(),
                     torch.tensor([T], dtype=torch.int32, device="cuda"), B, S)
    assert np.array_equal(got.cpu().numpy(), o.restore(x, T, bi, wi, B, S))


# two and eight chunks a lane (from 2^21 chunks on), the last workgroup part-filled, rows of 2- and 4-byte pieces; a last position of 2,
# which is no token
@pytest.mark.parametrize("B,S,heads,d,dtype", [(1, 1, 1, 64, torch.float16), (5, 13, 3, 5, torch.float16), (9, 7, 1, 1, torch.float32),
                                               (3, 43, 2, 33, torch.float16), (1, 300, 2, 64, torch.float16), (257, 32, 16, 64, torch.float32),
                                               (300, 32, 16, 64, torch.float32), (70, 16, 12, 64, torch.float16)])
@pytest.mark.parametrize("last", [0, 1, 2])
def test_packed_rows_of_positions(B, S, heads, d, dtype, last):
    from effective_transformer_amd import ops
    H = heads * d
    rng = np.random.RandomState(B + S + H + last)
    mask = _mask(B, S, rng)
    if B * S > 1:
        mask[-1, -1] = last
    gen = torch.Generator(device="cuda").manual_seed(H)

    def t(*shape):
        return torch.randn(*shape, device="cuda", dtype=torch.float32, generator=gen).mul_(0.05).to(dtype)

    w = [t(H, H), t(H), t(H, H), t(H), t(H, H), t(H), t(H, H), t(H), t(H), t(H), t(H, 4 * H), t(4 * H), t(4 * H, H), t(H), t(H), t(H)]
    enc = ops.EffectiveTransformerEncoder(1, heads, d, w, dtype, "cuda")
    x, m = t(B, S, H), torch.from_numpy(mask).cuda()
    attr = (m > 0)[:, None, :].expand(B, S, S).to(dtype).contiguous()
    h, vwn, bidx, widx = ops.effective_transformer_input(x, m, B, S, S, heads, d)
    h = ops.effective_transformer(h, h, attr, vwn, bidx, widx, enc.layers[0], B, S, S, heads, d)
    want = ops.effective_transformer_output(h, vwn, bidx, widx, B, S, S, heads, d)
    got = enc(x, m, attr)
    assert torch.equal(got, want)
    assert not got[~(m == 1)].any() and got[m == 1].abs().sum() > 0
