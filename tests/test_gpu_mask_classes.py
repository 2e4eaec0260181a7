"""The classes of mask rows where rows are no whole number of 16 bytes: a single value that is not what the plain form has is seen,
wherever it lies."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows whose ends lie at every place of a 16-byte piece, lengths around them, a mask off the 16-byte boundaries
@pytest.mark.parametrize("S", [65, 67, 70, 73, 101, 127, 891])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_one_value_off(S, dtype, shift):
    from effective_transformer_amd import kernel_ops as ko, ops
    gen = torch.Generator(device="cuda").manual_seed(S + shift)
    B, heads, d = (12 if S > 500 else 96), 1, 64
    lens = torch.randint(17, S + 1, (B,), generator=torch.Generator().manual_seed(S))
    lens[0], lens[1] = S, S - 1
    T = int(lens.sum())
    pos = torch.cat([torch.arange(n) for n in lens]).int()
    seq = torch.repeat_interleave(torch.arange(B), lens).int()
    bidx, widx = torch.zeros(B * S, dtype=torch.int32), torch.zeros(B * S, dtype=torch.int32)
    bidx[:T], widx[:T] = seq, pos
    qkv = torch.randn(T, 3 * d, device="cuda", generator=gen).to(dtype)
    room = torch.zeros(B * S * S + 8, device="cuda", dtype=dtype)
    mask = room[shift:shift + B * S * S].view(B, S, S)
    mask.copy_((torch.arange(S)[None, None] < lens[:, None, None]).expand(B, S, S).to(dtype))
    # one value of one row of every sequence: at the start and the end of a row, of a block's rows, and around the last token
    for b in range(B):
        n = int(lens[b])
        row = [0, 15, 7, min(16, n - 1), n - 1][b % 5]
        key = [0, n - 1, min(n, S - 1), S - 1, b * 5 % S, 1, S - 2][b % 7]
        mask[b, row, key] = 1 - mask[b, row, key]

    count, bidx, widx = torch.tensor([T], dtype=torch.int32, device="cuda"), bidx.cuda(), widx.cuda()
    args = (qkv[:, :d], qkv[:, d:2 * d], qkv[:, 2 * d:], 1, 3 * d, mask, count, B, S, heads, d, bidx, widx)
    starts = ops.sequence_starts(count, bidx, B, S)
    assert torch.equal(ko.attention(*args)[:T], ko.attention(*args, seq_start=starts)[:T])      # the second one reads every row of the mask
