"""A layer called without a sequence table makes its own, up to a size in one block of its first launch."""
import pytest
import torch

from effective_transformer_amd import ops

pytestmark = pytest.mark.gpu


# around what one block takes (2303 sequences, 2048 rows), fewer rows than a block has threads, sequences without a token
# in front, in between and at the end; weights handed over as they are or prepared
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("B,S,empty", [(1, 1, False), (3, 40, True), (217, 53, True), (2047, 1, False), (2304, 1, True), (128, 16, False),
                                       (38, 54, True), (31, 66, False)])
def test_same_bits_as_with_a_table(B, S, empty, dtype):
    print("sequence table", B, S, empty, dtype, flush=True)
    heads, H = 1, 64
    g = torch.Generator(device="cuda").manual_seed(B)
    lens = torch.randint(1, S + 1, (B,), device="cuda", generator=g)
    if empty:
        lens[0] = lens[-1] = lens[B // 2] = 0
    mask = (torch.arange(S, device="cuda")[None] < lens[:, None]).to(torch.int32)
    attn = mask[:, None].expand(B, S, S).to(dtype).contiguous()
    shapes = [(H, H), (H,)] * 4 + [(H,)] * 2 + [(H, 4 * H), (4 * H,), (4 * H, H), (H,)] + [(H,)] * 2
    flat = [(torch.randn(s, device="cuda", generator=g) * 0.1).to(dtype) for s in shapes]
    x = torch.randn(B, S, H, device="cuda", generator=g).to(dtype)
    packed, vwn, bidx, widx = ops.effective_transformer_input(x, mask, B, S, S, heads, H)
    count = int(lens.sum())
    table = ops.sequence_starts(vwn, bidx, B, S)
    starts = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"), lens.cumsum(0)])
    assert torch.equal(table[:B + 1].long(), starts)
    for prepared in (False, True):
        w = ops.LayerWeights.from_slots(x.device, dtype, flat)
        if prepared:
            w.prepare()
        args = (packed, packed, attn, vwn, bidx, widx, w, B, S, S, heads, H)
        want = ops.effective_transformer(*args, seq_start=table).view(B * S, H)[:count].clone()
        assert torch.equal(ops.effective_transformer(*args).view(B * S, H)[:count], want)
        assert torch.equal(ops.effective_transformer(*args, valid_word_num_hint=count).view(B * S, H)[:count], want)
