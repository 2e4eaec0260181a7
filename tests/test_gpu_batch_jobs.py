"""What a layer makes of its batch in the launch that prepares its weights (sequence table, classes of the mask rows) against the
same layer with a table handed over, whose classes come from a launch of their own."""
import pytest
import torch

from effective_transformer_amd import ops

pytestmark = pytest.mark.gpu


# more rows than one block reads in full (2048): 256 and 257 sequences (32 probes for one per thread, 8 for four), 1024 and 1025
# (searched for, and the starts by many blocks); positions with and without classes, sequences without a token in front, in a row
# and at the end, hidden sizes on split rows and on pair rows
@pytest.mark.parametrize("B,S,H,empty", [(256, 17, 64, False), (257, 17, 64, True), (1024, 5, 64, True), (1025, 5, 64, True), (3, 1024, 64, True),
                                         (40, 130, 64, True), (20, 130, 512, True), (70, 66, 64, False), (9, 300, 512, False)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("causal", [False, True])
def test_same_bits_as_with_a_table(B, S, H, empty, dtype, causal):
    print("batch jobs", B, S, H, empty, dtype, causal, flush=True)
    heads = H // 64
    g = torch.Generator(device="cuda").manual_seed(B + S)
    lens = torch.randint(max(1, 3 * S // 4), S + 1, (B,), device="cuda", generator=g)
    if empty:
        lens[0] = lens[-1] = lens[B // 2] = lens[B // 2 - 1] = 0
    mask = (torch.arange(S, device="cuda")[None] < lens[:, None]).to(torch.int32)
    if not causal:
        mask[:, ::7] &= (torch.rand(B, (S + 6) // 7, device="cuda", generator=g) < 0.8).int()       # holes
    attn = mask[:, None].expand(B, S, S).to(dtype).contiguous()
    if causal:
        attn = (attn * torch.ones(S, S, device="cuda", dtype=dtype).tril()).contiguous()
    shapes = [(H, H), (H,)] * 4 + [(H,)] * 2 + [(H, 4 * H), (4 * H,), (4 * H, H), (H,)] + [(H,)] * 2
    flat = [(torch.randn(s, device="cuda", generator=g) * 0.1).to(dtype) for s in shapes]
    x = torch.randn(B, S, H, device="cuda", generator=g).to(dtype)
    packed, vwn, bidx, widx = ops.effective_transformer_input(x, mask, B, S, S, heads, 64)
    count = int(mask.sum())
    table = ops.sequence_starts(vwn, bidx, B, S)
    w = ops.LayerWeights.from_slots(x.device, dtype, flat)
    args = (packed, packed, attn, vwn, bidx, widx, w, B, S, S, heads, 64)
    want = ops.effective_transformer(*args, seq_start=table).view(B * S, H)[:count].clone()
    assert torch.isfinite(want).all()
    assert torch.equal(ops.effective_transformer(*args).view(B * S, H)[:count], want)
    assert torch.equal(ops.effective_transformer(*args, valid_word_num_hint=count).view(B * S, H)[:count], want)
