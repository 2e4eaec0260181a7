"""Masks that look at keys behind a sequence's last token, or nowhere at all: the streaming attention kernels run no stage there,
and take what the mask says of those keys from its classes (layers) or from its rows (et_attention, which has no classes)."""
import numpy as np
import pytest
import torch

from effective_transformer_amd import kernel_ops, ops
from effective_transformer_amd.sample.workloads import Workload, make_layer_weights
from gpu_util import dev, run_encoder
from oracle import et_oracle as o

pytestmark = pytest.mark.gpu

FORMS = 8


def _attr(form, mask, rng):
    """[S,S] of one sequence whose tokens are `mask`."""
    S = len(mask)
    n = int(np.nonzero(mask)[0].max()) + 1
    keys = np.broadcast_to(mask[None], (S, S)).astype(np.float32)
    a = keys.copy()
    if form == 0:
        a = np.tril(a)                                       # causal: 0 behind the tokens
    elif form == 1:
        a = np.ones((S, S), np.float32)                      # every key: 1 behind the tokens
    elif form == 2:
        a[:, S - 1] = 1                                      # one key there, the last
    elif form == 3:
        a = (rng.random_sample((S, S)) < 0.7).astype(np.float32)
    elif form == 4:
        a[:] = 0                                             # nobody: the tokens masked like the rest
    elif form == 5:
        a[: n // 2, n:] = 1                                  # 1 there for the first queries, 0 for the others
    elif form == 6:
        a = np.tril(a)
        a[n // 3:, (n + S) // 2:] = rng.random_sample((S - n // 3, S - (n + S) // 2)) < 0.5
    else:
        a[n // 2:, n // 3] = 0.25                            # a weight in between, among the tokens
    return a


# lengths around a stage of 64 (fp32: 32) keys and the 256 (128) keys whose masks are looked at together; rows of a mask on
# 16-byte boundaries and odd ones
@pytest.mark.parametrize("shift", [0, 3])
@pytest.mark.parametrize("S,dtype", [(S, "fp16") for S in (65, 200, 257, 509, 512, 1023, 1024)] +
                         [(S, "fp32") for S in (33, 64, 150, 333, 512, 1021, 1024)])
def test_masks_behind_the_tokens(S, dtype, shift):
    print("masks behind the tokens", S, dtype, shift, flush=True)
    el = np.float16 if dtype == "fp16" else np.float32
    rng = np.random.RandomState(S + shift)
    lens = np.minimum([1, 63, 64, 65, S // 2, S - 1, S, 20], S)
    B = len(lens)
    mask = (np.arange(S)[None] < lens[:, None]).astype(np.int32)
    mask[4, S // 8:S // 4] = 0                               # a hole
    attr = np.stack([_attr((b + shift) % FORMS, mask[b], rng) for b in range(B)]).astype(el)

    # et_attention, packed rows, one head
    _, T, bi, wi, _ = o.input_op_fast(np.zeros((B, S, 1), np.float32), mask)
    qkv = o.rnd(rng.randn(T, 192), dtype)
    zero = np.zeros(64, el)
    q, k, v = np.ascontiguousarray(qkv[:, :64]), np.ascontiguousarray(qkv[:, 64:128]), np.ascontiguousarray(qkv[:, 128:])
    padded = o.add_qkv_bias_padding(q, zero, k, zero, v, zero, T, B, S, 1, 64, bi, wi, dtype)
    want = o.attention(*padded, attr, T, bi, wi, dtype)
    # Once as they are and once so often that the kernel takes two query tiles per wavefront; with the classes, which et_attention
    # has room for, and without.  (Without, keys are summed in another order.)
    for times in (1, -(-512 // (B * -(-S // 128)))):
        n = B * times
        pk, at = dev(np.tile(qkv, (times, 1))), dev(np.tile(attr, (times, 1, 1)))
        index = [torch.full((n * S,), -1, dtype=torch.int32, device="cuda") for _ in range(2)]
        index[0][:T * times] = dev((bi[None] + B * np.arange(times)[:, None]).reshape(-1).astype(np.int32))
        index[1][:T * times] = dev(np.tile(wi, times).astype(np.int32))
        count = torch.tensor([T * times], dtype=torch.int32, device="cuda")
        for starts in (None, ops.sequence_starts(count, index[0], n, S)):
            got = kernel_ops.attention(pk, pk[:, 64:], pk[:, 128:], 1, 192, at, count, n, S, 1, 64, *index, seq_start=starts)
            got = got[:T * times].cpu().numpy().reshape(times, T, 64)
            assert all(np.array_equal(g, got[0]) for g in got)
            # as in the tests of the kernels: fp16 has the oracle's exact sums against float ones and three roundings to half
            if dtype == "fp32":
                np.testing.assert_allclose(got[0], want, rtol=1e-4, atol=2e-5)
            else:
                np.testing.assert_allclose(got[0].astype(np.float32), want.astype(np.float32), rtol=4e-3, atol=4e-3)

    # a layer, which has the mask's classes made
    wl = Workload("behind", S, dtype, 1, B, S, 2, 64, 512)
    weights = make_layer_weights(wl, rng, random_affine=True)
    for slot in (0, 2, 4, 6):
        weights[slot] = weights[slot] * el(4)                # an attention that depends on its keys
    w = dict(wl=wl, x=rng.randn(B, S, wl.H).astype(el), weights=weights, mask=mask, attr_mask=attr)
    got, want = run_encoder(w), o.encoder(w["x"], mask, attr, weights, wl.heads, wl.d, dtype)
    valid = mask.astype(bool)
    err = np.abs(got[valid].astype(np.float64) - want[valid].astype(np.float64)).max()
    print("  max abs diff", err, flush=True)
    assert err < (2e-2 if dtype == "fp16" else 1e-4)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("form", ["causal", "ones"])
def test_padding_costs_little_under_any_mask(dtype, form):
    """et_attention on the same 32 sequences of up to 128 tokens in 512 positions and in 128: without stages behind the tokens
    it takes about the same time, with them three times as long and more."""
    heads, lens = 12, torch.randint(16, 129, (32,), generator=torch.Generator().manual_seed(1))

    def microseconds(S):
        mask = (torch.arange(S)[None] < lens[:, None])
        attr = torch.ones(32, S, S) if form == "ones" else torch.tril(mask[:, None].expand(32, S, S).float())
        attr, mask = attr.to(dtype).cuda(), mask.int().cuda()
        _, count, bi, wi = ops.effective_transformer_input(torch.zeros(32, S, 64, dtype=dtype, device="cuda"), mask, 32, S, S, 1, 64)
        qkv = torch.randn(int(count.item()), 3 * heads * 64, device="cuda").to(dtype)
        dst = torch.zeros(32 * S, heads * 64, dtype=dtype, device="cuda")
        times = []
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                kernel_ops.attention(qkv, qkv[:, heads * 64:], qkv[:, 2 * heads * 64:], 1, 3 * heads * 64, attr, count, 32, S,
                                     heads, 64, bi, wi, dst=dst)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 50)
        return min(times)

    narrow, wide = microseconds(128), microseconds(512)
    print("padding", dtype, form, "us", narrow, wide, flush=True)
    assert wide < 2 * narrow


def test_workspaces_with_and_without_room_for_the_classes():
    """et_attention takes a workspace that holds the sequence table alone and makes no classes then; the first size that holds
    both is et_seq_workspace_bytes' at 1024 positions.  A plain mask: the same bits either way."""
    from effective_transformer_amd import _lib
    lib, B, S = _lib.load(), 40, 1024
    rng = np.random.RandomState(5)
    lens = rng.randint(1, 200, size=B)
    mask = dev((np.arange(S)[None] < lens[:, None]).astype(np.int32))
    attr = mask[:, None].expand(B, S, S).half().contiguous()
    _, count, bi, wi = ops.effective_transformer_input(torch.zeros(B, S, 64, dtype=torch.float16, device="cuda"), mask, B, S, S, 1, 64)
    T = int(lens.sum())
    qkv = dev(rng.randn(T, 192).astype(np.float16))
    full = lib.et_seq_workspace_bytes(B)
    table = full - B * 64
    assert table == ((2 * B + 1) * 4 + 255) // 256 * 256
    want, h = None, ops.handle(qkv.device)
    for nbytes in (table, full - 1, full):
        ws = torch.zeros(full + 256, dtype=torch.uint8, device="cuda")
        dst = torch.zeros(T, 64, dtype=torch.float16, device="cuda")
        _lib.check(lib.et_attention(h, _lib.ET_FP16, qkv.data_ptr(), qkv[:, 64:].data_ptr(), qkv[:, 128:].data_ptr(), 1, 192,
                                    attr.data_ptr(), dst.data_ptr(), count.data_ptr(), B, S, 1, 64, bi.data_ptr(), wi.data_ptr(),
                                    ws.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream), h)
        want = dst if want is None else want
        assert torch.equal(dst, want)
        assert (ws[nbytes:] == 0).all() and bool((ws[table:] != 0).any()) == (nbytes == full)
    assert lib.et_attention(h, _lib.ET_FP16, qkv.data_ptr(), qkv.data_ptr(), qkv.data_ptr(), 1, 192, attr.data_ptr(),
                            want.data_ptr(), count.data_ptr(), B, S, 1, 64, bi.data_ptr(), wi.data_ptr(), ws.data_ptr(), table - 1,
                            None) == 2
