"""et_encoder, the stack in one call: the same bits as the ops one by one, its count word, and what it refuses."""
import ctypes as C

import numpy as np
import pytest
import torch

from effective_transformer_amd import _lib, ops
from effective_transformer_amd.sample.workloads import Workload, make_layer_weights
from gpu_util import TDT, dev

pytestmark = pytest.mark.gpu


def _batch(B, S, layers, dtype, share=0.6, heads=2):
    dt = TDT[dtype]
    wl = Workload("call", S, dtype, layers, B, S, heads, 64, 4 * heads * 64)
    rng = np.random.RandomState(B * 1000 + S)
    weights = [a for _ in range(layers) for a in make_layer_weights(wl, rng, random_affine=True)]
    lens = np.minimum(rng.randint(1, max(2, int(2 * share * S) + 1), size=B), S)
    mask = (np.arange(S)[None] < lens[:, None]).astype(np.int32)
    attr = np.ascontiguousarray(np.broadcast_to(mask[:, None], (B, S, S)))
    enc = ops.EffectiveTransformerEncoder(layers, heads, 64, weights, dt, "cuda")
    return wl, enc, dev(rng.randn(B, S, wl.H), dt), dev(mask), dev(attr, dt), int(lens.sum())


def _one_by_one(wl, enc, x, mask, attr):
    B, S = mask.shape
    h, vwn, bidx, widx = ops.effective_transformer_input(x, mask, B, S, S, wl.heads, 64)
    for w in enc.layers:
        h = ops.effective_transformer(h, h, attr, vwn, bidx, widx, w, B, S, S, wl.heads, 64)
    return ops.effective_transformer_output(h, vwn, bidx, widx, B, S, S, wl.heads, 64)


# a handful of positions and some hundreds, all valid and few, one layer (which does not wait for the count) and more
@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
@pytest.mark.parametrize("B,S,layers,share", [(1, 1, 2, 1), (1, 8, 1, 0.6), (1, 8, 3, 0.6), (8, 32, 2, 1), (8, 32, 2, 0.3),
                                              (257, 1, 2, 1), (9, 32, 2, 0.3), (5, 100, 2, 0.6), (20, 64, 1, 0.6)])
def test_same_bits_as_the_ops(B, S, layers, share, dtype):
    print("encoder call", B, S, layers, share, dtype, flush=True)
    wl, enc, x, mask, attr, _ = _batch(B, S, layers, dtype, share)
    want = _one_by_one(wl, enc, x, mask, attr)
    assert torch.equal(enc(x, mask, attr), want)
    assert torch.equal(enc(x, mask, attr, sync_count=False), want)


def _call(enc, batch, ws, layers=None, ws_bytes=None, dtype=_lib.ET_FP16, weights="table"):
    lib = _lib.load()
    _, table, prepared = enc._layer_table()
    return lib.et_encoder(ops.handle(enc.device), dtype, len(enc.layers) if layers is None else layers,
                          table if weights == "table" else weights, prepared, None if batch is None else C.byref(batch),
                          enc.head_num, enc.size_per_head, ws.data_ptr(), ws.numel() if ws_bytes is None else ws_bytes,
                          torch.cuda.current_stream().cuda_stream)


def _struct(x, mask, attr, out):
    b = _lib.EncoderBatch()
    b.from_tensor, b.mask, b.attr_mask, b.out = x.data_ptr(), mask.data_ptr(), attr.data_ptr(), out.data_ptr()
    b.batch_size, b.seq_len = mask.shape
    return b


@pytest.mark.parametrize("layers", [1, 2])
@pytest.mark.parametrize("word", [False, True])
@pytest.mark.parametrize("host_count", [False, True])
def test_count_word_and_host_count(word, host_count, layers):
    wl, enc, x, mask, attr, tokens = _batch(12, 40, layers, "fp16")
    want = enc(x, mask, attr)
    lib = _lib.load()
    out = torch.full_like(x, float("nan"))
    ws = torch.empty(lib.et_encoder_workspace_bytes(_lib.ET_FP16, 12, 40, wl.heads, 64), dtype=torch.uint8, device="cuda")
    b = _struct(x, mask, attr, out)
    pinned, count = torch.zeros(1, dtype=torch.int64, pin_memory=True), C.c_int32(-7)
    if word:
        b.count_word = pinned.data_ptr()
    if host_count:
        b.valid_word_num = C.pointer(count)
    for _ in range(3):                                       # (the word of the pass before is not taken for this one's)
        assert _call(enc, b, ws) == 0
        if host_count:
            assert count.value == tokens
            count.value = -7
        if word and (host_count or layers > 1):
            assert int(pinned[0]) & 0xffffffff == tokens
    assert torch.equal(out, want)


def test_one_encoder_on_two_streams():
    """Calls that wait for their counts, on two streams in turn: each stream has its word and its workspace."""
    wl, enc, x, mask, attr, _ = _batch(12, 40, 2, "fp16")
    fewer = mask.clone()
    fewer[3:] = 0
    want = [enc(x, m, attr).clone() for m in (mask, fewer)]
    torch.cuda.synchronize()
    streams, got = [torch.cuda.Stream(), torch.cuda.Stream()], [[], []]
    for _ in range(10):
        for s, m, g in zip(streams, (mask, fewer), got):
            with torch.cuda.stream(s):
                g.append(enc(x, m, attr))
    torch.cuda.synchronize()
    for w, g in zip(want, got):
        assert all(torch.equal(o, w) for o in g)


@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
def test_single_layer_under_capture(dtype):
    """An encoder of one layer waits for nothing, so a caller may capture the call as it is (a deeper one with sync_count=False)."""
    wl, enc, x, mask, attr, _ = _batch(12, 40, 1, dtype)
    fewer, m = mask.clone(), mask.clone()
    fewer[5:, 10:] = 0
    want = [enc(x, k, attr).clone() for k in (mask, fewer)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = enc(x, m, attr)
    for i in (0, 1, 0, 1):
        m.copy_((mask, fewer)[i])
        graph.replay()
        assert torch.equal(out, want[i])
        assert torch.equal(enc(x, m, attr), want[i])         # eager work between the replays


@pytest.mark.parametrize("B,S", [(2, 40), (12, 40)])
def test_call_that_would_wait_under_capture(B, S):
    """A deeper encoder whose pinned word exists already (an earlier call on the stream that captures): the call does not wait
    while the stream is being captured, and the replays follow the mask."""
    wl, enc, x, mask, attr, _ = _batch(B, S, 2, "fp16")
    fewer, m = mask.clone(), mask.clone()
    fewer[B // 2:, 10:] = 0
    want = [enc(x, k, attr).clone() for k in (mask, fewer)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        enc(x, m, attr)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = enc(x, m, attr)
    for i in (0, 1, 0, 1):
        m.copy_((mask, fewer)[i])
        graph.replay()
        assert torch.equal(out, want[i])
        assert torch.equal(enc(x, m, attr), want[i])         # eager work between the replays


def test_refused_arguments():
    wl, enc, x, mask, attr, _ = _batch(2, 8, 2, "fp16")
    lib = _lib.load()
    h = ops.handle(enc.device)
    out = torch.zeros_like(x)
    nbytes = lib.et_encoder_workspace_bytes(_lib.ET_FP16, 2, 8, wl.heads, 64)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")

    def refused(status, message, call=None, **members):
        b = _struct(x, mask, attr, out)
        for k, v in members.items():
            setattr(b, k, v)
        assert _call(enc, b, ws, **(call or {})) == status
        assert message in lib.et_last_error(h).decode()

    emb = _lib.EmbeddingWeights()
    ids = torch.zeros(2, 8, dtype=torch.int32, device="cuda")
    refused(1, "dtype", call=dict(dtype=2))
    refused(1, "at least one layer", call=dict(layers=0))
    refused(1, "at least one layer", call=dict(weights=None))
    refused(1, "must be >= 1", batch_size=0)
    refused(1, "must be >= 1", seq_len=0)
    refused(1, "either from_tensor or embeddings", from_tensor=None)
    refused(1, "either from_tensor or embeddings", embeddings=C.pointer(emb))
    for member in ("mask", "attr_mask", "out"):
        refused(1, "null tensor", **{member: None})
    refused(1, "null tensor", from_tensor=None, embeddings=C.pointer(emb))
    refused(1, "null embedding", from_tensor=None, embeddings=C.pointer(emb), input_ids=ids.data_ptr())
    refused(1, "rows_bound", rows_bound=-1)
    refused(1, "rows_bound", rows_bound=17)
    refused(2, "et_encoder_workspace_bytes", call=dict(ws_bytes=nbytes - 1))
    refused(3, "65535", batch_size=65536, seq_len=1)
    refused(3, "1024", seq_len=1025)
    refused(1, "null weight", call=dict(weights=(_lib.LayerWeights * 2)()))
    assert _call(enc, None, ws) == 1 and "null batch" in lib.et_last_error(h).decode()
    torch.cuda.synchronize()
    assert (out == 0).all()
