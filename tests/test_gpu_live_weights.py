"""fp32 weights are read by every call: tensors handed in once and changed in place are seen by the next pass."""
import numpy as np
import pytest
import torch

from effective_transformer_amd import _lib, kernel_ops, ops
from effective_transformer_amd.sample.workloads import Workload, make_layer_weights
from gpu_util import dev

pytestmark = pytest.mark.gpu


def _batch(B, S, heads, layers):
    wl = Workload("live_weights", S, "fp32", layers, B, S, heads, 64, 4 * heads * 64)
    rng = np.random.RandomState(B + S)
    weights = [dev(a) for _ in range(layers) for a in make_layer_weights(wl, rng, random_affine=True)]
    lens = rng.randint(1, S + 1, size=B)
    mask = (np.arange(S)[None] < lens[:, None]).astype(np.int32)
    attr = np.ascontiguousarray(np.broadcast_to(mask[:, None], (B, S, S))).astype(np.float32)
    return wl, weights, dev(rng.randn(B, S, wl.H).astype(np.float32)), dev(mask), dev(attr)


# one layer and more, a handful of rows and enough for the large tiles
@pytest.mark.parametrize("B,S,heads,layers", [(1, 8, 2, 1), (8, 32, 12, 2), (60, 64, 4, 2)])
def test_weights_changed_in_place(B, S, heads, layers):
    print("live weights", B, S, heads, layers, flush=True)
    wl, weights, x, mask, attr = _batch(B, S, heads, layers)
    enc = ops.EffectiveTransformerEncoder(layers, heads, 64, weights, torch.float32)
    before = enc(x, mask, attr)
    graph = enc.make_graph(x, mask, attr)
    assert torch.equal(graph(), before)
    for t in weights:
        t.mul_(1.5).add_(0.01)
    fresh = ops.EffectiveTransformerEncoder(layers, heads, 64, [t.clone() for t in weights], torch.float32)
    want = fresh(x, mask, attr)
    assert not torch.equal(want, before)
    assert torch.equal(enc(x, mask, attr), want)
    assert torch.equal(graph(), want)


# who keeps the weights as they are may hand split copies over (et_layer_prepared): the same bits
@pytest.mark.parametrize("which", ["all", "qkv", "rest"])
def test_split_copies_handed_over(which):
    wl, weights, x, mask, attr = _batch(8, 32, 12, 1)
    to, vwn, bidx, widx = ops.effective_transformer_input(x, mask, wl.B, wl.S, wl.S, wl.heads, wl.d)
    lw = ops.LayerWeights.from_slots(x.device, torch.float32, weights)
    T = int(vwn.item())
    args = (to, to, attr, vwn, bidx, widx, lw, wl.B, wl.S, wl.S, wl.heads, wl.d, T)
    want = ops.effective_transformer(*args)
    prep, keep = _lib.LayerPrepared(), []
    for name, field in (("attr_kernel_q", "attr_kernel_Q_t"), ("attr_kernel_k", "attr_kernel_K_t"),
                        ("attr_kernel_v", "attr_kernel_V_t"), ("attr_output_kernel", "attr_output_kernel_t"),
                        ("inter_kernel", "inter_kernel_t"), ("output_kernel", "output_kernel_t")):
        if which == "all" or (which == "qkv") == (name in ("attr_kernel_q", "attr_kernel_k", "attr_kernel_v")):
            keep.append(kernel_ops.transpose_weight(lw.t[name]))
            setattr(prep, field, keep[-1].data_ptr())
    lw.prepared = prep
    got = ops.effective_transformer(*args)
    assert torch.equal(got.reshape(-1, wl.H)[:T], want.reshape(-1, wl.H)[:T])
