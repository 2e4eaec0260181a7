"""Tensors that do not fit each other are refused by the host before anything is launched; a batch of fewer sequences than its
masks hold is not one of them."""
import threading

import numpy as np
import pytest
import torch

from effective_transformer_amd import _lib, ops


def _encoder(heads=2, d=64, dtype=torch.float32):
    enc = ops.EffectiveTransformerEncoder.__new__(ops.EffectiveTransformerEncoder)     # no weights: nothing may get as far
    enc.head_num, enc.size_per_head, enc.dtype = heads, d, dtype
    return enc


# the other tensors are those of 4 sequences of 8 positions, hidden size 128
@pytest.mark.parametrize("x,mask,attr", [((5, 8, 128), (4, 8), (4, 8, 8)),      # rows of the masks that do not exist
                                         ((4, 7, 128), (4, 8), (4, 8, 8)), ((4, 8, 64), (4, 8), (4, 8, 8)),
                                         ((4, 8, 192), (4, 8), (4, 8, 8)), ((32, 128), (4, 8), (4, 8, 8)),
                                         ((4, 8, 128), (4, 8), (3, 8, 8)), ((4, 8, 128), (4, 8), (4, 1, 8)),
                                         ((4, 8, 128), (4, 8), (4, 8, 9))])
def test_tensors_that_do_not_fit_the_batch(x, mask, attr):
    with pytest.raises(ValueError, match="must be \\["):
        _encoder()(torch.zeros(x), torch.zeros(mask, dtype=torch.int32), torch.zeros(attr))


@pytest.mark.parametrize("ids,types,attr,hidden", [((3, 8), None, (4, 8, 8), 128), ((4, 7), None, (4, 8, 8), 128),
                                                   ((4, 8), (3, 8), (4, 8, 8), 128), ((4, 8), (4, 8), (3, 8, 8), 128),
                                                   ((4, 8), (4, 8), (4, 8, 8), 64), ((4, 8), (4, 8), (4, 8, 8), 256)])
def test_ids_that_do_not_fit_the_batch(ids, types, attr, hidden):
    class Embeddings:
        dtype = torch.float32
    Embeddings.hidden = hidden
    z = lambda shape: None if shape is None else torch.zeros(shape, dtype=torch.int32)
    with pytest.raises(ValueError, match="must be \\[|columns"):
        _encoder().forward_ids(z(ids), z(types), z((4, 8)), torch.zeros(attr), Embeddings())


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
def test_fewer_sequences_than_the_masks_hold(dtype):
    from gpu_util import TDT, dev
    from oracle import et_oracle as o
    w = o.make_workload("cfg1", layers=1)
    wl, dt = w["wl"], TDT[dtype]
    enc = ops.EffectiveTransformerEncoder(1, wl.heads, wl.d, w["weights"], dt, "cuda")
    x, mask, attr = dev(w["x"], dt), dev(w["mask"].astype(np.int32)), dev(w["attr_mask"], dt)
    want = enc(x[:3], mask[:3], attr[:3])
    got = enc(x[:3], mask, attr)
    assert got.shape == x[:3].shape and torch.equal(got, want)
    assert torch.equal(enc(x[:3], mask, attr, sync_count=False), want)
    for same in (attr[:, None], attr.reshape(-1)):                    # [B,1,S,S], flat
        assert torch.equal(enc(x[:3], mask, same), want)


def _layer(n):
    slots = [torch.full((4, 4), float(n)) for _ in range(16)]
    return ops.LayerWeights.from_slots(torch.device("cpu"), torch.float32, slots)


def test_weight_structs_changed_after_a_call():
    """The structs a layer carries are what the next call hands over, also once an earlier call has put them into a table."""
    enc, other = _encoder(), _encoder()
    for e in (enc, other):
        e.layers, e._table, e._lock = [_layer(0), _layer(1)], None, threading.Lock()
    enc._layer_table()
    bias = torch.ones(4)
    enc.layers[1].struct.inter_bias = bias.data_ptr()                   # a member
    assert enc._layer_table()[1][1].inter_bias == bias.data_ptr()
    enc.layers[0].struct = _lib.LayerWeights()                          # the whole struct
    assert not enc._layer_table()[1][0].inter_bias
    enc.layers[0].struct.inter_bias = bias.data_ptr()
    other.layers[1] = enc.layers[0]                                     # a layer in two encoders' tables
    for e, l in ((other, 1), (enc, 0)):
        assert e._layer_table()[1][l].inter_bias == bias.data_ptr()
    enc.layers[0].struct.inter_bias = None
    for e, l in ((other, 1), (enc, 0)):
        assert not e._layer_table()[1][l].inter_bias
    enc.layers[1].prepared = _lib.LayerPrepared()
    enc.layers[1].prepared.inter_kernel_t = bias.data_ptr()
    assert enc._layer_table()[2][1].inter_kernel_t == bias.data_ptr()
    enc.layers = [enc.layers[0], enc.layers[1], enc.layers[0]]          # one layer twice
    enc._layer_table()
    enc.layers[0].struct.inter_bias = bias.data_ptr()
    t = enc._layer_table()[1]
    assert t[0].inter_bias == t[2].inter_bias == bias.data_ptr()
