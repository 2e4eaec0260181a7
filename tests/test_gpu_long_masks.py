"""Layers of more than 64 (fp16) or 32 (fp32) positions: blocks of queries whose mask rows simply end with the sequence take a way of
their own through the attention kernel, decided on the device from the mask."""
import numpy as np
import pytest

from effective_transformer_amd.sample.workloads import Workload, make_layer_weights
from oracle import et_oracle as o
from gpu_util import run_encoder

pytestmark = pytest.mark.gpu


# around a block of 16 queries, a stage of 64 keys and a workgroup's 64 or 128 queries; a length that is no multiple of 8
@pytest.mark.parametrize("S,B,dtype", [(S, B, "fp16") for S, B in [(65, 6), (80, 300), (101, 64), (127, 6), (128, 6), (129, 6),
                                                                    (150, 64), (192, 7), (257, 130), (1023, 6), (1024, 6)]] +
                         [(S, B, "fp32") for S, B in [(33, 6), (50, 200), (64, 6), (65, 6), (101, 60), (128, 6), (129, 6), (150, 40), (160, 6), (255, 6), (513, 6), (1023, 6), (1024, 6)]])
def test_masks_of_every_kind(S, B, dtype):
    print("long masks", S, B, dtype, flush=True)
    el = np.float16 if dtype == "fp16" else np.float32
    wl = Workload("long_masks", S, dtype, 1, B, S, 2, 64, 512)
    rng = np.random.RandomState(S)
    weights = make_layer_weights(wl, rng, random_affine=True)
    for slot in (0, 2, 4, 6):
        weights[slot] = weights[slot] * el(4)        # an attention that depends on its keys
    w = dict(wl=wl, x=rng.randn(B, S, wl.H).astype(el), weights=weights)
    lens = rng.randint(1, S + 1, size=B)
    lens[:6] = np.minimum([S, S, 1, 128, 65, S - 1], S)
    mask = (np.arange(S)[None] < lens[:, None]).astype(np.int32)
    mask[3, 20:90] = 0                                       # a hole
    attr = np.ascontiguousarray(np.broadcast_to(mask[:, None], (B, S, S))).astype(el)
    plain = dict(w, mask=mask, attr_mask=attr)
    # a mask of 2^-24 where it was 0 weighs a key with exp(-10000 + ...) = 0 all the same, but is not the plain form
    faint = dict(plain, attr_mask=np.where(attr == 0, el(6e-8), attr))
    assert (faint["attr_mask"] != attr).any()
    got = run_encoder(plain)
    assert np.array_equal(got, run_encoder(faint))
    sub = slice(0, 6)
    mixed = attr[sub].copy()
    mixed[0] = np.tril(mixed[0])                             # causal
    mixed[1, S // 2, S // 3] = 0                             # one block of queries differs
    mixed[4] = (rng.random_sample((S, S)) < 0.7)             # not tied to the tokens at all
    small = dict(w, wl=Workload(**{**wl.__dict__, "B": 6}), x=w["x"][sub], mask=mask[sub], attr_mask=mixed)
    got, want = run_encoder(small), o.encoder(small["x"], small["mask"], mixed, w["weights"], wl.heads, wl.d, dtype)
    valid = small["mask"].astype(bool)
    err = np.abs(got[valid].astype(np.float64) - want[valid].astype(np.float64)).max()
    print("  max abs diff", err, flush=True)
    assert err < (2e-2 if dtype == "fp16" else 1e-4)


# At 1024 positions the maximum is not clamped at 0: keys behind the last token (score -10000, value 0) take weight where every
# score of a query lies about as low.  Q and K are their biases here, so that a head's scores are one number, exactly: fp32
# -20000 and -9999 after scaling, fp16 -infinity (the score is stored in half) and an ordinary one.  The tolerances are those of
# the layer (fp32 1e-4, fp16 2e-2): a wrong weight moves the attention's output by its own size.
@pytest.mark.parametrize("dtype", ["fp32", "fp16"])
@pytest.mark.parametrize("S", [1024, 1023])
def test_scores_below_the_mask_bias(S, dtype):
    print("scores below the mask bias", S, dtype, flush=True)
    el = np.float16 if dtype == "fp16" else np.float32
    lens = np.array([1, 40, 700, 1000, S - 1])
    B = len(lens)
    wl = Workload("low_scores", S, dtype, 1, B, S, 2, 64, 512)
    rng = np.random.RandomState(S)
    weights = make_layer_weights(wl, rng, random_affine=True)
    for slot in (0, 1, 2, 3):
        weights[slot] = np.zeros_like(weights[slot])
    q, k = weights[1].reshape(2, 64), weights[3].reshape(2, 64)
    q[:] = 0
    q[:, 0], k[:, 0] = (16, (-10000, -4999.5)) if dtype == "fp32" else ((1000, 1), (-1000, 1))
    mask = (np.arange(S)[None] < lens[:, None]).astype(np.int32)
    mask[2, 20:90] = 0                                       # a hole: keys that the mask does not hide, score and value 0
    attr = np.ascontiguousarray(np.broadcast_to(mask[:, None], (B, S, S))).astype(el)
    attr[2, :, 20:90] = 1
    # (the last query's row is not of the plain form: its block takes the general path, the others are as they were)
    attr[3, 999, 1] = 0
    w = dict(wl=wl, x=rng.randn(B, S, wl.H).astype(el), weights=weights, mask=mask, attr_mask=attr)
    got, want = run_encoder(w), o.encoder(w["x"], mask, attr, weights, wl.heads, wl.d, dtype)
    valid = mask.astype(bool)
    assert np.isfinite(want[valid]).all()
    err = np.abs(got[valid].astype(np.float64) - want[valid].astype(np.float64)).max()
    print("  max abs diff", err, flush=True)
    assert err < (2e-2 if dtype == "fp16" else 1e-4)
