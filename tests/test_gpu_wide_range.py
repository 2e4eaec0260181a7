"""fp32 layers on pair rows whose weights or rows hold values of very different size: heads of Q and K, biases and tokens may differ
by any power of two, values of one row or column by 2^20, and the layer's rows keep the precision of float."""
import numpy as np
import pytest
import torch

from effective_transformer_amd import _lib, kernel_ops as k, ops
from oracle import et_oracle as o
from gpu_util import dev

pytestmark = pytest.mark.gpu

HEADS, D, H = 8, 64, 512
Q, BQ, K, BK, V, BV, OUT, BO, LN1B, LN1G, UP, BUP, DOWN, BDOWN, LN2B, LN2G = range(16)


def _weights(rng):
    """A layer in which attention and FFN outweigh what is added to them, so that a fault in either is not hidden by it."""
    w = []
    for i in range(4):
        w += [rng.randn(H, H) * (0.02 if i < 2 else 0.1), rng.randn(H) * 0.02]
    w += [rng.randn(H) * 0.02, 0.1 + rng.randn(H) * 0.005, rng.randn(H, 4 * H) * 0.3, rng.randn(4 * H) * 0.02,
          rng.randn(4 * H, H) * 0.1, rng.randn(H) * 0.02, rng.randn(H) * 0.05, 1 + rng.randn(H) * 0.05]
    return [t.astype(np.float32) for t in w]


# Each changes a layer so that its result is (nearly) the one of an ordinary layer: what is large is switched off, or a power of
# two is moved from one matrix into the next.
def _plain(w, x, by):
    pass


def _qk_head(w, x, by):
    for at in (Q, BQ):
        w[at][..., 64:128] *= by
    for at in (K, BK):
        w[at][..., 64:128] /= by


def _neuron_off(w, x, by):
    """One entry of the first FFN bias large and negative: its GELU is 0."""
    w[BUP][5] = -by


def _unseen_token(w, x, by):
    """The last token of every sequence has large values in V (each factor within what a row and a column hold), and nobody sees it
    but its own query (UNSEEN)."""
    s = np.sqrt(by)
    x[..., 7] = 0
    x[np.arange(len(x)), _lengths(x.shape[1]) - 1, 7] = s
    w[Q][7], w[K][7] = 0, 0
    w[V][7] *= s


def _v_head(w, x, by):
    """A head of V and its rows of the output kernel: what a row and a column hold reaches 2^20 down."""
    s = np.sqrt(by)
    for at in (V, BV):
        w[at][..., 64:128] *= s
    w[OUT][64:128] /= s


CHANGES = [_plain, _qk_head, _neuron_off, _unseen_token, _v_head]
UNSEEN = [_unseen_token]


def _lengths(S):
    return np.array([S, S - 3, S - 7])


# both fp32 attention kernels
@pytest.mark.parametrize("S", [20, 40])
@pytest.mark.parametrize("by", [2.0 ** 20, 2.0 ** 30, 2.0 ** 40])
@pytest.mark.parametrize("change", CHANGES, ids=lambda f: f.__name__[1:])
@pytest.mark.parametrize("split_copies", [False, True])
def test_layer(change, by, S, split_copies):
    print("wide layer", change.__name__, by, S, split_copies, flush=True)
    B = 3
    rng = np.random.RandomState(S)
    w = _weights(rng)
    x, to = (rng.randn(B, S, H).astype(np.float32) for _ in range(2))
    x *= 0.05
    change(w, to, np.float32(by))
    lens = _lengths(S)
    mask = (np.arange(S)[None] < lens[:, None]).astype(np.int32)
    attr = np.ascontiguousarray(np.broadcast_to(mask[:, None], (B, S, S))).astype(np.float32)
    if change in UNSEEN:
        for b in range(B):
            attr[b, :lens[b] - 1, lens[b] - 1] = 0
    packed, T, bi, wi = o.input_op_fast(x, mask)[:4]
    packed_to = o.input_op_fast(to, mask)[0]
    want = o.layer(packed, packed_to, attr, T, bi, wi, w, B, S, HEADS, D, "fp32").astype(np.float64)
    dx, count, dbi, dwi = ops.effective_transformer_input(dev(x), dev(mask), B, S, S, HEADS, D)
    dto = ops.effective_transformer_input(dev(to), dev(mask), B, S, S, HEADS, D)[0]
    lw = ops.LayerWeights.from_slots(torch.device("cuda"), torch.float32, [dev(t) for t in w])
    if split_copies:                                         # et_layer_prepared: split rows of the weights instead of the floats
        copies = [k.transpose_weight(dev(w[i])) for i in (Q, K, V, OUT, UP, DOWN)]
        prep = _lib.LayerPrepared()
        for name, t in zip(("attr_kernel_Q_t", "attr_kernel_K_t", "attr_kernel_V_t", "attr_output_kernel_t", "inter_kernel_t",
                            "output_kernel_t"), copies):
            setattr(prep, name, t.data_ptr())
        lw.prepared = prep
    got = ops.effective_transformer(dx, dto, dev(attr), count, dbi, dwi, lw, B, S, S, HEADS, D)
    got = got.reshape(-1, H)[:T].cpu().numpy().astype(np.float64)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    if change in UNSEEN:
        keep = np.ones(T, bool)
        keep[np.cumsum(lens) - 1] = False
        want, got = want[keep], got[keep]
    # row by row; the oracle is float32 itself: about 1e-7 per product on either side, and what these wider layers make of the
    # first ones' (scores of up to a few units: 4 x the error of plain layers, 2e-6 in test_gpu_pair.py)
    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    print("largest error %.2e" % err.max(), flush=True)
    assert err.max() <= 8e-6, (err.max(), int(err.argmax()))
