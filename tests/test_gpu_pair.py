"""fp32 products on pair rows (csrc/gemm_pair.hip) against float64, at the edges of their tiles, and layers that run on them."""
import numpy as np
import pytest
import torch

from effective_transformer_amd import _lib, kernel_ops as k, ops
from oracle import et_oracle as o
from gpu_util import dev

pytestmark = pytest.mark.gpu


def _operands(m, n, kk, positive=False):
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n * 3 + kk)
    a = torch.randn(m, kk, device="cuda", generator=g)
    b = torch.randn(kk, n, device="cuda", generator=g) * 0.02
    bias = torch.randn(n, device="cuda", generator=g)
    return (a.abs(), b.abs(), bias) if positive else (a, b, bias)


def _rel(got, want):
    return ((got - want).norm() / want.norm()).item()


# rows and columns around 32, 64, 96, 128, 192 and 256 (tiles' sides), one and an odd number of chunks of 64 k, fewer stages than
# a ring holds, grids of one to several rounds of the chip (every tile shape is picked by one of them)
@pytest.mark.parametrize("m,n,kk", [(1, 16, 64), (31, 48, 64), (33, 64, 192), (64, 112, 320), (65, 768, 768), (127, 144, 128),
                                    (257, 144, 448), (600, 768, 1024), (700, 3072, 768), (1025, 2304, 768), (1500, 768, 2048),
                                    (4000, 2304, 512), (5761, 784, 768), (8000, 768, 1536), (9000, 1536, 128)])
@pytest.mark.parametrize("positive", [False, True])
def test_gemm_pair(m, n, kk, positive):
    print("gemm_pair", m, n, kk, positive, flush=True)
    a, b, bias = _operands(m, n, kk, positive)
    pa = k.pair_rows(a)
    pb, stats = k.pair_weight(b, bias)
    # h holds 11 bits, l 11 of the rest: half a unit of 2^-22 of the value at most, 2^-40 of the row's bound below that
    assert ((pa.values() - a.double()).abs() <= a.double().abs() * 2.0 ** -23 + a.abs().amax(1, keepdim=True).double() * 2.0 ** -39).all()
    assert torch.allclose(pa.norm[:m], a.norm(dim=1), rtol=1e-6)
    assert stats[0::2].max() >= b.norm(dim=0).max() * 0.999 and stats[1::2].max() == bias.abs().max()
    want = (a.cpu().double() @ b.cpu().double()).cuda()
    got = k.gemm_pair(pa, pb)
    # two operands rounded to 23 bits (rms 0.44 units of 2^-23 each), h.h + h.l + l.h without l.l (as much again), and a chunk of
    # six roundings per 64 k: below what split rows have from k = 512 on, below twice that at any k
    split = _rel(k.gemm_split(k.split_rows(a), k.transpose_weight(b)), want)
    err = _rel(got, want)
    assert err <= (split if kk >= 512 else max(2 * split, 2e-7)), (err, split)
    assert torch.equal(k.gemm_pair(pa, pb, bias=bias), got + bias)
    # a row has the same bits whatever the number of rows (other tiles), and rows beyond the device's count stay as they are
    for rows in (1, (m + 1) // 2):
        assert torch.equal(k.gemm_pair(k.pair_rows(a[:rows].contiguous()), pb), got[:rows])
    count = torch.tensor([m // 2], dtype=torch.int32, device="cuda")
    part = k.gemm_pair(pa, pb, m_dev=count)
    assert torch.equal(part[:m // 2], got[:m // 2]) and (part[m // 2:] == 0).all()
    rows = k.pair_rows(a, m_dev=count)
    assert torch.equal(rows.rows[:m // 2], pa.rows[:m // 2]) and (rows.rows[m // 2:] == 0).all()
    if n % 32 == 0:
        act = k.gemm_pair(pa, pb, bias=bias, stats=stats, gelu=True)
        ref = torch.nn.functional.gelu(want + bias.double(), approximate="tanh")
        assert torch.isfinite(act.rows.float()).all() and _rel(act.values(), ref) < 1e-6


# pair rows as the result: widths that fill a wavefront's columns in part, rows that end inside the 16 whose exponents 16 lanes
# share, every tile shape, more weight statistics than one wavefront requests at once; row by row (another lane's exponent would be off
# by powers of two), the rows' sizes far apart; off: a bias that switches its column off
@pytest.mark.parametrize("m,n,kk", [(1, 32, 64), (7, 96, 128), (50, 160, 192), (67, 1056, 768), (331, 800, 512), (1500, 800, 768),
                                    (3001, 1184, 768), (9003, 1056, 512), (40, 8192, 64), (300, 4608, 1024)])
@pytest.mark.parametrize("off", [0.0, -1e6, -1e12])
def test_pair_rows_out(m, n, kk, off):
    print("pair rows out", m, n, kk, off, flush=True)
    a, b, bias = _operands(m, n, kk, False)
    bias[n // 2] += off
    a *= torch.logspace(-3, 1, 5, device="cuda").repeat((m + 4) // 5)[:m, None]
    pb, stats = k.pair_weight(b, bias)
    act = k.gemm_pair(k.pair_rows(a), pb, bias=bias, stats=stats, gelu=True).values()
    want = torch.nn.functional.gelu((a.cpu().double() @ b.cpu().double()).cuda() + bias.double(), approximate="tanh")
    # The product's own error, a few units of 2^-24 of |a| |column| (and as much of the bias's rounding), which GELU's slope of at most
    # 1.13 passes on; h + l: 2^-23 of a value and 2^-39 of the row's bound, which is no more than |a| |column| + the largest bias
    # above 0 or 0.171, so far below the first; GELU's exp2 and reciprocal a unit each, of v where the result is 0.  What does not
    # enter: a bias far below 0.
    sizes = a.double().norm(dim=1)[:, None] * b.double().norm(dim=0)[None] + bias.clamp(-8, 8).abs().double()[None]
    bound = a.double().norm(dim=1) * b.double().norm(dim=0).max() * 1.03 + bias.clamp(min=0).max().double()
    assert ((act - want).abs() <= 2.0 ** -20 * want.abs() + 2.0 ** -22 * sizes + 2.0 ** -39 * bound.clamp(min=0.171)[:, None]).all()


# the exponents take what rows and columns differ by: the same relative error at 1e30, 1e-30 and in between, row by row; zero
# rows and columns are zero; what a row or a column cannot hold (2^-39 of its largest value) is all that is lost, also where its
# largest value meets zeros
def test_magnitudes():
    a, b, _ = _operands(70, 64, 768)
    rows = torch.tensor([1e30, 1e-25, 1.0, 1e5, 1e-5], device="cuda").repeat(14)[:, None]
    cols = torch.tensor([1e-12, 1e6, 1.0, 1e-4], device="cuda").repeat(16)[None]
    a, b = a * rows, b * cols
    a[3], b[:, 5] = 0, 0
    got = k.gemm_pair(k.pair_rows(a), k.pair_weight(b)[0]).double().cpu()
    want = a.cpu().double() @ b.cpu().double()
    assert (got[3] == 0).all() and (got[:, 5] == 0).all()
    # operands off by 2^-23 each, l.l of 2^-22 at most, a chunk's sums and theirs by a few units
    scale = a.cpu().double().abs() @ b.cpu().double().abs()
    assert ((got - want).abs() <= 2.0 ** -20 * scale).all()
    for spread in (2.0 ** 12, 2.0 ** 20, 2.0 ** 30):
        a, b, _ = _operands(40, 64, 768)
        a[:, 5] *= spread                                    # large values of A meet zeros, but in column 3
        b[5], b[5, 3] = 0, 0.01
        b[9, :32] *= spread                                  # and large values of half the columns of B
        a[:, 9] = 0
        got = k.gemm_pair(k.pair_rows(a), k.pair_weight(b)[0]).double().cpu()
        a, b = a.cpu().double(), b.cpu().double()
        lost = a.abs().amax(1, keepdim=True) * b.abs().sum(0) + a.abs().sum(1, keepdim=True) * b.abs().amax(0)
        assert ((got - a @ b).abs() <= 2.0 ** -20 * (a.abs() @ b.abs()) + 2.0 ** -39 * lost).all()
    wide = torch.randn(8, 768, device="cuda") * torch.logspace(0, -9, 768, device="cuda")
    err = (k.pair_rows(wide).values() - wide.double()).abs()
    assert (err <= wide.double().abs() * 2.0 ** -23 + wide.abs().amax(1, keepdim=True).double() * 2.0 ** -39).all()


# infinities and NaN reach the results of their row and no others
def test_special_values():
    a, b, bias = _operands(40, 64, 128)
    clean = k.gemm_pair(k.pair_rows(a), k.pair_weight(b)[0])
    a[7, 3], a[9, 100], a[11] = float("inf"), float("nan"), 3.4e38
    got = k.gemm_pair(k.pair_rows(a), k.pair_weight(b)[0])
    assert torch.isnan(got[7]).all() and torch.isnan(got[9]).all()
    keep = [r for r in range(40) if r not in (7, 9, 11)]
    assert torch.equal(got[keep], clean[keep])
    assert torch.allclose(got[11].double(), 3.4e38 * b.double().sum(0), rtol=1e-4, atol=1e33)


# layers on pair rows: head sizes with and without an attention kernel that writes them, hidden sizes of one and an odd number of
# chunks, positions of either fp32 attention kernel; weights and rows of very different sizes.  Split and plain copies of the
# weights: the same bits.
@pytest.mark.parametrize("heads,d,B,S", [(8, 64, 3, 32), (16, 32, 3, 20), (9, 64, 2, 40), (12, 64, 5, 130)])
@pytest.mark.parametrize("scale", [1.0, 1e3])
def test_layer(heads, d, B, S, scale):
    print("layer", heads, d, B, S, scale, flush=True)
    H = heads * d
    rng = np.random.RandomState(B * S + heads)
    w = []
    for i in range(4):
        w += [rng.randn(H, H).astype(np.float32) * 0.02 / (scale if i < 2 else 1), rng.randn(H).astype(np.float32) * 0.02]
    w += [rng.randn(H).astype(np.float32) * 0.05, 1 + rng.randn(H).astype(np.float32) * 0.05,
          rng.randn(H, 4 * H).astype(np.float32) * 0.02, rng.randn(4 * H).astype(np.float32) * 0.02,
          rng.randn(4 * H, H).astype(np.float32) * 0.02, rng.randn(H).astype(np.float32) * 0.02,
          rng.randn(H).astype(np.float32) * 0.05, 1 + rng.randn(H).astype(np.float32) * 0.05]
    lens = rng.randint(1, S + 1, size=B)
    mask = (np.arange(S)[None] < lens[:, None]).astype(np.int32)
    attr = np.ascontiguousarray(np.broadcast_to(mask[:, None], (B, S, S))).astype(np.float32)
    x = rng.randn(B, S, H).astype(np.float32) * scale
    enc = ops.EffectiveTransformerEncoder(2, heads, d, [dev(t) for t in w + w], torch.float32)
    got = enc(dev(x), dev(mask), dev(attr)).cpu().numpy().astype(np.float64)
    want = o.encoder(x, mask, attr, w + w, heads, d, "fp32").astype(np.float64)
    valid = mask.astype(bool)
    # (the oracle is float32 itself: about 1e-7 per product on either side, eight of them in a row)
    assert (got[~valid] == 0).all()
    assert np.linalg.norm(got[valid] - want[valid]) <= 2e-6 * np.linalg.norm(want[valid])


# split copies of the weights (et_layer_prepared) hold the same floats: the same bits.  Widths that end inside the 256 k a block looks
# at for the columns' largest values.
@pytest.mark.parametrize("heads", [8, 9, 17])
def test_split_copies(heads):
    print("split copies", heads, flush=True)
    d, B, S, H = 64, 2, 24, heads * 64
    g = torch.Generator(device="cuda").manual_seed(heads)
    sizes = [(H, H), (H,)] * 4 + [(H,), (H,), (H, 4 * H), (4 * H,), (4 * H, H), (H,), (H,), (H,)]
    w = [torch.randn(*s, device="cuda", generator=g) * 0.05 for s in sizes]
    x = torch.randn(B, S, H, device="cuda", generator=g)
    mask = torch.ones(B, S, dtype=torch.int32, device="cuda")
    attr = torch.ones(B, S, S, device="cuda")
    dx, count, bi, wi = ops.effective_transformer_input(x, mask, B, S, S, heads, d)
    lw = ops.LayerWeights.from_slots(torch.device("cuda"), torch.float32, w)
    plain = ops.effective_transformer(dx, dx, attr, count, bi, wi, lw, B, S, S, heads, d)
    copies = [k.transpose_weight(w[i]) for i in (0, 2, 4, 6, 10, 12)]
    lw.prepared = _lib.LayerPrepared(*[t.data_ptr() for t in copies])
    assert torch.equal(ops.effective_transformer(dx, dx, attr, count, bi, wi, lw, B, S, S, heads, d), plain)


# the streaming attention of layers on pair rows (more than 32 positions): lengths around its stages of 32 keys and blocks of 64
# queries, holes, masks that are read and masks that are not, rows of a mask on 16-byte boundaries and odd ones; wide: scores tens
# apart, so that the exponents' reference moves
@pytest.mark.parametrize("S", [33, 64, 101, 200, 1024])
@pytest.mark.parametrize("wide", [False, True])
def test_attention_on_pair_rows(S, wide):
    print("attention on pair rows", S, wide, flush=True)
    heads, d, H = 8, 64, 512
    rng = np.random.RandomState(S)
    w = []
    for i in range(4):
        w += [rng.randn(H, H).astype(np.float32) * (0.2 if wide and i < 2 else 0.02), rng.randn(H).astype(np.float32) * 0.02]
    w += [rng.randn(H).astype(np.float32) * 0.05, 1 + rng.randn(H).astype(np.float32) * 0.05,
          rng.randn(H, 4 * H).astype(np.float32) * 0.02, rng.randn(4 * H).astype(np.float32) * 0.02,
          rng.randn(4 * H, H).astype(np.float32) * 0.02, rng.randn(H).astype(np.float32) * 0.02,
          rng.randn(H).astype(np.float32) * 0.05, 1 + rng.randn(H).astype(np.float32) * 0.05]
    lens = np.minimum([1, 31, 32, 33, S // 2, S - 1, S] if S < 1024 else [S, 65, S // 2], S)
    B = len(lens)
    mask = (np.arange(S)[None] < lens[:, None]).astype(np.int32)
    mask[-1, S // 8:S // 4] = 0                              # a hole
    attr = np.ascontiguousarray(np.broadcast_to(mask[:, None], (B, S, S))).astype(np.float32)
    attr[1] = np.tril(attr[1])                               # causal
    attr[2] = 1                                              # every key
    attr[-2, : S // 2] = rng.random_sample((S // 2, S)) < 0.6
    x = rng.randn(B, S, H).astype(np.float32)
    got = ops.EffectiveTransformerEncoder(1, heads, d, [dev(t) for t in w], torch.float32)(dev(x), dev(mask), dev(attr)).cpu().numpy()
    want = o.encoder(x, mask, attr, w, heads, d, "fp32").astype(np.float64)
    valid = mask.astype(bool)
    # as above, and what the roundings of a score (a few units of the sum of its products, on either side) make of a weight
    q, k_ = (np.abs(x[valid] @ w[2 * i]).reshape(-1, heads, d) for i in range(2))
    score = np.sqrt((q ** 2).sum(-1)).max() * np.sqrt((k_ ** 2).sum(-1)).max() / 8
    tol = 2e-6 + 4 * 2.0 ** -24 * score
    assert (got[~valid] == 0).all()
    assert np.linalg.norm(got[valid] - want[valid]) <= tol * np.linalg.norm(want[valid])
    assert np.abs(got[valid] - want[valid]).max() <= 12 * tol * np.abs(want[valid]).max()
