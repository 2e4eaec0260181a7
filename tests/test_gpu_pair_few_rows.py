"""fp32 products on pair rows of few rows: the tiles of 16 and 32 rows, in strips of columns, give the bits of products of many rows."""
import pytest
import torch

from effective_transformer_amd import kernel_ops as k
from test_gpu_head_exponents import _layer, _run, _spread_heads

pytestmark = pytest.mark.gpu


# rows that end inside a tile, the last counts for which 16 x 32 is one round of 256 CUs and the first ones beyond; columns in one strip, in
# several and in strips of one tile; one stage to more than the ring holds, odd and even
@pytest.mark.parametrize("n,kk", [(768, 768), (768, 2048), (512, 64), (512, 448), (2304, 512), (48, 576), (784, 192), (3072, 768), (1024, 1024)])
@pytest.mark.parametrize("m", [1, 15, 17, 48, 100, 170, 171, 240, 257, 340, 500])
def test_bits_of_many_rows(m, n, kk):
    print("pair few rows", m, n, kk, flush=True)
    many = 2600
    g = torch.Generator(device="cuda").manual_seed(n + kk)
    a = torch.randn(many, kk, device="cuda", generator=g)
    b = torch.randn(kk, n, device="cuda", generator=g) * 0.02
    bias = torch.randn(n, device="cuda", generator=g)
    pb, stats = k.pair_weight(b, bias)
    want = k.gemm_pair(k.pair_rows(a), pb, bias=bias)
    pa = k.pair_rows(a[:m].contiguous())
    assert torch.equal(k.gemm_pair(pa, pb, bias=bias), want[:m])
    rows = m // 2
    part = k.gemm_pair(pa, pb, bias=bias, m_dev=torch.tensor([rows], dtype=torch.int32, device="cuda"))
    assert torch.equal(part[:rows], want[:rows]) and (part[rows:] == 0).all()
    if n % 32 == 0:
        act = k.gemm_pair(k.pair_rows(a), pb, bias=bias, stats=stats, gelu=True)
        few = k.gemm_pair(pa, pb, bias=bias, stats=stats, gelu=True)
        assert torch.equal(few.rows[:m], act.rows[:m]) and torch.equal(few.exp[:m], act.exp[:m])


# output products with an exponent per head on 32 x 32 tiles, against a sequence alone on 16 x 32
@pytest.mark.parametrize("heads,S,B", [(12, 40, 6), (16, 33, 5), (8, 50, 8), (12, 15, 1), (32, 17, 3)])
def test_head_exponents(heads, S, B):
    w = _spread_heads(_layer(heads, 64, heads), heads, 64)
    x = torch.randn(B, S, heads * 64, generator=torch.Generator().manual_seed(B))
    got = _run(x, w, heads, 64)
    for b in range(B):
        assert torch.equal(_run(x[b:b + 1], w, heads, 64)[0], got[b]), "sequence %d" % b
