"""Weights as pair rows: a column's exponent comes from its largest value wherever in the column that stands."""
import pytest
import torch

pytestmark = pytest.mark.gpu
if torch.cuda.is_available():
    from effective_transformer_amd import kernel_ops as k


# one block of 256 k and a part of one, as many blocks as one pass of the four wavefronts takes (16), one more, three passes;
# columns that fill a tile of 64 in part
@pytest.mark.parametrize("n,kk", [(16, 64), (80, 320), (768, 768), (64, 1088), (112, 4096), (80, 4160), (16, 8256)])
def test_largest_value_anywhere(n, kk):
    print("largest value", n, kk, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + kk)
    b = torch.randn(kk, n, device="cuda", generator=g)
    cols = torch.arange(n, device="cuda")
    at = (cols * 257 + kk - 1) % kk                              # the last k, then another block of 256 for every column
    b[at, cols] = torch.ldexp(torch.full((n,), -1.5, device="cuda"), (cols % 40 + 4).int())
    rows = k.pair_weight(b)[0]
    want = (cols % 40 + 4 + 1 - 15).int()                        # 1.5 2^e lies below 2^(e + 1), which a pair holds as 2^15
    assert torch.equal(rows.exp[:n], want)
    # h + l: half a unit of the 23rd bit of a value, 2^-39 of the column's bound below that
    got, ref = rows.values()[:n], b.t().double()
    assert ((got - ref).abs() <= ref.abs() * 2.0 ** -23 + ref.abs().amax(1, keepdim=True) * 2.0 ** -39).all()
