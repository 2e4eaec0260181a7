"""fp32 products on split rows (csrc/gemm_split.hip) against float64, at the edges of their tiles."""
import pytest
import torch

from effective_transformer_amd import kernel_ops as k

pytestmark = pytest.mark.gpu


def _joined(s):
    """The float64 sum of the three pieces of split rows [m, 3 n]."""
    return s.double().reshape(s.shape[0], -1, 3, 32).sum(2).reshape(s.shape[0], -1)


def _operands(m, n, kk, positive=False):
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n * 3 + kk)
    a = torch.randn(m, kk, device="cuda", generator=g)
    b = torch.randn(kk, n, device="cuda", generator=g) * 0.02
    bias = torch.randn(n, device="cuda", generator=g)
    return (a.abs(), b.abs(), bias) if positive else (a, b, bias)


# rows and columns around 32, 64, 128 and 256 (tiles' sides), one and an odd number of k-steps of 32, fewer k-steps
# than the LDS ring of the small tiles holds, and grids of one to several rounds of the chip
@pytest.mark.parametrize("m,n,kk", [(1, 4, 32), (31, 36, 32), (33, 64, 96), (64, 100, 160), (65, 768, 768), (127, 132, 64),
                                    (160, 768, 3072), (257, 136, 96), (700, 768, 3072), (1025, 2304, 768),
                                    (4200, 768, 768), (9000, 1536, 128),
                                    # tiles of 192 and of 96 rows: last row of a tile, one behind it, one and several rounds
                                    (7872, 768, 768), (5761, 772, 768), (7999, 768, 3072), (8000, 2304, 96), (3072, 768, 768), (3073, 768, 3072),
                                    (1000, 2304, 768)])
@pytest.mark.parametrize("positive", [False, True])
def test_gemm_split(m, n, kk, positive):
    print("gemm_split", m, n, kk, positive, flush=True)
    a, b, bias = _operands(m, n, kk, positive)
    sa, sb = k.split_rows(a), k.transpose_weight(b)
    assert torch.equal(_joined(sa).float(), a) and torch.equal(_joined(sb).float(), b.t())      # the pieces are exact
    want = (a.cpu().double() @ b.cpu().double()).cuda()
    got = k.gemm_split(sa, sb)
    err = ((got - want).norm() / want.norm()).item()
    native = ((k.gemm(a, b) - want).norm() / want.norm()).item()
    # no further from float64 than the fp32 matrix instructions (short sums: both round once or twice)
    assert err <= max(native * 1.05, 6e-8), (err, native)
    assert torch.equal(k.gemm_split(sa, sb, bias=bias), got + bias)
    # a row has the same bits whatever the number of rows (other tiles), and rows beyond the device's count stay as they are
    for rows in (1, (m + 1) // 2):
        assert torch.equal(k.gemm_split(sa[:rows].contiguous(), sb), got[:rows])
    part = k.gemm_split(sa, sb, m_dev=torch.tensor([m // 2], dtype=torch.int32, device="cuda"))
    assert torch.equal(part[:m // 2], got[:m // 2]) and (part[m // 2:] == 0).all()
    if n % 32 == 0:
        act = _joined(k.gemm_split(sa, sb, bias=bias, gelu=True))
        ref = torch.nn.functional.gelu(want + bias.double(), approximate="tanh")
        assert ((act - ref).norm() / ref.norm()).item() < 1e-6


def test_split_rows_device_count_and_special_values():
    a = torch.tensor([[0.0, -0.0, 1e-30, -3.4e37, 1 + 2.0 ** -23, 2.0 ** -126] + [0.1] * 58] * 5, device="cuda")
    s = k.split_rows(a, m_dev=torch.tensor([3], dtype=torch.int32, device="cuda"))
    assert torch.equal(_joined(s[:3]).float(), a[:3]) and (s[3:] == 0).all()


def test_gemm_split_refuses_other_shapes():
    a, b, bias = _operands(8, 36, 64)
    sa, sb = k.split_rows(a), k.transpose_weight(b)
    with pytest.raises(Exception, match="gelu n % 32"):
        k.gemm_split(sa, sb, bias=bias, gelu=True)
    with pytest.raises(Exception, match="multiple of 32"):
        k.transpose_weight(torch.zeros(48, 36, device="cuda"))
