"""The 32 x 32 tile of the fp16 product on k-contiguous weights (few rows and columns) against the [k][n] kernel's bits and
float64, at its edges and where the next tile takes over."""
import pytest
import torch

from effective_transformer_amd import kernel_ops as k

pytestmark = pytest.mark.gpu


# n = 768 fills the chip with 32 x 32 tiles up to 320 rows; one to more k-pairs than the LDS ring holds; ragged columns
@pytest.mark.parametrize("m,n,kk", [(1, 8, 64), (31, 24, 128), (32, 40, 64 * 5), (33, 768, 64 * 6), (17, 3072, 768), (320, 768, 3072),
                                    (321, 768, 768), (64, 1000, 4096)])
def test_small_tiles(m, n, kk):
    print("small tiles", m, n, kk, flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n + kk)
    a = torch.randn(m, kk, device="cuda", generator=g).half()
    b = (torch.randn(kk, n, device="cuda", generator=g) * 0.05).half()
    bias = torch.randn(n, device="cuda", generator=g).half()
    bt = k.transpose_weight(b)
    got = k.gemm_bt(a, bt)
    assert torch.equal(got, k.gemm(a, b))
    want = a.cpu().double() @ b.cpu().double()
    # one rounding to half, and float sums of kk products of half numbers in front of it
    err = (got.cpu().double() - want).abs()
    bound = want.abs() * 2.0 ** -11 + 2.0 ** -24 + kk * 2.0 ** -24 * (a.cpu().double().abs() @ b.cpu().double().abs())
    assert (err <= bound).all()
    assert torch.equal(k.gemm_bt(a, bt, bias=bias), got + bias)
    assert torch.equal(k.gemm_bt(a, bt, bias=bias, gelu=True), k.gemm(a, b, bias=bias, gelu=True))
    rows = torch.tensor([m // 2], dtype=torch.int32, device="cuda")
    out = torch.full_like(got, 7)
    k.gemm_bt(a, bt, m_dev=rows, out=out)
    assert torch.equal(out[:m // 2], got[:m // 2]) and (out[m // 2:] == 7).all()
