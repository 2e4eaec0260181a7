"""fp16 products whose row count only the device knows, and those of a handful of rows: the bits are those of any other tile."""
import pytest
import torch

from effective_transformer_amd import kernel_ops as k

pytestmark = pytest.mark.gpu


# bounds of less than one row tile up to several rounds of the persistent kernel (from 128 tiles of 256 x 256 on); n and k that leave
# rests in every tile's columns, and the shortest k of the ring
@pytest.mark.parametrize("n,kk", [(768, 768), (2304, 768), (3072, 768), (768, 3072), (1008, 320), (48, 128), (24, 64), (200, 832), (768, 896)])
@pytest.mark.parametrize("bound", [40, 1000, 4100, 12000])
@pytest.mark.parametrize("gelu", [False, True])
def test_rows_on_the_device(bound, n, kk, gelu):
    g = torch.Generator(device="cuda").manual_seed(bound + n + kk)
    a = torch.randn(bound, kk, device="cuda", generator=g).half()
    bt = (torch.randn(n, kk, device="cuda", generator=g) * 0.03).half()
    bias = torch.randn(n, device="cuda", generator=g).half()
    want = k.gemm_bt(a, bt, bias=bias, gelu=gelu)
    # every row's bits are the same in any tile, so one launch over all rows is the reference for each count
    ref = a.double() @ bt.double().t()
    if not gelu:
        # half rounding of the product and of its sum with the bias, and fp32 accumulation in order: kk roundings of 2^-24 of the
        # sum of |a b|
        tol = 2.0 ** -10 * (ref.abs() + bias.double().abs()) + kk * 2.0 ** -24 * (a.double().abs() @ bt.double().abs().t()) + 1e-6
        assert ((want.double() - ref - bias.double()).abs() <= tol).all()
    # (a handful of rows: one wavefront per 16 x 16 tile, with fewer, as many and more pairs of k-steps than its ring holds)
    for t in (1, 15, 16, 17, 33, 100):
        if t <= bound:
            assert torch.equal(k.gemm_bt(a[:t], bt, bias=bias, gelu=gelu), want[:t]), t
    edges = {0, 1, bound // 9, bound // 3, bound * 3 // 5, bound - 1, bound, bound + 3}
    # rounds of the chip at the tiles' heights and widths: counts on both sides of what each serves
    for rows in (32, 64, 96, 128, 160, 192, 224, 256):
        for cols in (32, 64, 128, 192, 256):
            serves = 256 // -(-n // cols) * rows
            edges |= {t for t in (serves, serves + 1) if 0 < t < bound}
    for t in sorted(edges):
        out = torch.full((bound, n), 7.0, device="cuda", dtype=torch.float16)
        k.gemm_bt(a, bt, bias=bias, gelu=gelu, m_dev=torch.tensor([t], dtype=torch.int32, device="cuda"), out=out)
        t = min(t, bound)
        assert torch.equal(out[:t], want[:t]), t
        assert (out[t:] == 7.0).all(), t
