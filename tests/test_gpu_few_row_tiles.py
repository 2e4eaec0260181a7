"""fp16 products of a handful of rows, whose operands four wavefronts bring for one: the bits of the [k][n] kernel, which has tiles of
its own."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# one chunk of k to what the ring holds, nine, and more than that, odd and even; rows and columns that end inside a tile, one row, a tile
# for every CU; a k of no whole number of chunks and more tiles than CUs, which go another way
@pytest.mark.parametrize("k", [256, 512, 768, 1024, 2048, 2240, 2304, 2560, 2816, 3072, 8192])
@pytest.mark.parametrize("m,n", [(1, 768), (16, 768), (20, 768), (37, 1024), (85, 768), (97, 768), (33, 40), (5, 8), (16, 4096)])
@pytest.mark.parametrize("on_device", [False, True])
def test_bits_of_many_rows(m, n, k, on_device):
    from effective_transformer_amd import kernel_ops as ko
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    many = 640
    a = torch.randn(many, k, device="cuda", dtype=torch.float16, generator=gen)
    bt = torch.randn(n, k, device="cuda", dtype=torch.float16, generator=gen).mul_(k ** -0.5)
    w = bt.t().contiguous()
    bias = torch.randn(n, device="cuda", dtype=torch.float16, generator=gen)
    rows = max(m - 7, 0) if on_device else m
    count = torch.tensor([rows], dtype=torch.int32, device="cuda") if on_device else None
    for gelu in (False, True):
        for add in ((bias, None) if not gelu else (bias,)):
            want = ko.gemm(a, w, add, gelu=gelu)
            out = torch.full((m, n), 3.0, device="cuda", dtype=torch.float16)
            for _ in range(2):                     # (the second one right behind the first)
                ko.gemm_bt(a[:m].contiguous(), bt, add, m_dev=count, out=out, gelu=gelu)
            assert torch.equal(out[:rows], want[:rows])
            assert (out[rows:] == 3.0).all()
    if m <= 33 and n <= 1024:
        exact = a[:rows].double() @ bt.double().t() + bias.double()
        got = ko.gemm_bt(a[:m].contiguous(), bt, bias)[:rows].double()
        # a rounding of the product and one of the sum with the bias, 2^-11 of each, and k roundings in float
        assert ((got - exact).abs() <= (exact.abs() + (exact - bias.double()).abs()) * 2.0 ** -11 * 1.01 + 1e-4).all()
