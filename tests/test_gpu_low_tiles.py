"""fp16 products of narrow outputs on the persistent kernel's low tiles: the bits of small products, tile by tile."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# 192 rows a tile (13097 x 1024, 13000 x 1024, 25000 x 512) and 160 (the others); k of two and three pairs of k-steps and more; a last
# round that is shared by two workgroups a tile, rows that end inside a tile, one tile for each workgroup
@pytest.mark.parametrize("m,n,k", [(13097, 1024, 4096), (13097, 1024, 1024), (13000, 1024, 2048), (12290, 768, 3072), (12290, 768, 768),
                                   (11201, 768, 3072), (25000, 512, 512), (40000, 128, 128), (40001, 192, 192), (39999, 256, 256)])
@pytest.mark.parametrize("on_device", [False, True])
def test_bits_of_small_products(m, n, k, on_device):
    from effective_transformer_amd import kernel_ops as ko
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn(m, k, device="cuda", dtype=torch.float16, generator=gen)
    bt = torch.randn(n, k, device="cuda", dtype=torch.float16, generator=gen).mul_(k ** -0.5)
    bias = torch.randn(n, device="cuda", dtype=torch.float16, generator=gen)
    rows = m - 7 if on_device else m
    out = torch.full((m, n), 3.0, device="cuda", dtype=torch.float16)
    for _ in range(2):                         # (the second one right behind the first)
        ko.gemm_bt(a, bt, bias, m_dev=torch.tensor([rows], dtype=torch.int32, device="cuda") if on_device else None, out=out)
    for first in list(range(0, rows, 1500)) + [rows - 300]:
        last = min(first + 333, rows)
        assert torch.equal(ko.gemm_bt(a[first:last].contiguous(), bt, bias), out[first:last]), (first, last)
    assert (out[rows:] == 3.0).all()
