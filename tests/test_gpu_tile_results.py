"""How the tiles of small fp16 products on k-contiguous weights leave: every tile shape with rows and columns that end inside it, against
the [k][n] kernel's bits, and what lies behind C's rows."""
import pytest
import torch

from effective_transformer_amd import kernel_ops as ko

pytestmark = pytest.mark.gpu


# one of every tile (row blocks x column blocks, d: two workgroups a CU) that a device of 256 CUs chooses, the last one rounds of them
TILES = [(49, 2152, 192), (40, 4112, 192), (258, 3304, 192), (4167, 72, 192), (289, 4120, 192), (291, 4120, 768), (676, 4112, 192), (5461, 136, 192),
         (5590, 328, 192), (5581, 328, 768), (5948, 648, 192), (5902, 648, 768), (5893, 1288, 192), (5471, 264, 768), (5464, 656, 192),
         (674, 4112, 768), (5379, 1032, 192), (4429, 1288, 768), (5394, 1544, 192), (5387, 1040, 2112), (5898, 1928, 192)]


@pytest.mark.parametrize("m,n,k", TILES)
@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("on_device", [False, True])
def test_every_tile(m, n, k, gelu, on_device):
    print("tile results", m, n, k, gelu, on_device, flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn(m, k, device="cuda", dtype=torch.float16, generator=g)
    w = torch.randn(k, n, device="cuda", dtype=torch.float16, generator=g).mul_(k ** -0.5)
    bias = torch.randn(n, device="cuda", dtype=torch.float16, generator=g)
    want = ko.gemm(a, w, bias=bias, gelu=gelu)
    bt = ko.transpose_weight(w)
    rows = m - 37 if on_device else m
    out = torch.full((m + 300, n), 7.0, device="cuda", dtype=torch.float16)
    ko.gemm_bt(a, bt, bias, m=m, out=out, gelu=gelu, m_dev=torch.tensor([rows], dtype=torch.int32, device="cuda") if on_device else None)
    assert torch.equal(out[:rows], want[:rows])
    assert (out[rows:] == 7.0).all()
    if not gelu:
        assert torch.equal(ko.gemm_bt(a, bt), ko.gemm(a, w))


# a C and a bias one, two and three values off the 8-byte boundaries, which C's stores of 2 to 16 bytes a lane then lie across; the last
# ones are few enough for tiles of 16 x 16, which such a C does not go to
@pytest.mark.parametrize("m,n,k", TILES + [(20, 768, 192), (5, 8, 256), (33, 40, 768)])
@pytest.mark.parametrize("on_device", [False, True])
def test_results_off_their_boundaries(m, n, k, on_device):
    print("off the boundaries", m, n, k, on_device, flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn(m, k, device="cuda", dtype=torch.float16, generator=g)
    w = torch.randn(k, n, device="cuda", dtype=torch.float16, generator=g).mul_(k ** -0.5)
    values = torch.randn(n + 8, device="cuda", dtype=torch.float16, generator=g)
    bt = ko.transpose_weight(w)
    rows = max(m - 7, 0) if on_device else m
    count = torch.tensor([rows], dtype=torch.int32, device="cuda") if on_device else None
    for shift in (1, 2, 3):
        bias = values[shift:shift + n]
        for gelu in (False, True):
            want = ko.gemm(a, w, bias=bias.clone(), gelu=gelu)
            room = torch.full((m * n + 16,), 7.0, device="cuda", dtype=torch.float16)
            ko.gemm_bt(a, bt, bias, out=room[shift:shift + m * n].view(m, n), gelu=gelu, m_dev=count)
            assert torch.equal(room[shift:shift + rows * n].view(rows, n), want[:rows]), (shift, gelu)
            assert (room[:shift] == 7.0).all() and (room[shift + rows * n:] == 7.0).all(), (shift, gelu)


# turned weights, which leave through a descriptor as well
@pytest.mark.parametrize("k,n", [(64, 64), (72, 200), (768, 40)])
def test_turned_weights_off_their_boundaries(k, n):
    w = torch.randn(k, n, device="cuda", dtype=torch.float16)
    for shift in (1, 2, 3):
        room = torch.full((n * k + 16,), 7.0, device="cuda", dtype=torch.float16)
        ko.transpose_weight(w, out=room[shift:shift + n * k].view(n, k))
        assert torch.equal(room[shift:shift + n * k].view(n, k), w.t())
        assert (room[:shift] == 7.0).all() and (room[shift + n * k:] == 7.0).all()


# rows of C so long that a tile's last one lies more than 4 GB behind its first
def test_longest_rows():
    m, n, k = 33, (1 << 26) + 8, 64
    print("longest rows", m, n, k, flush=True)
    g = torch.Generator(device="cuda").manual_seed(3)
    a = torch.randn(m, k, device="cuda", dtype=torch.float16, generator=g)
    bt = torch.empty(n, k, device="cuda", dtype=torch.float16)
    picks = [0, 1000, (1 << 24) - 8, (1 << 25) + 16, n - 264]
    for p in picks:
        bt[p:p + 264] = torch.randn(264, k, device="cuda", dtype=torch.float16, generator=g)
    out = ko.gemm_bt(a, bt, out=torch.empty(m, n, device="cuda", dtype=torch.float16))
    for p in picks:
        assert torch.equal(out[:, p:p + 264], ko.gemm_bt(a, bt[p:p + 264].contiguous())), p


# ... and a C and a bias off the 8-byte boundaries: the last row of the first 32 begins behind 4 GB (from 69 273 672 columns on), a lane's first
# row does (80 000 008), two tiles of rows; once with a row count on the device
@pytest.mark.parametrize("m,n,shift,on_device", [(33, 69273672, 1, False), (33, 80000008, 2, True), (200, (1 << 24) + 8, 3, False)])
def test_longest_rows_off_their_boundaries(m, n, shift, on_device):
    k = 64
    print("longest rows off their boundaries", m, n, shift, on_device, flush=True)
    g = torch.Generator(device="cuda").manual_seed(m + n)
    a = torch.randn(m, k, device="cuda", dtype=torch.float16, generator=g)
    bt = torch.empty(n, k, device="cuda", dtype=torch.float16)
    bias = torch.randn(n + 8, device="cuda", dtype=torch.float16, generator=g)[shift:shift + n]
    picks = [0, 1000, (1 << 23) - 8, n // 2 + 16, n - 264]
    for p in picks:
        bt[p:p + 264] = torch.randn(264, k, device="cuda", dtype=torch.float16, generator=g)
    rows = m - 2 if on_device else m
    room = torch.full((m * n + 8,), 7.0, device="cuda", dtype=torch.float16)
    out = room[shift:shift + m * n].view(m, n)
    ko.gemm_bt(a, bt, bias, out=out, m_dev=torch.tensor([rows], dtype=torch.int32, device="cuda") if on_device else None)
    for p in picks:
        want = ko.gemm_bt(a, bt[p:p + 264].contiguous(), bias[p:p + 264].contiguous())
        assert torch.equal(out[:rows, p:p + 264], want[:rows]), p
    assert (out[rows:] == 7.0).all() and (room[:shift] == 7.0).all() and (room[shift + m * n:] == 7.0).all()
