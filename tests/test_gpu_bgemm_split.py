"""The GEMM kernel that splits the depth over a block's waves: four and eight of them, depths that end inside a unit and inside a batch
of units, both sides of the switch, and matrices that are addressed by pointer because a row, or the filters, are too long for 32 bits."""
import pytest
import torch

import dabnn_amd as dab

pytestmark = pytest.mark.gpu


def words(g, *shape):
    return torch.randint(-2**63, 2**63 - 1, shape, dtype=torch.int64, device="cuda", generator=g)


def counts(a, b):
    """Mismatches of columns of a [k][m] and rows of b [n][k], whole numbers from +-1 products."""
    bits = torch.arange(64, device="cuda")
    pm = lambda w: ((w.unsqueeze(-1) >> bits) & 1).float().mul_(-2).add_(1)
    k = a.shape[0]
    pa, pb = pm(a.T.contiguous()).reshape(a.shape[1], k * 64), pm(b).reshape(b.shape[0], k * 64)
    return (k * 64 - pb @ pa.T) / 2


def check(m, n, k, lda, ldb, g):
    a, b = torch.empty((k, lda), dtype=torch.int64, device="cuda"), torch.empty((n, ldb), dtype=torch.int64, device="cuda")
    a[:, :m], b[:, :k] = words(g, k, m), words(g, n, k)
    if lda > m:
        a[:, m:m + 64] = -1  # what no output may see
    if ldb > k:
        b[:, k:k + 64] = -1
    want = counts(a[:, :m].contiguous(), b[:, :k].contiguous())
    c = torch.full((n, m), 3.0, device="cuda")
    dab.bgemm(m, n, k, a, lda, b, ldb, c, m)
    assert torch.equal(c, want + 3)
    dab.bgemm_overwrite(m, n, k, a, lda, b, ldb, c, m)
    assert torch.equal(c, want)


@pytest.mark.parametrize("m,n,k", [(40, 33, k) for k in (13, 16, 17, 31, 32, 33, 44, 45, 47, 48, 49, 63, 64, 65, 96, 97, 128, 129, 160)] +
                         [(32, 512 * 32, 48), (32, 513 * 32, 48), (32, 513 * 32, 49), (32, 513 * 32, 33), (32, 512 * 32 - 5, 45), (200, 1000, 150), (512, 1024, 72), (510, 1023, 71)])
def test_waves_and_units(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    check(m, n, k, m + 1, k + 3, g)


@pytest.mark.parametrize("m,n,k,lda,ldb", [(40, 3, 50, 40, 2**23), (40, 3, 50, 40, 2**23 - 1), (40, 70, 80, 2**22, 80), (40, 70, 64, 2**22, 64), (40, 70, 63, 2**22, 63)])
def test_long_rows_and_filters(m, n, k, lda, ldb):
    g = torch.Generator(device="cuda").manual_seed(k)
    check(m, n, k, lda, ldb, g)


@pytest.mark.parametrize("n,h,cin,cout,k", [(1, 9, 64, 8, 5), (8, 14, 256, 256, 5), (2, 13, 192, 40, 5), (3, 7, 320, 24, 7), (2, 16, 128, 72, 4), (5, 11, 448, 96, 3)])
def test_windows(n, h, cin, cout, k):
    """Windows (a BinConv layer off fp32 input) against a +-1 convolution; padding is -1."""
    g = torch.Generator(device="cuda").manual_seed(n + cin + k)
    x, w = torch.randn((n, h, h, cin), device="cuda", generator=g), torch.randn((cout, k, k, cin), device="cuda", generator=g)
    packed = dab.pack_mat(w).reshape(cout, -1)
    if packed.shape[1] % 2:
        packed = torch.cat([packed, torch.zeros((cout, 1), dtype=torch.int64, device="cuda")], 1)
    got = dab.BinConv(packed.contiguous(), k, k, k // 2, k // 2, 1, 1)(x)
    sign = lambda t: torch.where(t > 0, 1.0, -1.0)
    p = k // 2
    xs = torch.nn.functional.pad(sign(x).permute(0, 3, 1, 2), (p, p, p, p), value=-1.0)
    want = (k * k * cin - torch.nn.functional.conv2d(xs.cpu(), sign(w).permute(0, 3, 1, 2).cpu())) / 2
    assert torch.equal(got.cpu(), want.permute(0, 2, 3, 1))
