"""
The float64 update of few clusters as a product of matrices: sums against plain float64 sums, counts exactly, at the
edges of its tiles (16 clusters, 16 columns with the column of counts among them, 4 rows, 64 rows a wave), the same bits
from call to call, and values that are not finite only in the means that they belong to.
"""
import pytest
import torch

from heat_amd import _native

pytestmark = pytest.mark.gpu

SHAPES = [(4096, 1, 1), (4097, 15, 16), (5000, 16, 17), (9999, 18, 16), (20011, 31, 33), (4100, 47, 32), (70001, 2, 128),
          (131, 18, 16), (33000, 127, 16), (6000, 63, 15), (300007, 18, 16)]


def _update(x, lab, k, counts=True):
    c = torch.full((k, x.shape[1]), -1.0, dtype=torch.float64, device=x.device)
    cnt = torch.full((k,), -1, dtype=torch.int64, device=x.device)
    _native.update(x, lab, c, cnt, _native.Workspace(x.device))
    return c, cnt


@pytest.mark.parametrize("n,d,k", SHAPES)
def test_means(n, d, k):
    g = torch.Generator(device="cuda").manual_seed(n + d + k)
    x = torch.randn((n, d + 2), generator=g, device="cuda", dtype=torch.float64)[:, 1 : d + 1] * 3 + 1
    lab = torch.randint(0, max(1, k - 1), (n,), generator=g, device="cuda", dtype=torch.int32)  # the last cluster is empty
    c, cnt = _update(x, lab, k)
    want_n = torch.bincount(lab.long(), minlength=k)
    assert torch.equal(cnt, want_n)
    sums = torch.zeros((k, d), dtype=torch.float64).index_add_(0, lab.cpu().long(), x.cpu())
    size = torch.zeros((k, d), dtype=torch.float64).index_add_(0, lab.cpu().long(), x.abs().cpu())
    den = want_n.cpu().clamp_min(1).float().double()[:, None]
    # two orders of adding n values of sum s of magnitudes differ by less than 2 n 2^-53 s
    bound = (2 * want_n.cpu().double()[:, None] + 4) * 2.0**-53 * size / den + 1e-300
    assert bool(((c.cpu() - sums / den).abs() <= bound).all())
    again, _ = _update(x, lab, k)
    assert torch.equal(c, again)


def test_not_finite():
    n, d, k = 50000, 18, 16
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn((n, d), generator=g, device="cuda", dtype=torch.float64)
    lab = torch.randint(0, k, (n,), generator=g, device="cuda", dtype=torch.int32)
    clean, _ = _update(x, lab, k)
    inf, nan = float("inf"), float("nan")
    put = [(11, 0, inf), (40000, 17, -inf), (77, 5, nan), (30001, 7, inf)]
    for r, col, v in put:
        x[r, col] = v
    other = int((lab == lab[30001]).nonzero()[-1])
    x[other, 7] = -inf
    c, _ = _update(x, lab, k)
    touched = torch.zeros((k, d), dtype=torch.bool, device="cuda")
    for r, col, v in put:
        touched[int(lab[r]), col] = True
        want = nan if (r, col) == (30001, 7) else v
        got = float(c[int(lab[r]), col])
        assert got == want or (want != want and got != got), (r, col, got)
    assert torch.equal(c[~touched], clean[~touched])


def test_step_as_assign_and_update():
    n, d, k = 40000, 18, 16
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((n, d), generator=g, device="cuda", dtype=torch.float64)
    c = x[:k].clone()
    lab, lab2 = (torch.empty(n, dtype=torch.int32, device="cuda") for _ in range(2))
    new = torch.empty_like(c)
    sh = torch.zeros((), dtype=torch.float64, device="cuda")
    ws = _native.Workspace(x.device)
    _native.lloyd_step(x, c, new, lab, sh, None, ws)
    _native.assign(x, c, lab2, None, ws)
    want, _ = _update(x, lab2, k)
    assert torch.equal(lab, lab2) and torch.equal(new, want)
    ref = ((want - c) ** 2).sum()
    assert abs(float(sh) - float(ref)) <= 1e-13 * float(ref)


# (rows, columns, clusters): the largest number of rows for the product of more than 32 clusters
LINES = [(2000000, 1, 48), (1000000, 3, 64), (1000000, 15, 80), (700000, 18, 48), (700000, 2, 112), (500000, 18, 64), (500000, 15, 128)]


@pytest.mark.parametrize("n,d,k", LINES)
@pytest.mark.parametrize("more", [0, 1])
def test_means_at_the_lines(n, d, k, more):
    test_means(n + more, d, k)


def test_many_clusters_of_many_rows_are_sorted():
    # the product's sums are part of the scratch: not behind the lines
    size = lambda n, d, k: _native.workspace_bytes(n, d, k, _native.WS_UPDATE | _native.WS_F64)
    for n, d, k in LINES:
        assert size(n, d, k) > size(n + 1, d, k) + 256 * k * (d + 1) * 8 - 10000
    for d, k in ((18, 32), (7, 48), (12, 64)):  # any number of rows
        assert size(4000001, d, k) >= size(4000000, d, k)
        assert size(4000000, d, k) > size(3000000, d, k)
