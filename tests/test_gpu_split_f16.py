"""
The fp16-split matrix-core kernels: rows and centroids whose magnitudes leave the shared scale, non-finite rows, odd
widths, unaligned rows, the edges of tiles and blocks.

Tolerance of a squared distance, in units of u = 2^-24 (|x|^2 + |c|^2): the parts of an operand miss it by at most 2^-22
and the dropped product is below 2^-22 of |x c|, 3 * 4 u in all; three sums per 16 features, at most one u each; norms
of D terms, at most D / 8 + 4 u; final sum 1 u: (18 + 3 D / 16 + D / 8) u.
"""
import pytest
import torch

from heat_amd import _native

pytestmark = pytest.mark.gpu


def _check(x, c, lab, md):
    xd, cd = x.double(), c.double()
    ok = torch.isfinite(xd).all(1)
    xn, cn = (xd * xd).sum(1), (cd * cd).sum(1)
    d2 = ((xd[ok][:, None] - cd[None]) ** 2).sum(2)
    lab = lab.long()[ok]
    u = 2.0**-24 * (xn[ok] + cn[lab])
    tol = (18 + 5 * x.shape[1] / 16) * u + 1e-37
    got = d2.gather(1, lab[:, None])[:, 0]
    assert torch.all((md.double()[ok] - got).abs() <= tol)
    best, arg = d2.min(1)
    # the centroid chosen is the nearest one up to the error of both distances
    assert torch.all(got - best <= tol + (18 + 5 * x.shape[1] / 16) * 2.0**-24 * (xn[ok] + cn[arg]))


def _assign(x, c):
    lab = torch.full((x.shape[0],), -7, dtype=torch.int32, device=x.device)
    md = torch.full((x.shape[0],), -1.0, device=x.device)
    _native.assign(x, c, lab, md, _native.Workspace(x.device))
    return lab, md


@pytest.mark.parametrize("n,d,k", [(1, 17, 40), (63, 32, 33), (64, 32, 64), (65, 25, 96), (513, 31, 256), (1000, 33, 97),
                                   (777, 48, 128), (515, 50, 100), (2049, 63, 31), (400, 64, 200), (4097, 20, 500),
                                   # wide rows: tiles of 256 rows and 64 or 128 centroids, chunks of 32 features
                                   (255, 129, 64), (257, 160, 65), (600, 131, 7), (1025, 190, 129), (300, 257, 300),
                                   (90, 96, 500)])
@pytest.mark.parametrize("kind", ["plain", "rows", "centroids", "features"])
def test_assignment_over_magnitudes(cuda, n, d, k, kind):
    g = torch.Generator().manual_seed(n + d + k)
    x = torch.randn((n, d), generator=g)
    c = torch.randn((k, d), generator=g)
    if kind == "rows":  # rows from 1e-8 to 1e8 times the centroids' size, some of them zero
        x *= 10.0 ** (16 * torch.rand((n, 1), generator=g) - 8)
        x[::7] = 0.0
    elif kind == "centroids":  # centroids of all sizes, one of them zero
        c *= 10.0 ** (10 * torch.rand((k, 1), generator=g) - 5)
        c[k // 2] = 0.0
        x *= 10.0 ** (8 * torch.rand((n, 1), generator=g) - 4)
    elif kind == "features":
        s = 10.0 ** (6 * torch.rand((1, d), generator=g) - 3)
        x, c = x * s, c * s
    x, c = x.to(cuda), c.to(cuda)
    lab, md = _assign(x, c)
    assert int(lab.min()) >= 0 and int(lab.max()) < k
    _check(x, c, lab, md)
    # a row's result does not depend on the rows beside it
    lab2, md2 = _assign(x.flip(0).contiguous(), c)
    assert torch.equal(lab2.flip(0), lab) and torch.equal(md2.flip(0), md)
    # rows at any 4-byte boundary, wider leading dimension
    wide = torch.full((n, d + 3), float("nan"), device=cuda)
    wide[:, 1 : d + 1] = x
    lab3, md3 = _assign(wide[:, 1 : d + 1], c)
    assert torch.equal(lab3, lab) and torch.equal(md3, md)


@pytest.mark.parametrize("n,d,k", [(700, 160, 200), (300, 131, 60)])
def test_non_finite_rows_and_centroids_of_wide_rows(cuda, n, d, k):
    # as the fp32 products order them: a NaN among |c|^2 - 2 x.c counts as distance 0, the first one wins
    g = torch.Generator().manual_seed(d)
    x, c = torch.randn((n, d), generator=g), torch.randn((k, d), generator=g)
    want, want_md = _assign(x.to(cuda), c.to(cuda))
    y = x.clone()
    y[5, 3] = float("inf")
    y[130, 0] = float("nan")
    lab, md = _assign(y.to(cuda), c.to(cuda))
    rest = torch.ones(n, dtype=torch.bool)
    rest[[5, 130]] = False
    assert torch.equal(lab.cpu()[rest], want.cpu()[rest]) and torch.equal(md.cpu()[rest], want_md.cpu()[rest])
    assert int(lab[5]) == int((c[:, 3] > 0).nonzero()[0]) and float(md[5]) == 0.0
    assert int(lab[130]) == 0 and float(md[130]) == 0.0
    c2 = c.clone()
    c2[k - 1, 2] = float("nan")
    lab, md = _assign(x.to(cuda), c2.to(cuda))
    assert bool((lab == k - 1).all()) and bool((md == 0).all())
    c2[k - 1, 2] = float("inf")  # wins for the rows on its side
    lab, md = _assign(x.to(cuda), c2.to(cuda))
    side = (x[:, 2] > 0).to(cuda)
    assert bool((lab[side] == k - 1).all()) and not bool((lab[~side] == k - 1).any())
    c3 = c.clone()
    c3[1] = 2.0e19  # |c|^2 overflows: infinitely far
    lab, md = _assign(x.to(cuda), c3.to(cuda))
    assert not bool((lab == 1).any())


@pytest.mark.parametrize("n,d,k", [(300, 32, 64), (300, 50, 100), (300, 20, 40)])
def test_non_finite_rows_and_centroids(cuda, n, d, k):
    g = torch.Generator().manual_seed(d)
    x, c = torch.randn((n, d), generator=g), torch.randn((k, d), generator=g)
    want, want_md = _assign(x.to(cuda), c.to(cuda))
    y = x.clone()
    y[5, 3] = float("inf")
    y[70, d - 1] = -float("inf")
    y[130, 0] = float("nan")
    y[200] = 2.0e19  # |x|^2 overflows
    lab, md = _assign(y.to(cuda), c.to(cuda))
    rest = torch.ones(n, dtype=torch.bool)
    rest[[5, 70, 130, 200]] = False
    assert torch.equal(lab.cpu()[rest], want.cpu()[rest]) and torch.equal(md.cpu()[rest], want_md.cpu()[rest])
    # an infinite coordinate: the first centroid with -2 x c = -inf, as |c|^2 - 2 x.c orders them
    assert int(lab[5]) == int((c[:, 3] > 0).nonzero()[0]) and int(lab[70]) == int((c[:, d - 1] < 0).nonzero()[0])
    assert int(lab[130]) == 0
    assert int(lab[200]) == int(c.double().sum(1).argmax())
    # centroids that are not finite never win
    c2 = c.clone()
    c2[1] = float("nan")
    c2[k - 1, 2] = float("inf")
    lab, md = _assign(x.to(cuda), c2.to(cuda))
    assert not bool(((lab == 1) | (lab == k - 1)).any())
    keep = torch.tensor([i for i in range(k) if i not in (1, k - 1)])
    _check(x.to(cuda), c.to(cuda)[keep.to(cuda)], torch.searchsorted(keep, lab.cpu().long()).int().to(cuda), md)


@pytest.mark.parametrize("n,d,k", [(5000, 32, 256), (3001, 50, 100), (2000, 18, 490), (4000, 48, 70)])
def test_step_sums_rows_of_all_magnitudes(cuda, n, d, k):
    g = torch.Generator().manual_seed(n)
    x = torch.randn((n, d), generator=g) * 10.0 ** (4 * torch.rand((n, 1), generator=g) - 2)
    c = x[torch.randperm(n, generator=g)[:k]].clone()
    x, c = x.to(cuda), c.to(cuda)
    lab, _ = _assign(x, c)
    ws = _native.Workspace(cuda)
    new, lab2, shift = torch.empty_like(c), torch.empty_like(lab), torch.empty((), device=cuda)
    _native.lloyd_step(x, c, new, lab2, shift, None, ws)
    assert torch.equal(lab, lab2)
    cnt = torch.bincount(lab.long(), minlength=k)
    ref = torch.zeros((k, d), dtype=torch.float64, device=cuda).index_add_(0, lab.long(), x.double())
    ref = ref / cnt.clamp(min=1).double()[:, None]
    # rows rounded to 2^-28 of at most four times their norm or of 2^6 times the smallest centroid norm; where the rows
    # of a workgroup span too many magnitudes the two-pass update adds them in fp32: 2^-24 per addition
    norm = x.double().norm(dim=1)
    top = torch.zeros(k, dtype=torch.float64, device=cuda).scatter_reduce_(0, lab.long(), norm, "amax")
    top = torch.maximum(top, c.double().norm(dim=1).min())
    tol = 2.0**-24 * (ref.abs() + (cnt.clamp(min=4) * top)[:, None])
    assert torch.all((new.double() - ref).abs() <= tol)


@pytest.mark.parametrize("n,d", [(1, 3), (63, 2), (64, 18), (65, 33), (200, 7), (1003, 18), (321, 5)])
@pytest.mark.parametrize("metric", [_native.METRIC_EUCLID_QE, _native.METRIC_EUCLID, _native.METRIC_GAUSS,
                                    _native.METRIC_MANHATTAN])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_matrix_against_itself_has_the_bits_of_the_general_case(cuda, n, d, metric, dtype):
    # (the expansion of wide float32 rows runs on the matrix cores, the same kernel both times)
    g = torch.Generator().manual_seed(n + d)
    x = torch.randn((n, d), generator=g, dtype=dtype).to(cuda)
    x[0, d - 1] = float("nan")
    same, other = torch.empty((n, n), dtype=dtype, device=cuda), torch.empty((n, n), dtype=dtype, device=cuda)
    _native.pairwise(x, x, same, metric, 1.0)
    _native.pairwise(x, x.clone(), other, metric, 1.0)
    kind = torch.int32 if dtype == torch.float32 else torch.int64
    nan = torch.isnan(other)
    assert torch.equal(torch.isnan(same), nan) and torch.equal(same.view(kind)[~nan], other.view(kind)[~nan])
