"""
Direct Euclidean distances of large matrices, in 128 x 64 tiles: the same bits as small calls give, which take 64 x 64 ones
(every element is one chain over the features in both).  Row counts and widths around the edges of tiles and of the
staged chunks of 8, 16 and 24 features.
"""
import pytest
import torch

from heat_amd import _native

pytestmark = pytest.mark.gpu


def _pairwise(x, y, metric=_native.METRIC_EUCLID, sigma=1.0, ld=None):
    out = torch.full((x.shape[0], ld or y.shape[0]), -1.0, device=x.device)
    _native.pairwise(x, y, out[:, : y.shape[0]], metric, sigma)
    return out[:, : y.shape[0]]


def _blocks(x, y, out, metric, sigma=1.0):
    m, n = out.shape
    cuts = lambda s: sorted({0, min(s, 300), max(0, s // 2 - 150), min(s, s // 2 + 150), max(0, s - 300), s})
    for a, b in zip(cuts(m), cuts(m)[1:]):
        for c, d in zip(cuts(n), cuts(n)[1:]):
            if b - a <= 300 and d - c <= 300:
                assert torch.equal(out[a:b, c:d], _pairwise(x[a:b], y[c:d].clone(), metric, sigma)), (a, c)


@pytest.mark.parametrize("m,d", [(8192, 5), (8200, 8), (8256, 9), (8196, 16), (8320, 17), (8260, 18), (8192, 24), (8196, 25), (8200, 48)])
def test_against_itself(m, d):
    g = torch.Generator(device="cuda").manual_seed(m + d)
    x = torch.randn((m, d), generator=g, device="cuda")
    x[100] = x[m - 5]
    x[m - 77, 2] = float("nan")
    x[m // 2, 0] = float("inf")
    out = _pairwise(x, x)
    assert torch.equal(out.view(torch.int32), out.t().contiguous().view(torch.int32)) or torch.equal(
        torch.nan_to_num(out, nan=-7.0), torch.nan_to_num(out.t(), nan=-7.0))
    ok = torch.isfinite(x).all(1)
    assert bool((out.diagonal()[ok] == 0).all()) and float(out[100, m - 5]) == 0.0
    clean = torch.nan_to_num(x, nan=0.5, posinf=2.0)
    out = _pairwise(clean, clean)
    _blocks(clean, clean, out, _native.METRIC_EUCLID)


@pytest.mark.parametrize("m,n,d", [(8192, 4160, 6), (8190, 4163, 18), (16391, 2049, 33), (70, 300000, 12), (300001, 65, 7)])
def test_two_matrices(m, n, d):
    g = torch.Generator(device="cuda").manual_seed(m + n + d)
    x = torch.randn((m, d + 3), generator=g, device="cuda")[:, 1 : d + 1]
    y = torch.randn((n, d), generator=g, device="cuda")
    out = _pairwise(x, y)
    _blocks(x, y, out, _native.METRIC_EUCLID)
    gauss = _pairwise(x, y, _native.METRIC_GAUSS, 2.0, ld=(n + 7) // 4 * 4)
    _blocks(x, y, gauss, _native.METRIC_GAUSS, 2.0)
    rows = torch.arange(0, m, max(1, m // 50), device="cuda")
    want = (x[rows, None].double() - y[None].double()).pow(2).sum(2).sqrt()
    # d + 1 roundings of half an ulp each in the squared sum, one in the root
    assert bool(((out[rows].double() - want).abs() <= (0.5 * (d + 2) + 1) * 2.0**-23 * want + 1e-30).all())


# on both sides of the lines between large and small tiles
@pytest.mark.parametrize("m,d", [(8224, 8), (8320, 16), (8196, 17), (8208, 8), (8208, 16), (8200, 5), (8212, 9)])
def test_against_itself_at_the_lines(m, d):
    test_against_itself(m, d)


@pytest.mark.parametrize("m,n,d", [(1024, 40000, 32), (1023, 40000, 32), (1024, 35003, 9), (530000, 64, 5), (530001, 63, 16),
                                   (960, 40000, 9), (959, 40000, 9), (12288, 8192, 36), (12161, 8192, 33), (12161, 8191, 36), (12288, 8192, 37)])
def test_two_matrices_at_the_lines(m, n, d):
    test_two_matrices(m, n, d)
