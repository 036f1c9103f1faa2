"""
The upper of two middle values: in the lower one's run of equals, in its last byte's histogram, or above every value that
shares its leading 24 bits (where the last pass finds it); with clusters around the rows per workgroup of both sizes.
Order statistics and one interpolation in float64: the same bits as from sorted values.
"""
import pytest
import torch

from heat_amd import _native

pytestmark = pytest.mark.gpu

KINDS = ["normal", "few values", "ulps", "two far values", "signs", "inf"]


def _values(kind, n, d, g):
    x = torch.randn((n, d), generator=g)
    if kind == "few values":
        x = torch.randint(-2, 3, (n, d), generator=g).float()
    elif kind == "ulps":  # all values within 200 ulps: the middle ones share 24 bits
        x = (torch.randint(0, 200, (n, d), generator=g) + 0x3F800000).to(torch.int32).view(torch.float32)
    elif kind == "two far values":
        x = torch.where(torch.rand((n, d), generator=g) < 0.5, -1e30, 1e-30)
    elif kind == "signs":
        x = torch.where(torch.rand((n, d), generator=g) < 0.5, -x.abs(), x.abs()) * 1e-40
    elif kind == "inf":
        x[torch.rand((n, d), generator=g) < 0.3] = float("inf")
    return x


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,d,sizes", [(40, 3, [2, 4, 1, 33]), (6144, 17, [1024, 1025, 2048, 2047]), (9000, 33, [4096, 4097, 806, 1])])
def test_median(n, d, sizes, kind):
    g = torch.Generator().manual_seed(n + d)
    x = _values(kind, n, d, g)
    lab = torch.repeat_interleave(torch.arange(len(sizes)), torch.tensor(sizes))
    assert len(lab) == n
    perm = torch.randperm(n, generator=g)
    lab = lab[perm].to(torch.int32)
    out = torch.empty((len(sizes), d), device="cuda")
    _native.update_median(x.cuda(), lab.cuda(), out, _native.Workspace(torch.device("cuda")))
    for k in range(len(sizes)):
        v = x[lab == k].sort(0).values.double()
        m = v.shape[0]
        lo, hi = v[(m - 1) // 2], v[m // 2]
        want = lo.float() if m % 2 else (lo + (hi - lo) * 0.5).float()
        assert torch.equal(torch.nan_to_num(out[k].cpu(), nan=-7.0), torch.nan_to_num(want, nan=-7.0)), (k, kind)


def test_median_of_many_rows():
    # more than 2 000 000 rows: the larger workgroups
    n = 2000002
    x = torch.randn((n, 2), generator=torch.Generator(device="cuda").manual_seed(1), device="cuda")
    out = torch.empty((1, 2), device="cuda")
    _native.update_median(x, torch.zeros(n, dtype=torch.int32, device="cuda"), out, _native.Workspace(x.device))
    v = x.sort(0).values.double()
    lo, hi = v[n // 2 - 1], v[n // 2]
    assert torch.equal(out[0], (lo + (hi - lo) * 0.5).float())


@pytest.mark.parametrize("n,k", [(61440, 1), (61439, 1), (122881, 1), (143361, 1), (204801, 2), (300001, 3)])  # 1024 to 4096 rows a workgroup
@pytest.mark.parametrize("d", [1, 5])
def test_median_of_few_clusters(n, k, d):
    g = torch.Generator().manual_seed(n)
    x = torch.randn((n, d), generator=g)
    lab = torch.randint(0, k, (n,), generator=g, dtype=torch.int32)
    out = torch.empty((k, d), device="cuda")
    _native.update_median(x.cuda(), lab.cuda(), out, _native.Workspace(torch.device("cuda")))
    for j in range(k):
        v = x[lab == j].sort(0).values.double()
        lo, hi = v[(len(v) - 1) // 2], v[len(v) // 2]
        assert torch.equal(out[j].cpu(), (lo + (hi - lo) * 0.5).float()), j


# around the lines between 1024, 2048 and 4096 rows a workgroup
@pytest.mark.parametrize("n,d,k", [(300000, 2, 3), (300001, 2, 3), (300001, 3, 111), (300001, 3, 112), (500000, 23, 4), (500001, 23, 4),
                                   (500001, 24, 4), (1200000, 24, 444), (1200000, 24, 445), (1200001, 24, 4),
                                   (1200000, 32, 64), (1200001, 24, 64), (2000001, 24, 64)])
def test_median_across_the_lines(n, d, k):
    g = torch.Generator(device="cuda").manual_seed(n + d + k)
    x = torch.randn((n, d), generator=g, device="cuda").mul_(4).round_()
    lab = torch.randint(0, k, (n,), generator=g, dtype=torch.int32, device="cuda")
    out = torch.empty((k, d), device="cuda")
    _native.update_median(x, lab, out, _native.Workspace(x.device))
    for j in {0, k // 2, k - 1}:
        v = x[lab == j].sort(0).values.double()
        lo, hi = v[(len(v) - 1) // 2], v[len(v) // 2]
        assert torch.equal(out[j], (lo + (hi - lo) * 0.5).float()), j
