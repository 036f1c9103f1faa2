"""
The float64 step of few clusters in one pass: labels, smallest distances and means are the same bits as those of the
assignment and the update called one after the other, at the edges of its tiles and with rows at any 8-byte boundary.
"""
import pytest
import torch

from heat_amd import _native

pytestmark = pytest.mark.gpu

SHAPES = [(4096, 1, 1), (4097, 2, 16), (5000, 3, 17), (9999, 8, 32), (20011, 9, 5), (70001, 15, 16), (4100, 16, 31), (33000, 17, 2),
          (131072, 18, 16), (131073, 23, 32), (131199, 24, 7), (600001, 13, 12), (600001, 13, 13), (499999, 9, 16), (600001, 14, 16), (300007, 25, 16), (50000, 31, 32), (50000, 32, 16), (50000, 31, 33)]


def _both(x, c):
    n, d = x.shape
    k = c.shape[0]
    dev = x.device
    ws = _native.Workspace(dev)
    lab, want_lab = torch.full((2, n), -7, dtype=torch.int32, device=dev)
    new, want_new = torch.full((2, k, d), -1.0, dtype=torch.float64, device=dev)
    shift, sse = (torch.empty((), dtype=torch.float64, device=dev) for _ in range(2))
    _native.lloyd_step(x, c, new, lab, shift, sse, ws)
    md = torch.empty((n,), dtype=torch.float64, device=dev)
    _native.assign(x, c, want_lab, md, ws)
    _native.update(x, want_lab, want_new, torch.empty((k,), dtype=torch.int64, device=dev), ws)
    torch.cuda.synchronize()
    assert torch.equal(lab, want_lab)
    assert torch.equal(new.view(torch.int64), want_new.view(torch.int64))
    return new, shift, sse, md


@pytest.mark.parametrize("n,d,k", SHAPES)
@pytest.mark.parametrize("pad", [0, 3])
def test_as_assignment_and_update(cuda, n, d, k, pad):
    g = torch.Generator(device="cuda").manual_seed(n + d + k)
    x = torch.randn((n, d + pad), generator=g, device=cuda, dtype=torch.float64)[:, pad // 2 : pad // 2 + d]
    if pad == 0:
        x = x.contiguous()
    c = x[torch.randperm(n, generator=g, device=cuda)[:k]].clone()
    if k > 2:
        c[2] = c[0]  # equal centroids: the first wins, the other is empty
    new, shift, sse, md = _both(x, c)
    # sums of squares in another order: n 2^-53 of the sum, twice
    assert abs(float(shift) - float(((c - new) ** 2).sum())) <= 2 * k * d * 2.0**-53 * float(shift) + 1e-300
    assert abs(float(sse) - float(md.sum())) <= 2 * n * 2.0**-53 * float(sse)


def test_not_finite(cuda):
    n, d, k = 50000, 18, 16
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((n, d), generator=g, device=cuda, dtype=torch.float64)
    c = x[:k].clone()
    inf, nan = float("inf"), float("nan")
    for r, col, v in [(11111, 0, inf), (40000, 17, -inf), (777, 5, nan), (30001, 7, inf), (n - 1, 17, nan)]:
        x[r, col] = v
    _both(x, c)
    c[3, 4] = nan
    c[9, 0] = inf
    _both(x, c)
