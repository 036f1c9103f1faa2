"""
65 to 512 features by one fp16 product per feature, in calls large enough for it: labels and distances are bit for bit those
of the kernels that a call with less scratch takes.

Shapes at the edges of the tiles; a kernel's way through many tiles (looking first given up and taken up again); rows left
open that fill several lists; and the line from which on the kernel runs.
"""
import pytest
import torch

from heat_amd import _native
from test_gpu_fp32_products import _data
from test_gpu_panel import KINDS, _call

pytestmark = pytest.mark.gpu


def _rows(kind, n, d, k, dev):
    g = torch.Generator(device=dev).manual_seed(1000 * d + k)
    if kind == "noise":
        x = torch.randn((n, d), generator=g, device=dev)
    else:
        box, sigma = {"blobs": (5.0, 0.5), "far": (100.0, 1.0)}[kind]
        centre = (torch.rand((k, d), generator=g, device=dev) * 2 - 1) * box
        x = torch.randn((n, d), generator=g, device=dev) * sigma
        x += centre[torch.randint(k, (n,), generator=g, device=dev)]
    assert k <= n  # the centroids are rows
    return x, x[torch.randperm(n, generator=g, device=dev)[:k]].clone()


def _scratch(n, d, k):
    need = _native.workspace_bytes(n, d, k, _native.WS_ASSIGN)
    return need, need // 256 * 256 - 256  # with and without room for the fp16 centroids


def _compare(x, c):
    n, d = x.shape
    got = []
    for nbytes in _scratch(n, d, c.shape[0]):
        lab = torch.full((n,), -7, dtype=torch.int32, device=x.device)
        md = torch.full((n,), -1.0, device=x.device)
        alone = lab.clone()
        _call(x, c, lab, md, nbytes)
        _call(x, c, alone, None, nbytes)
        assert torch.equal(lab, alone)
        got.append((lab, md.view(torch.int32)))
    assert torch.equal(got[0][0], got[1][0]), int((got[0][0] != got[1][0]).sum())
    assert torch.equal(got[0][1], got[1][1]), int((got[0][1] != got[1][1]).sum())


def _runs(n, d, k, dev):
    """Whether a call lays out fp16 centroids: they are the last thing in its scratch."""
    x, c = _rows("noise", n, d, k, dev)
    need = _native.workspace_bytes(n, d, k, _native.WS_ASSIGN)
    ws = torch.full((need,), 0xAB, dtype=torch.uint8, device=dev)
    lab = torch.empty(n, dtype=torch.int32, device=dev)
    _native.check(_native.load().hkm_assign_f32(x.data_ptr(), n, d, d, c.data_ptr(), c.shape[0], d, lab.data_ptr(), None, ws.data_ptr(),
                                                need, torch.cuda.current_stream().cuda_stream))
    return bool((ws[-4096:] != 0xAB).any())


EDGES = [(32000, 65, 1000), (32226, 75, 993), (15625, 100, 2048), (246200, 128, 130), (7813, 128, 4096), (620160, 129, 129),
         (249300, 139, 321), (80001, 140, 1000), (249513, 267, 513), (266667, 200, 300), (332469, 268, 385), (249513, 300, 513),
         (128000, 500, 1000), (125000, 512, 1024), (992249, 300, 129), (64001, 200, 1000), (128000, 268, 500), (62500, 512, 1024),
         (15625, 431, 4096)]


@pytest.mark.parametrize("i,shape", list(enumerate(EDGES)))
def test_edges(i, shape):
    n, d, k = shape
    dev = torch.device("cuda")
    assert _runs(n, d, k, dev)
    for kind in ("blobs", ("far", "noise")[i % 2]):
        _compare(*_rows(kind, n, d, k, dev))


@pytest.mark.parametrize("shape", [(32226, 75, 993), (32001, 100, 1000), (80001, 140, 1000), (128001, 268, 1000)])
@pytest.mark.parametrize("kind", KINDS)
def test_kinds_of_data(kind, shape):
    _compare(*_data(kind, *shape, torch.device("cuda")))


@pytest.mark.parametrize("shape", [(32001, 100, 1000), (80001, 200, 1000), (246200, 128, 130), (332469, 268, 385)])
@pytest.mark.parametrize("odd", [None, float("nan"), 1e25])
def test_rows_and_centroids_out_of_range(shape, odd):
    x, c = _rows("blobs", *shape, torch.device("cuda"))
    x[5::97] = float("nan")
    x[7::101] = 1e30
    x[11::103, 3] = float("inf")
    if odd is not None:
        c[17] = odd
    _compare(x, c)


def test_strided_rows():
    n, d, k = 80001, 131, 1000
    dev = torch.device("cuda")
    x0, c0 = _rows("blobs", n, d, k, dev)
    x, c = (torch.full((t.shape[0], d + 3), 1e9, device=dev) for t in (x0, c0))
    x[:, 1 : d + 1], c[:, 1 : d + 1] = x0, c0
    lab, want = (torch.empty(n, dtype=torch.int32, device=dev) for _ in range(2))
    need, small = _scratch(n, d, k)
    _call(x[:, 1 : d + 1], c[:, 1 : d + 1], lab, None, need)
    _call(x0, c0, want, None, small)
    assert torch.equal(lab, want)
    _compare(x[:, 1 : d + 1], c[:, 1 : d + 1])


# Rows far from the centroids' scale stay open.  A workgroup (512 of 128 rows a tile; 256 from 268 features on) that met three
# tiles of them leaves out the next 29, looks at one, and goes on either way: more than 64 tiles each, open for the first
# 10 (taken up again when the rows are decidable), 36 (given up, looked at, given up again), or in turn.
@pytest.mark.parametrize("wgs,d,k", [(512, 65, 300), (256, 268, 400)])
@pytest.mark.parametrize("open_tiles", ["10", "36", "thirds"])
def test_given_up_and_taken_up_again(wgs, d, k, open_tiles):
    dev = torch.device("cuda")
    n = 66 * wgs * 128 + 77
    x, c = _rows("blobs", n, d, k, dev)
    if open_tiles == "thirds":
        for t in range(0, 66, 3):
            x[t * wgs * 128 : (t + 1) * wgs * 128] += 3000.0
    else:
        x[: int(open_tiles) * wgs * 128] += 3000.0
    _compare(x, c)


# About one row in six is left open, and a range of rows (64 of them, 8 tiles of centroids) is looked through in seven parts.
@pytest.mark.parametrize("n,d,k", [(400003, 100, 1024), (400003, 300, 1000)])
def test_open_rows_fill_several_lists(n, d, k):
    dev = torch.device("cuda")
    x, c = _rows("blobs", n, d, k, dev)
    x[::6] += 3000.0
    _compare(x, c)


@pytest.mark.parametrize("shape,runs", [((31999, 100, 1000), False), ((32000, 100, 1000), True), ((63999, 200, 1000), False),
                                        ((64000, 200, 1000), True), ((62499, 300, 1024), False), ((62500, 300, 1024), True),
                                        ((128000, 512, 500), True), ((256514, 400, 499), True), ((256513, 400, 499), False),
                                        ((1000003, 200, 128), False), ((1000003, 129, 65), False)])
def test_line(shape, runs):
    assert _runs(*shape, torch.device("cuda")) == runs
