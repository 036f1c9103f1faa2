"""
65 to 512 features, with and without scratch for the fp16 centroids of the kernel by one product per feature: labels and
distances are those of fp32 products in either.

These calls are too small for that kernel to run (test_gpu_panel_large has those); their shapes lie at the edges of its tiles.
The reference is the restatement of the fp32 arithmetic in test_gpu_fp32_products.
"""
import pytest
import torch

from heat_amd import _native
from test_gpu_fp32_products import _data, _reference

pytestmark = pytest.mark.gpu

SHAPES = [(7813, 65, 1024), (8065, 75, 993), (8001, 100, 1000), (62501, 128, 129), (123079, 140, 65), (40001, 139, 200),
          (41000, 129, 321), (26700, 267, 300), (26700, 268, 385), (15625, 300, 513), (8000, 500, 1000), (7813, 512, 1024)]
KINDS = ["blobs", "zeros", "twins", "sizes", "at 100", "columns", "counts"]


def _call(x, c, labels, min_d2, nbytes):
    n, d = x.shape
    ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    lib = _native.load()
    _native.check(lib.hkm_assign_f32(x.data_ptr(), n, d, x.stride(0), c.data_ptr(), c.shape[0], c.stride(0), labels.data_ptr(),
                                     min_d2.data_ptr() if min_d2 is not None else None, ws.data_ptr(), nbytes,
                                     torch.cuda.current_stream().cuda_stream))


@pytest.mark.parametrize("i,shape", list(enumerate(SHAPES)))
def test_as_fp32_products(i, shape):
    n, d, k = shape
    dev = torch.device("cuda")
    for kind in {"blobs", KINDS[i % len(KINDS)], KINDS[(i + 3) % len(KINDS)]}:
        x, c = _data(kind, n, d, k, dev)
        lab = torch.full((n,), -7, dtype=torch.int32, device=dev)
        alone = lab.clone()
        md = torch.full((n,), -1.0, device=dev)
        need = _native.workspace_bytes(n, d, k, _native.WS_ASSIGN)
        _call(x, c, lab, md, need)
        _call(x, c, alone, None, need)
        want, want_md, _ = _reference(x, c)
        assert torch.equal(lab.long(), want), (kind, int((lab.long() != want).sum()))
        assert torch.equal(alone, lab), kind
        assert torch.equal(md, want_md), kind
        # scratch without room for the fp16 centroids: the kernels that take none, the same results
        small = lab.clone().fill_(-7)
        _call(x, c, small, None, need // 256 * 256 - 256)
        assert torch.equal(small, lab), kind


def test_rows_and_centroids_out_of_range():
    n, d, k = 8000, 200, 1000
    dev = torch.device("cuda")
    x, c = _data("blobs", n, d, k, dev)
    x[5::97] = float("nan")
    x[7::101] = 1e30
    x[11::103, 3] = float("inf")
    lab, small = (torch.empty(n, dtype=torch.int32, device=dev) for _ in range(2))
    need = _native.workspace_bytes(n, d, k, _native.WS_ASSIGN)
    for odd in (None, float("nan"), 1e25):
        if odd is not None:
            c[17] = odd
        _call(x, c, lab, None, need)
        _call(x, c, small, None, need // 256 * 256 - 256)
        assert torch.equal(lab, small), odd


@pytest.mark.parametrize("shape", [(8001, 100, 1000), (8000, 200, 1000), (62501, 128, 129), (26700, 268, 385)])
@pytest.mark.parametrize("odd", [None, float("nan"), 1e25])
def test_distances_of_rows_out_of_range(shape, odd):
    # rows whose distances are all infinite or not numbers: the same bits as of the kernels that take no fp16 centroids
    n, d, k = shape
    dev = torch.device("cuda")
    x, c = _data("blobs", n, d, k, dev)
    x[5::97] = float("nan")
    x[7::101] = 1e30
    x[11::103, 3] = float("inf")
    if odd is not None:
        c[17] = odd
    need = _native.workspace_bytes(n, d, k, _native.WS_ASSIGN)
    got = []
    for nbytes in (need, need // 256 * 256 - 256):
        lab = torch.full((n,), -7, dtype=torch.int32, device=dev)
        md = torch.full((n,), -1.0, device=dev)
        _call(x, c, lab, md, nbytes)
        got.append((lab, md.view(torch.int32)))
    assert torch.equal(got[0][0], got[1][0])
    assert torch.equal(got[0][1], got[1][1])


def test_strided_rows():
    n, d, k = 9001, 131, 1000
    dev = torch.device("cuda")
    x0, c0 = _data("blobs", n, d, k, dev)
    x, c = (torch.full((t.shape[0], d + 3), 1e9, device=dev) for t in (x0, c0))
    x[:, 1 : d + 1], c[:, 1 : d + 1] = x0, c0
    lab, want = (torch.empty(n, dtype=torch.int32, device=dev) for _ in range(2))
    need = _native.workspace_bytes(n, d, k, _native.WS_ASSIGN)
    _call(x[:, 1 : d + 1], c[:, 1 : d + 1], lab, None, need)
    _call(x0, c0, want, None, need)
    assert torch.equal(lab, want)
