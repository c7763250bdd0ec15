"""Voxelisation through the cell bitmap and through the sort, and the collation kernel, against the oracle."""
import numpy as np
import pytest
import torch

import pcengine_amd as pe
from oracle import oracle as orc
from pcengine_amd import backend, utils
from tests.util import DEV

pytestmark = pytest.mark.gpu


def _points(n, side, dtype, seed):
    """n points whose voxels fill a box of side x side x side cells from corner to corner, some of them repeated."""
    rng = np.random.default_rng(seed)
    cells = rng.integers(0, side, size=(n, 3))
    cells[0], cells[-1] = 0, side - 1
    if n > 8:
        cells[1:n // 4] = cells[n // 2:n // 2 + n // 4 - 1]
    return ((cells - side // 2 + rng.uniform(0.1, 0.9, size=(n, 3))) * 0.5).astype(dtype)


# the bitmap takes a box of fewer than 32 (16 n + 65536 - 1) cells: 128^3 is that for one point, 161^3 is the first cube
# that is not for 4097
@pytest.mark.parametrize("n,side", [(1, 1), (2, 127), (2, 129), (255, 128), (257, 130), (4097, 161), (4097, 162), (4097, 500),
                                    (70001, 33), (70001, 300), (70001, 700)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_voxelize_both_ways(n, side, dtype):
    pts = _points(n, side, dtype, n + side)
    want, first, inverse = orc.sparse_quantize(pts, (0.5, 0.5, 0.5))
    pd = torch.as_tensor(pts, device=DEV)
    coords, index, inv, (lo, hi) = backend.voxelize(pd, 0.5, 5, return_index=True, return_inverse=True)
    c = coords.cpu().numpy()
    assert (c[:, 0] == 5).all() and np.array_equal(c[:, 1:], want)
    assert index.dtype == inv.dtype == torch.int32
    assert np.array_equal(index.cpu().numpy(), first) and np.array_equal(inv.cpu().numpy(), inverse)
    assert lo == want.min(0).tolist() and hi == want.max(0).tolist()
    coords, index, inv = utils.sparse_quantize(pd, 0.5, return_index=True, return_inverse=True)
    assert coords.dtype == torch.int32 and index.dtype == inv.dtype == torch.int64 and coords.is_contiguous()
    assert np.array_equal(coords.cpu().numpy(), want)
    assert np.array_equal(index.cpu().numpy(), first) and np.array_equal(inv.cpu().numpy(), inverse)


# boxes on both sides of the largest map, 16384 (16 n + 65536 - 1) cells: 1024^3 is that for two points, 1291^3 is the first
# cube that is not for 4097; 1 200 000 points in as many blocks are more than one round of the kernel that adds up the tiles
@pytest.mark.parametrize("n,side", [(2, 1024), (2, 1025), (300, 130), (4097, 1290), (4097, 1291), (70001, 900), (1200000, 1800)])
def test_voxelize_large_boxes(n, side):
    pts = _points(n, side, np.float32, n + side)
    want, first, inverse = orc.sparse_quantize(pts, (0.5, 0.5, 0.5))
    coords, index, inv = utils.sparse_quantize(torch.as_tensor(pts, device=DEV), 0.5, return_index=True, return_inverse=True)
    assert np.array_equal(coords.cpu().numpy(), want)
    assert np.array_equal(index.cpu().numpy(), first) and np.array_equal(inv.cpu().numpy(), inverse)


# the most points whose blocks have bitmaps of their own and more than those, in boxes on both sides of 2^31 cells
@pytest.mark.parametrize("n,side", [(1 << 22, 1200), (1 << 22, 1300), ((1 << 22) + 1, 1290), ((1 << 22) + 1, 1291), (4300001, 200)])
def test_voxelize_many_points(n, side):
    pts = _points(n, side, np.float32, side)
    want, first, inverse = orc.sparse_quantize(pts, (0.5, 0.5, 0.5))
    coords, index, inv = utils.sparse_quantize(torch.as_tensor(pts, device=DEV), 0.5, return_index=True, return_inverse=True)
    assert np.array_equal(coords.cpu().numpy(), want)
    assert np.array_equal(index.cpu().numpy(), first) and np.array_equal(inv.cpu().numpy(), inverse)


@pytest.mark.parametrize("rows", [[1], [3, 0, 5], [256, 257, 1], [70000, 1, 12345], [7] * 64, [7] * 65])
def test_collate(rows):
    rng = np.random.default_rng(len(rows))
    clouds = [torch.as_tensor(rng.integers(-50, 1000, size=(r, 3)).astype(np.int32), device=DEV) for r in rows]
    batch = utils.sparse_collate([pe.spTensor(torch.ones((len(c), 2), device=DEV), c, coords_max=[0, 0, 0]) for c in clouds])
    want = torch.cat([torch.cat([torch.full((len(c), 1), k, dtype=torch.int32, device=DEV), c], dim=1) for k, c in enumerate(clouds)])
    assert batch.coords.dtype == torch.int32 and torch.equal(batch.coords, want)
    assert batch.coords_max == want[:, 1:].amax(dim=0).tolist() and batch.batchsize == len(rows)
    assert (backend.collate_coords(clouds) is None) == (len(rows) > 64)


def test_collate_other_layouts():
    a = torch.tensor([[1, 2, 3], [4, 5, 6]], device=DEV)                 # int64
    b = torch.tensor([[9, 8, 7, 0]], dtype=torch.int32, device=DEV)[:, :3]
    batch = utils.sparse_collate([pe.spTensor(torch.ones((len(c), 1), device=DEV), c, coords_max=[0, 0, 0]) for c in (a, b)])
    assert batch.coords.tolist() == [[0, 1, 2, 3], [0, 4, 5, 6], [1, 9, 8, 7]] and batch.coords_max == [9, 8, 7]
