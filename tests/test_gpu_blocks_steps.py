"""The block kernel where its tiles have few steps (offsets times chunks of 64 channels): fewer than the steps whose weights it holds, as
many, and more, for each width of its wavefronts' columns and with half a last chunk."""
import numpy as np
import pytest

from tests.test_gpu_blocks import run
from tests.util import gpu_map

pytestmark = pytest.mark.gpu


def _groups(shape, count):
    """`count` copies of a little shape of voxels, far from one another."""
    at = 6 * np.stack(np.meshgrid(np.arange(20), np.arange(20), np.arange(8), indexing="ij"), -1).reshape(-1, 3)[:count]
    pts = (at[:, None, :] + np.asarray(shape)[None, :, :]).reshape(-1, 3)
    pts = np.concatenate([np.zeros((len(pts), 1), int), pts], axis=1)
    return pts[np.lexsort(pts.T[::-1])].astype(np.int32)


SHAPES = {1: [[0, 0, 0]], 2: [[0, 0, 0], [0, 0, 1]], 3: [[0, 0, 0], [0, 0, 1], [0, 0, 2]], 4: [[0, 0, 0], [0, 0, 1], [0, 1, 0], [0, 1, 1]],
          8: [[x, y, z] for x in (0, 1) for y in (0, 1) for z in (0, 1)]}


@pytest.mark.parametrize("offsets", sorted(SHAPES))
@pytest.mark.parametrize("c_in", [64, 96, 128, 160, 320])
@pytest.mark.parametrize("c_out", [128, 192, 256])
def test_few_steps(offsets, c_in, c_out):
    km = gpu_map(_groups(SHAPES[offsets], 700 if c_in == 64 else 150), (3, 3, 3))
    run(km, c_in, c_out)
