"""Maxima of coordinate columns in one launch, against torch's, and what is left to torch."""
import pytest
import torch

import pcengine_amd as pe
from pcengine_amd import _lib, backend
from tests.util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 150001, 256 * 1024 + 1, 700000])
@pytest.mark.parametrize("width", [2, 3, 4])
def test_against_torch(n, width):
    g = torch.Generator(device=DEV).manual_seed(n)
    c = torch.randint(-2 ** 31, 2 ** 31 - 1, (n, width), generator=g, device=DEV, dtype=torch.int64).int()
    assert backend.coords_upper(c) == c[:, 1:].amax(dim=0).tolist()
    c[:, 1:] = -5 - c[:, 1:].abs() // 2
    c[n - 1, width - 1] = -1                 # the last row counts
    assert backend.coords_upper(c) == c[:, 1:].amax(dim=0).tolist()
    assert pe.spTensor(torch.zeros((n, 1), device=DEV), c).coords_max == c[:, 1:].amax(dim=0).tolist()


def test_other_layouts_go_to_torch():
    c = torch.randint(0, 100, (50, 8), device=DEV, dtype=torch.int32)
    for t in (c, c[:, :4], c.long(), c.cpu(), c.float()):
        assert pe.spTensor(t, t).coords_max == t[:, 1:].amax(dim=0).tolist()
    with pytest.raises((RuntimeError, IndexError)):
        pe.spTensor(c, torch.zeros((0, 4), dtype=torch.int32, device=DEV))
    ws, up = torch.empty(1, dtype=torch.uint8, device=DEV), (_lib.c_int32 * 3)()
    lib = _lib.load()
    assert lib.pce_column_max(c.data_ptr(), 50, 5, ws.data_ptr(), 1 << 20, up, 0) == _lib.PCE_EINVAL
    assert lib.pce_column_max(c.data_ptr(), 50, 4, ws.data_ptr(), 1, up, 0) == _lib.PCE_EWORKSPACE
