"""Collation of tensors that do not live on the current device: torch's operations take them, a launch would not."""
import torch
import pytest

import pcengine_amd as pe
from pcengine_amd import backend, utils
from tests.util import DEV

pytestmark = pytest.mark.gpu


def test_collation_follows_the_tensors_device(monkeypatch):
    clouds = [torch.tensor([[1, 2, 3], [4, 5, 6]], dtype=torch.int32, device=DEV), torch.tensor([[9, 0, 2]], dtype=torch.int32, device=DEV)]
    batch = lambda: utils.sparse_collate([pe.spTensor(torch.ones((len(c), 1), device=DEV), c, coords_max=[0, 0, 0]) for c in clouds])
    here = batch()
    assert backend.collate_coords(clouds) is not None
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    assert backend.collate_coords(clouds) is None
    there = batch()
    assert torch.equal(here.coords, there.coords) and here.coords_max == there.coords_max == [9, 5, 6]
