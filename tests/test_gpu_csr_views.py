"""CSR-coded views written with the pair lists (maps that have a row order) against those of a build without one."""
import pytest
import torch

from pcengine_amd import synth
from tests.util import gpu_map

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ks", [(3, 3, 3), (3, 3, 1), (1, 3, 3), (5, 1, 1), (1, 1, 1)])
@pytest.mark.parametrize("n,extent,batch", [(1, 3, 0), (64, 6, 0), (65, 5, 1), (5000, 20, 1), (5000, 60, 2), (9000, 24, 0)])
def test_views(ks, n, extent, batch):
    coords = synth.random_cloud(seed=n, n=n, extent=extent, batches=max(batch, 1))
    a = gpu_map(coords, ks, want_csr=True, batchsize=batch)
    b = gpu_map(coords, ks, want_csr=True, batchsize=batch, want_order=False)
    assert a.order is not None and b.order is None and a.M == b.M
    for name in ("imap", "omap", "icsr", "icode", "ocsr", "ocode", "islot", "oslot", "nbr_out"):
        assert torch.equal(getattr(a, name), getattr(b, name)), name
