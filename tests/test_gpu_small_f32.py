"""fp32 layers and plain products in 32 x 32 tiles of 16 x 16 sums (few rows): tile edges, channel and column remainders, kernel
volumes, and with the offsets in shares, against float64 sums."""
import pytest
import torch

from pcengine_amd import backend, synth
from pcengine_amd.backend import DATAFLOW_OS
from tests.util import DEV, gpu_map

pytestmark = pytest.mark.gpu


def reference(f, w, km):
    f, w = f.double(), w.double()
    y = f @ w[km.kv // 2] if km.subm else torch.zeros((km.n_out, w.shape[2]), dtype=torch.float64, device=f.device)
    kpos = km.kpos.cpu().tolist()
    for k in range(km.kv):
        i, o = km.imap[kpos[k]:kpos[k + 1]].long(), km.omap[kpos[k]:kpos[k + 1]].long()
        if len(i):
            y.index_add_(0, o, f[i] @ w[k])
    return y


@pytest.mark.parametrize("n,extent", [(1, 2), (31, 6), (32, 6), (33, 6), (64, 4), (700, 9), (3000, 14)])
@pytest.mark.parametrize("c_in,c_out", [(4, 8), (20, 40), (36, 24), (64, 64), (100, 136), (256, 256)])
@pytest.mark.parametrize("ks,stride", [((3, 3, 3), (1, 1, 1)), ((2, 2, 2), (2, 2, 2)), ((1, 3, 3), (1, 1, 1))])
def test_layers(n, extent, c_in, c_out, ks, stride):
    if n == 1 and stride != (1, 1, 1):
        pytest.skip("the one voxel lies outside the coarse bound")
    km = gpu_map(synth.random_cloud(seed=n, n=n, extent=extent), ks, stride)
    f = torch.as_tensor(synth.features(1, km.n_in, c_in), device=DEV)
    w = torch.as_tensor(synth.weights(2, km.kv, c_in, c_out), device=DEV)
    b, r = (torch.as_tensor(synth.features(s, m, c_out), device=DEV) for s, m in ((3, 1), (4, km.n_out)))
    want = reference(f, w, km)
    # fp32 sums of fp32 products, rounded once per term: 2^-24 sqrt(terms) of their 2-norm, and the epilogue's few
    tol = 2 ** -24 * (km.kv * c_in + 4) ** 0.5
    for split in (False, True):
        got = backend.conv_forward(f, w, km, DATAFLOW_OS, split_offsets=split)
        assert ((got - want).norm() / want.norm()).item() <= tol, split
        got = backend.conv_forward(f, w, km, DATAFLOW_OS, split_offsets=split, bias=b[0], residual=r, act="relu")
        full = torch.relu(want + b[0].double() + r.double())
        assert ((got - full).norm() / full.norm()).item() <= 2 * tol, split


@pytest.mark.parametrize("n", [1, 31, 33, 2048, 5000])
@pytest.mark.parametrize("c_in,c_out", [(64, 8), (100, 40), (256, 256)])
def test_plain_products(n, c_in, c_out):
    f = torch.as_tensor(synth.features(1, n, c_in), device=DEV)
    w = torch.as_tensor(synth.weights(2, 1, c_in, c_out)[0], device=DEV)
    want = f.double() @ w.double()
    got = backend.dense_forward(f, w)
    assert ((got - want).norm() / want.norm()).item() <= 2 ** -24 * (c_in + 1) ** 0.5


def test_rows_of_a_tile_keep_to_themselves():
    """A NaN row reaches its neighbours only, an infinite weight the rows of the tiles that have the offset only."""
    km = gpu_map(synth.random_cloud(seed=9, n=400, extent=30), (3, 3, 3))
    f = torch.as_tensor(synth.features(1, km.n_in, 64), device=DEV)
    w = torch.as_tensor(synth.weights(2, 27, 64, 32), device=DEV)
    f[7, 3] = float("nan")
    got = backend.conv_forward(f, w, km, DATAFLOW_OS, split_offsets=False)
    reached = torch.zeros(km.n_out, dtype=torch.bool, device=DEV)
    reached[7] = True
    reached[km.omap[km.imap == 7].long()] = True
    assert torch.equal(torch.isnan(got).all(dim=1), reached) and torch.equal(torch.isnan(got).any(dim=1), reached)
