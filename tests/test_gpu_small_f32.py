"""fp32 layers and plain products in 32 x 32 tiles of 16 x 16 sums (few rows): tile edges, channel and column remainders, kernel
volumes, and with the offsets in shares, against float64 sums; and bit for bit against the tiles that many rows take."""
import numpy as np
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


# a product of up to 640, 1280 or 2560 tiles of 32 x 32 (64, 96, 256 channels) takes the small ones: 1501 rows do, 41 002 do not
@pytest.mark.parametrize("c_in,c_out", [(64, 64), (68, 64), (100, 40), (124, 36), (256, 256)])
def test_products_are_the_large_tiles_bit_for_bit(c_in, c_out):
    f = torch.as_tensor(synth.features(1, 41002, c_in), device=DEV)
    w = torch.as_tensor(synth.weights(2, 1, c_in, c_out)[0], device=DEV)
    b = torch.as_tensor(synth.features(3, 1, c_out)[0], device=DEV)
    for kw in (dict(), dict(bias=b, act="relu")):
        assert torch.equal(backend.dense_forward(f[:1501].clone(), w, **kw), backend.dense_forward(f, w, **kw)[:1501])


# a layer of up to 1280 tiles of 32 x 32 (5120 where the last chunk of 32 channels is full) takes the small ones: the cloud by
# itself does, so many copies of it do not
@pytest.mark.parametrize("c_in,c_out,copies,most", [(20, 40, 14, 1280), (36, 24, 26, 1280), (40, 136, 6, 1280), (64, 64, 50, 5120), (100, 136, 6, 1280),
                                                    (128, 40, 50, 5120)])
def test_layers_are_the_large_tiles_bit_for_bit(c_in, c_out, copies, most):
    one = synth.random_cloud(seed=4, n=3011, extent=15)
    one = one[np.lexsort(one[:, ::-1].T)]
    step = np.array([0, int(one[:, 1].max()) + 3, 0, 0], one.dtype)
    alone, many = (gpu_map(c, (3, 3, 3), batchsize=1) for c in (one, np.concatenate([one + k * step for k in range(copies)])))
    rows = alone.n_out
    assert -(-rows // 32) * -(-c_out // 32) <= 1280 and copies * rows // 32 * -(-c_out // 32) > most
    f = torch.as_tensor(synth.features(1, rows, c_in), device=DEV)
    w = torch.as_tensor(synth.weights(2, 27, c_in, c_out), device=DEV)
    b = torch.as_tensor(synth.features(3, 1, c_out)[0], device=DEV)
    for kw in (dict(), dict(bias=b, act="relu")):
        want = backend.conv_forward(f, w, alone, DATAFLOW_OS, split_offsets=False, **kw)
        got = backend.conv_forward(f.repeat(copies, 1), w, many, DATAFLOW_OS, split_offsets=False, **kw)
        assert all(torch.equal(part, want) for part in got.view(copies, rows, c_out))


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
    # the infinite weight: where a row has the offset, and nowhere in tiles of 32 rows none of which has it (a row without it
    # beside one that has it multiplies a zero)
    f[7, 3] = 0.5
    want = backend.conv_forward(f, w, km, DATAFLOW_OS, split_offsets=False)
    w[0, 9, 5] = float("inf")
    got = backend.conv_forward(f, w, km, DATAFLOW_OS, split_offsets=False)
    has, tiles = (torch.zeros(n, dtype=torch.bool, device=DEV) for n in (km.n_out, -(-km.n_out // 32)))
    at = km.omap[:int(km.kpos[1])].long()
    has[at], tiles[at // 32] = True, True
    tiles = tiles.repeat_interleave(32)[:km.n_out]
    assert has.any() and not tiles.all()
    other = torch.arange(32, device=DEV) != 5
    assert not torch.isfinite(got[has, 5]).any() and torch.equal(got[~tiles], want[~tiles]) and torch.equal(got[:, other], want[:, other])
