"""Kernel gradient of fp32 layers through LDS rings: tile, run, block and channel edges, against float64."""
import numpy as np
import pytest
import torch

from pcengine_amd import backend, synth
from tests.util import DEV, gpu_map

pytestmark = pytest.mark.gpu


def reference(x, g, km, transposed):
    kpos = km.kpos.cpu().tolist()
    want = torch.zeros((km.kv, x.shape[1], g.shape[1]), dtype=torch.float64, device=DEV)
    for k in range(km.kv):
        i, o = km.imap[kpos[k]:kpos[k + 1]].long(), km.omap[kpos[k]:kpos[k + 1]].long()
        i, o = (o, i) if transposed else (i, o)
        want[k] = x[i].double().t() @ g[o].double()
    if km.subm:
        want[km.kv // 2] += x.double().t() @ g.double()
    return want


@pytest.mark.parametrize("c_in,c_out", [(4, 4), (4, 64), (68, 20), (96, 96), (100, 128), (132, 196), (128, 64), (192, 100), (256, 384), (160, 4)])
@pytest.mark.parametrize("n,extent,ks,stride,transposed", [
    (1, 2, (3, 3, 3), (1, 1, 1), False), (40, 30, (3, 3, 3), (1, 1, 1), False), (127, 6, (3, 3, 3), (1, 1, 1), False),
    (130, 6, (1, 1, 3), (1, 1, 1), False), (5000, 18, (3, 3, 3), (1, 1, 1), False), (5000, 18, (2, 2, 2), (2, 2, 2), True),
    (3000, 40, (2, 2, 2), (2, 2, 2), False), (40000, 39, (3, 3, 3), (1, 1, 1), False)])
def test_kernel_gradient(n, extent, ks, stride, transposed, c_in, c_out):
    km = gpu_map(synth.random_cloud(seed=n, n=n, extent=extent), ks, stride)
    n_in, n_out = (km.n_out, km.n_in) if transposed else (km.n_in, km.n_out)
    x = torch.as_tensor(synth.features(1, n_in, c_in), device=DEV)
    g = torch.as_tensor(synth.features(2, n_out, c_out), device=DEV)
    got = backend.conv_wgrad(x, g, km, transposed).double()
    want = reference(x, g, km, transposed)
    # a product is rounded and added: T such additions in a row are off by at most 2^-24 sqrt(T) of their 2-norm.  128 pairs, two
    # roundings each, then at most 256 tiles a run and as many runs an offset
    tol = 2 ** -24 * np.sqrt(2 * 128 + 256 + 256)
    assert ((got - want).norm() / want.norm()).item() <= tol
    empty = want.abs().sum(dim=(1, 2)) == 0
    assert bool((got[empty] == 0).all())


@pytest.mark.parametrize("n,extent", [(9000, 45), (10500, 48), (12600, 51), (16000, 54), (19000, 57), (21500, 59)])
@pytest.mark.parametrize("c_in,c_out", [(4, 16), (32, 32), (32, 36), (64, 64)])
def test_one_block_of_either_number_of_workgroups(n, extent, c_in, c_out):
    """240 to 600 tiles in a single block of channels: where the number of workgroups changes with the tiles and the widths."""
    km = gpu_map(synth.random_cloud(seed=n, n=n, extent=extent), (3, 3, 3))
    x = torch.as_tensor(synth.features(1, km.n_in, c_in), device=DEV)
    g = torch.as_tensor(synth.features(2, km.n_out, c_out), device=DEV)
    want = reference(x, g, km, False)
    # (as above; a run is at most three tiles, and an offset's runs no more than its tiles)
    tol = 2 ** -24 * np.sqrt(2 * 128 + 3 + 256)
    assert ((backend.conv_wgrad(x, g, km).double() - want).norm() / want.norm()).item() <= tol


def test_infinite_and_nan_rows_reach_their_own_sums_only():
    km = gpu_map(synth.random_cloud(seed=3, n=700, extent=12), (3, 3, 3))
    x = torch.as_tensor(synth.features(1, km.n_in, 96), device=DEV)
    g = torch.as_tensor(synth.features(2, km.n_out, 64), device=DEV)
    x[5, 7], g[500, 3] = float("inf"), float("nan")
    got, want = backend.conv_wgrad(x, g, km).double(), reference(x, g, km, False)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))


def test_dense_layer():
    x = torch.as_tensor(synth.features(1, 3001, 96), device=DEV)
    g = torch.as_tensor(synth.features(2, 3001, 128), device=DEV)
    want = x.double().t() @ g.double()
    assert ((backend.dense_wgrad(x, g).double() - want).norm() / want.norm()).item() <= 2 ** -24 * np.sqrt(2 * 128 + 512)
