"""Kernel gradient of wide fp16 layers (128 x 128 blocks through LDS rings): tile, run and channel edges, against float64."""
import numpy as np
import pytest
import torch

from pcengine_amd import backend, synth
from tests.util import DEV, gpu_map

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c_in,c_out", [(72, 8), (8, 72), (128, 128), (136, 200), (264, 72), (256, 384)])
@pytest.mark.parametrize("n,extent,ks,stride,transposed", [
    (1, 2, (3, 3, 3), (1, 1, 1), False), (40, 30, (3, 3, 3), (1, 1, 1), False), (127, 6, (3, 3, 3), (1, 1, 1), False),
    (130, 6, (1, 1, 3), (1, 1, 1), False), (5000, 18, (3, 3, 3), (1, 1, 1), False), (5000, 18, (2, 2, 2), (2, 2, 2), True),
    (3000, 40, (2, 2, 2), (2, 2, 2), False)])
def test_kernel_gradient(n, extent, ks, stride, transposed, c_in, c_out):
    coords = synth.random_cloud(seed=n, n=n, extent=extent)
    km = gpu_map(coords, ks, stride)
    n_in, n_out = (km.n_out, km.n_in) if transposed else (km.n_in, km.n_out)
    x = torch.as_tensor(synth.features(1, n_in, c_in), device=DEV).half()
    g = torch.as_tensor(synth.features(2, n_out, c_out), device=DEV).half()
    got = backend.conv_wgrad(x, g, km, transposed).double()
    want = torch.zeros((km.kv, c_in, c_out), dtype=torch.float64, device=DEV)
    kpos = km.kpos.cpu().tolist()
    for k in range(km.kv):
        i, o = km.imap[kpos[k]:kpos[k + 1]].long(), km.omap[kpos[k]:kpos[k + 1]].long()
        i, o = (o, i) if transposed else (i, o)
        want[k] = x[i].double().t() @ g[o].double()
    if km.subm:
        want[km.kv // 2] += x.double().t() @ g.double()
    # exact products, fp32 sums of at most n terms: 2^-24 sqrt(n) of their 2-norm
    tol = 2 ** -24 * np.sqrt(max(n_in, n_out) + 1)
    assert ((got - want).norm() / want.norm()).item() <= tol
    empty = want.abs().sum(dim=(1, 2)) == 0
    assert bool((got[empty] == 0).all())


@pytest.mark.parametrize("n,extent,c_in,c_out", [(30000, 35, 256, 256), (72000, 59, 256, 256), (72000, 59, 384, 256), (72000, 59, 136, 136)])
def test_long_runs_are_added_up_in_chains(n, extent, c_in, c_out):
    km = gpu_map(synth.random_cloud(seed=7, n=n, extent=extent), (3, 3, 3))
    gen = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn((km.n_in, c_in), generator=gen, device=DEV).half()
    g = torch.randn((km.n_out, c_out), generator=gen, device=DEV).half()
    got = backend.conv_wgrad(x, g, km).double()
    kpos = km.kpos.cpu().tolist()
    want = torch.stack([x.double().t() @ g.double() if k == 13 else
                        x[km.imap[kpos[k]:kpos[k + 1]].long()].double().t() @ g[km.omap[kpos[k]:kpos[k + 1]].long()].double() for k in range(27)])
    # T additions in a row, each off by up to half a unit of a partial sum whose variance grows evenly: 2^-24 sqrt(T / 6) of the
    # result.  Chains of 8 tiles of 128 pairs, two roundings for 16 of them; then at most 32 chains a run, 8 runs an offset
    tol = 2 ** -24 * np.sqrt((8 * 128 / 8 + 32 + 8) / 6)
    assert ((got - want).norm() / want.norm()).item() <= tol
