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
