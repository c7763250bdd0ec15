"""Weights and features that are not finite reach the rows that have such an offset or neighbour and no others (block kernel)."""
import pytest
import torch

from pcengine_amd import backend, synth
from pcengine_amd.backend import DATAFLOW_OS
from tests.test_gpu_blocks import REL_L2, reference
from tests.util import DEV, gpu_map

pytestmark = pytest.mark.gpu


def check(km, w, transposed=False):
    n_in = km.n_out if transposed else km.n_in
    f = torch.as_tensor(synth.features(1, n_in, w.shape[1]), device=DEV).half()
    f[f == 0] = 0.5
    got = backend.conv_forward(f, w, km, DATAFLOW_OS, transposed=transposed)
    assert transposed in km._blocks
    want = reference(f, w, km, transposed)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()] > 0, want[want.isinf()] > 0)
    fine = want.isfinite()
    assert bool(fine.any()) and not bool(fine.all())
    assert ((got.double() - want)[fine].norm() / want[fine].norm()).item() <= REL_L2


@pytest.mark.parametrize("c_in,c_out", [(64, 96), (96, 192), (128, 256), (64, 264)])
@pytest.mark.parametrize("n,extent", [(600, 40), (1500, 14), (20000, 36)])
def test_submanifold_layers(n, extent, c_in, c_out):
    km = gpu_map(synth.random_cloud(seed=3, n=n, extent=extent), (3, 3, 3), batchsize=1)
    w = torch.as_tensor(synth.weights(2, 27, c_in, c_out), device=DEV).half()
    w[4, 5, 7] = float("inf")
    check(km, w.clone())
    w[20, 33, c_out - 1] = float("nan")          # another offset, the last column
    w[4, 6, 7] = float("-inf")                   # a column with both infinities
    w[26, :, 9] = float("inf")
    w[0, 11] = float("-inf")                     # every column
    check(km, w)


def test_strided_and_transposed_layers():
    coords = synth.sphere_plane_cloud()
    km = gpu_map(coords, (2, 2, 2), (2, 2, 2), want_nbr_in=True)
    for transposed in (False, True):
        w = torch.as_tensor(synth.weights(2, 8, 128, 96), device=DEV).half()
        w[3, 5, 7], w[6, 100, 95] = float("inf"), float("nan")
        check(km, w, transposed)


def test_layer_of_many_pairs():
    """Tiles cut into parts, and every weight of an offset infinite."""
    km = gpu_map(synth.random_cloud(seed=3, n=30000, extent=34), (3, 3, 3), batchsize=1)
    assert backend._lib.load().pce_conv_osb_scratch_bytes(km.n_out, km.M, 256, 256, 27) > 0
    w = torch.as_tensor(synth.weights(2, 27, 256, 256), device=DEV).half()
    w[2] = float("inf")
    w[2, 0, 0] = 1.0
    f = torch.ones((km.n_out, 256), dtype=torch.float16, device=DEV)
    got = backend.conv_forward(f, w, km, DATAFLOW_OS)
    has = km.nbr_out.view(27, -1)[2] >= 0
    assert torch.equal(got.isinf().all(dim=1), has) and bool(got[~has].isfinite().all())


@pytest.mark.parametrize("c_in,c_out", [(64, 96), (96, 192), (128, 256)])
def test_features(c_in, c_out):
    km = gpu_map(synth.random_cloud(seed=3, n=1500, extent=14), (3, 3, 3), batchsize=1)
    f = torch.as_tensor(synth.features(1, km.n_in, c_in), device=DEV).half()
    f[5, 3], f[6, c_in - 1], f[900] = float("inf"), float("-inf"), float("nan")
    w = torch.as_tensor(synth.weights(2, 27, c_in, c_out), device=DEV).half()
    w[w == 0] = 0.5
    got, want = backend.conv_forward(f, w, km, DATAFLOW_OS), reference(f, w, km, False)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert bool(want.isinf().any()) and bool(want.isfinite().any())
