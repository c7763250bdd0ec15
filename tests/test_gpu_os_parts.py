"""Output-stationary fp32 layers of few rows: offsets shared out over workgroups, column slabs of 32, 64 and 128."""
import numpy as np
import pytest
import torch

from pcengine_amd import _lib, backend, synth
from pcengine_amd.backend import DATAFLOW_FDS, DATAFLOW_OS
from tests.test_gpu_blocks import reference
from tests.util import DEV, gpu_map

pytestmark = pytest.mark.gpu

# fp32 sums of up to 27 * 512 rounded products: 2^-24 * sqrt(13824) = 7e-6
REL_L2 = 7e-6


def run(km, c_in, c_out, transposed=False, split=None, wide=False, buffer=None, dataflow=DATAFLOW_OS):
    n_in, n_out = (km.n_out, km.n_in) if transposed else (km.n_in, km.n_out)
    need = _lib.load().pce_conv_os_workspace_bytes(_lib.PCE_F32, n_out, c_in, c_out, km.kv)
    if split is not None:
        assert (need > 0) == split, (n_out, c_in, c_out, need)
    f = torch.as_tensor(synth.features(1, n_in, c_in), device=DEV).float()
    w = torch.as_tensor(synth.weights(2, km.kv, c_in, c_out), device=DEV).float()
    bias = torch.as_tensor(synth.features(3, 1, c_out)[0], device=DEV).float()
    res = torch.as_tensor(synth.features(4, n_out, c_out), device=DEV).float()
    x, out = f, None
    if wide:
        both = torch.full((n_in, c_in + 24), 7.0, device=DEV)
        x = both[:, 16:16 + c_in]
        x.copy_(f)
        whole = torch.full((n_out, c_out + 40), -3.0, device=DEV)
        out = whole[:, 8:8 + c_out]
    for kw in (dict(), dict(bias=bias), dict(bias=bias, residual=res, act="relu")):
        got = backend.conv_forward(x, w, km, dataflow, transposed=transposed, out=out, buffer=buffer, **kw)
        want = reference(f, w, km, transposed, kw.get("bias"), kw.get("residual"), kw.get("act"))
        err = ((got.double() - want).norm() / want.norm()).item()
        assert err <= REL_L2, (n_out, c_in, c_out, transposed, err)
    if wide:
        assert bool((whole[:, :8] == -3.0).all()) and bool((whole[:, 8 + c_out:] == -3.0).all())


@pytest.mark.parametrize("n", [1, 2, 127, 128, 129, 1000, 9000, 20000, 34000])
def test_rows(n):
    rng = np.random.default_rng(n)
    cells = rng.permutation(40 ** 3)[:n]
    coords = np.stack([0 * cells, cells // 1600, cells // 40 % 40, cells % 40], axis=1)
    km = gpu_map(coords[np.argsort(cells)].astype(np.int32), (3, 3, 3), batchsize=1)
    run(km, 128, 96)
    run(km, 64, 256)
    run(km, 64, 256, dataflow=DATAFLOW_FDS)     # pair tiles and centre product take the same slabs


@pytest.mark.parametrize("c_in,c_out,split", [(16, 16, False), (32, 32, True), (40, 36, True), (29, 35, True), (64, 20, True), (96, 7, True),
                                              (128, 264, True), (512, 512, True)])
def test_widths(c_in, c_out, split):
    km = gpu_map(synth.random_cloud(seed=3, n=1500, extent=14), (3, 3, 3))
    run(km, c_in, c_out, split=split)
    if c_in % 8 == 0 and c_out % 8 == 0:
        run(km, c_in, c_out, wide=True)
        run(km, c_in, c_out, buffer=torch.empty(8 << 20, device=DEV))


def test_strided_and_transposed_tables():
    coords = synth.sphere_plane_cloud()
    km = gpu_map(coords, (2, 2, 2), (2, 2, 2), want_nbr_in=True)
    run(km, 128, 96)
    run(km, 96, 128, transposed=True)
    run(gpu_map(coords, (3, 3, 3), (2, 2, 2), (1, 1, 1), want_nbr_in=True), 64, 64, transposed=True)


def test_non_finite_rows_reach_their_neighbours():
    km = gpu_map(synth.random_cloud(seed=3, n=1500, extent=14), (3, 3, 3))
    f = torch.randn((km.n_in, 64), device=DEV)
    f[5], f[900] = float("inf"), float("nan")
    w = torch.rand((27, 64, 32), device=DEV) + 0.1
    want = reference(f, w, km, False)
    got = backend.conv_forward(f, w, km, DATAFLOW_OS)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())


def test_entry_point_checks_its_workspace():
    lib = _lib.load()
    assert lib.pce_conv_os_workspace_bytes(_lib.PCE_F16, 100, 256, 256, 27) == 0
    assert lib.pce_conv_os_workspace_bytes(_lib.PCE_F32, 0, 256, 256, 27) == 0
    need = lib.pce_conv_os_workspace_bytes(_lib.PCE_F32, 100, 256, 256, 27)
    assert need == 27 * 100 * 256 * 4
    for ws, size in ((None, need), (8, need), (16, need - 1)):
        assert lib.pce_conv_fwd_os_parts(16, 16, 16, _lib.PCE_F32, 100, 100, 256, 256, 27, 16, ws, size, None, None) == _lib.PCE_EINVAL


@pytest.mark.parametrize("side,c_in,c_out,groups", [(12, 64, 128, 9), (16, 32, 64, 8), (16, 64, 64, 8), (16, 96, 96, 5), (16, 256, 96, 5), (20, 32, 32, 8),
                                                    (20, 40, 72, 2), (23, 64, 64, 2), (18, 64, 64, 5)])
def test_error_of_groups_of_offsets(side, c_in, c_out, groups):
    """However few workgroups the offsets are shared out to, they are added up in as many groups as the workspace holds sums."""
    coords = np.stack([0 * np.arange(side ** 3), *np.unravel_index(np.arange(side ** 3), (side,) * 3)], axis=1).astype(np.int32)
    km = gpu_map(coords, (3, 3, 3), batchsize=1)
    n = km.n_out
    assert _lib.load().pce_conv_os_workspace_bytes(_lib.PCE_F32, n, c_in, c_out, 27) == groups * n * c_out * 4
    gen = torch.Generator(device=DEV).manual_seed(1)
    f = torch.randn((n, c_in), generator=gen, device=DEV)
    w = torch.randn((27, c_in, c_out), generator=gen, device=DEV) * 0.1
    want = reference(f, w, km, False)
    # T additions in a row, each off by up to half a unit of a partial sum whose variance grows evenly: 2^-24 sqrt(T / 6)
    tol = 2.0 ** -24 * ((-(-27 // groups) * c_in + groups) / 6) ** 0.5
    for kw in (dict(), dict(bias=torch.zeros(c_out + 1, device=DEV)[1:])):      # (odd pointers: the shares' sums)
        got = backend.conv_forward(f, w, km, DATAFLOW_OS, **kw)
        assert ((got.double() - want).norm() / want.norm()).item() <= tol
