"""Block output-stationary kernel (``pce_conv_fwd_osb``) and its row order: tile and window edges, every column-block
width, channel tails, items cut into parts and whole ones, submanifold, strided and transposed tables."""
import numpy as np
import pytest
import torch

from pcengine_amd import _lib, backend, synth
from pcengine_amd.backend import DATAFLOW_OS
from tests.util import DEV, gpu_map

pytestmark = pytest.mark.gpu

# fp32 sums of exact products, one rounding to fp16: half a unit in the last place, 2^-11 relative at most and 2^-11 / sqrt(3) in
# the mean over mantissas; the fp32 sums of up to 27 * 512 terms add less than 2^-24 * sqrt(13824) = 7e-6
REL_L2 = 3.0e-4


def reference(f, w, km, transposed, bias=None, res=None, act=None):
    f, w = f.double(), w.double()
    n_out = km.n_in if transposed else km.n_out
    y = f @ w[13] if km.subm else torch.zeros((n_out, w.shape[2]), dtype=torch.float64, device=f.device)
    kpos = km.kpos.cpu().tolist()
    for k in range(km.kv):
        i, o = km.imap[kpos[k]:kpos[k + 1]].long(), km.omap[kpos[k]:kpos[k + 1]].long()
        if len(i):
            i, o = (o, i) if transposed else (i, o)
            y.index_add_(0, o, f[i] @ w[k])
    for extra in (bias, res):
        y = y if extra is None else y + extra.double()
    return torch.relu(y) if act == "relu" else y


def run(km, c_in, c_out, transposed=False, epilogue=True, wide=False):
    n_in, n_out = (km.n_out, km.n_in) if transposed else (km.n_in, km.n_out)
    assert backend.osb_takes(km.kv, c_in, c_out, torch.float16)
    f = torch.as_tensor(synth.features(1, n_in, c_in), device=DEV).half()
    w = torch.as_tensor(synth.weights(2, km.kv, c_in, c_out), device=DEV).half()
    kw = dict(bias=torch.as_tensor(synth.features(3, 1, c_out)[0], device=DEV).half(),
              residual=torch.as_tensor(synth.features(4, n_out, c_out), device=DEV).half(), act="relu") if epilogue else {}
    x, out = f, None
    if wide:      # column slices of wider matrices, whose other columns survive
        both = torch.full((n_in, c_in + 24), 7.0, dtype=torch.float16, device=DEV)
        x = both[:, 16:16 + c_in]
        x.copy_(f)
        whole = torch.full((n_out, c_out + 40), -3.0, dtype=torch.float16, device=DEV)
        out = whole[:, 8:8 + c_out]
    got = backend.conv_forward(x, w, km, DATAFLOW_OS, transposed=transposed, out=out, **kw)
    want = reference(f, w, km, transposed, kw.get("bias"), kw.get("residual"), kw.get("act"))
    err = ((got.double() - want).norm() / want.norm()).item()
    assert err <= REL_L2, (km.n_out, c_in, c_out, transposed, err)
    if wide:
        assert bool((whole[:, :8] == -3.0).all()) and bool((whole[:, 8 + c_out:] == -3.0).all())
    assert (transposed in km._blocks)


@pytest.mark.parametrize("c_in,c_out", [(64, 72), (96, 96), (64, 128), (160, 136), (128, 192), (192, 256), (64, 264), (256, 512), (96, 1024)])
def test_widths(c_in, c_out):
    km = gpu_map(synth.random_cloud(seed=3, n=1500, extent=14), (3, 3, 3))
    run(km, c_in, c_out)
    run(km, c_in, c_out, epilogue=False, wide=True)


@pytest.mark.parametrize("n", [1, 2, 15, 17, 127, 128, 129, 1000, 8191, 8192, 8193, 20000])
def test_rows_around_blocks_tiles_and_windows(n):
    rng = np.random.default_rng(n)
    cells = rng.permutation(40 ** 3)[:n]      # exactly n voxels
    coords = np.stack([0 * cells, cells // 1600, cells // 40 % 40, cells % 40], axis=1)
    coords = coords[np.argsort(cells)].astype(np.int32)
    km = gpu_map(coords, (3, 3, 3), batchsize=1)
    assert km.n_in == n
    run(km, 128, 128)


@pytest.mark.parametrize("n,extent", [(3000, 200), (60000, 400), (30000, 34), (72000, 60), (140000, 75)])
def test_sparse_and_dense_clouds(n, extent):
    """Fewer items than workgroups, a last round that is cut, several rounds; tiles without any offset but the centre."""
    km = gpu_map(synth.random_cloud(seed=5, n=n, extent=extent, batches=2), (3, 3, 3), batchsize=2)
    run(km, 64, 96)
    run(km, 256, 256)


@pytest.mark.parametrize("cloud", ["surface", "random"])
def test_strided_and_transposed_tables(cloud):
    coords = synth.sphere_plane_cloud() if cloud == "surface" else synth.random_cloud(seed=6, n=9000, extent=26)
    km = gpu_map(coords, (2, 2, 2), (2, 2, 2), want_nbr_in=True)
    run(km, 64, 128)
    run(km, 128, 96, transposed=True)
    run(gpu_map(coords, (3, 3, 3), (2, 2, 2), (1, 1, 1), want_nbr_in=True), 96, 128)


@pytest.mark.parametrize("n,extent", [(5, 3), (4000, 60), (30000, 40)])
def test_order_is_a_permutation_with_the_blocks_patterns(n, extent):
    km = gpu_map(synth.random_cloud(seed=8, n=n, extent=extent), (3, 3, 3), batchsize=1)
    n = km.n_out
    table = (km.nbr_out.view(27, n) >= 0).cpu().numpy()
    pattern = (table.astype(np.int64) << np.arange(27)[:, None]).sum(0)
    known = backend.block_order(km).cpu().numpy()
    assert km.order is not None           # the patterns came with the map; without them they are read from the table
    km.order = None
    km.__dict__.pop("_blocks")
    read = backend.block_order(km).cpu().numpy()
    at = (n + 63) // 64 * 64
    for order in (known, read):
        perm, blocks = order[:n], order[at:at + (n + 15) // 16].astype(np.int64)
        assert np.array_equal(np.sort(perm), np.arange(n))
        assert np.array_equal(perm // 8192, np.arange(n) // 8192)          # rows stay in their window
        padded = np.concatenate([pattern[perm], np.zeros(-n % 16, np.int64)])
        assert np.array_equal(np.bitwise_or.reduce(padded.reshape(-1, 16), axis=1), blocks)
    assert np.array_equal(known, read)


def test_entry_point_refuses_what_it_does_not_take():
    lib = _lib.load()
    for dtype, ci, co, kv in ((_lib.PCE_F32, 64, 96, 27), (_lib.PCE_F16, 48, 96, 27), (_lib.PCE_F16, 80, 96, 27),
                              (_lib.PCE_F16, 64, 64, 27), (_lib.PCE_F16, 64, 100, 27), (_lib.PCE_F16, 64, 96, 125), (_lib.PCE_F16, 64, 96, 1)):
        assert lib.pce_conv_osb_takes(dtype, ci, co, kv) == 0
        rc = lib.pce_conv_fwd_osb(16, 16, 16, dtype, 10, 10, 0, ci, co, kv, 16, 16, 16, 1 << 40, None, None)
        assert rc == _lib.PCE_EINVAL
    assert lib.pce_conv_fwd_osb(16, 16, 16, _lib.PCE_F16, 10, 10, 0, 64, 96, 27, 16, 16, 16, 64, None, None) == _lib.PCE_EWORKSPACE
    assert lib.pce_osb_order(16, None, -1, 27, 100, 16, 50, None) == _lib.PCE_EWORKSPACE
