"""The counting sort of the row order where a workgroup takes more than 256 rows: its edges, its longest workgroups, rows with
records of all neighbours and without."""
import numpy as np
import pytest
import torch

from pcengine_amd import _lib, backend, synth
from tests.util import DEV, dev_coords

pytestmark = pytest.mark.gpu
TAIL = 8192


def _low(m):
    return np.log2((m & -m).astype(np.float64)).astype(np.int64)


def _keys(m):
    """Sort key of rows with neighbours: one by its offset, two by both, three and more by the two lowest (behind those)."""
    rest = m & (m - 1)
    first, second = _low(m), _low(np.where(rest == 0, 1, rest))
    return np.where(rest == 0, first, np.where((rest & (rest - 1)) == 0, 0, 1024) + 32 + first * 32 + second)


def _check(order, nbr, mid, counts):
    """order: the array of the library; nbr: the [kv, n] neighbour table it was made from."""
    kv, n = nbr.shape
    has = nbr >= 0
    if mid >= 0:
        has[mid] = False
    masks = (has.astype(np.int64) << np.arange(kv)[:, None]).sum(axis=0)
    pc = has.sum(axis=0)
    heavy, nonzero, single = int((pc >= 3).sum()), int((pc >= 1).sum()), int((pc == 1).sum())
    assert counts == (heavy, nonzero, single)
    perm = order[:n].astype(np.int64)
    assert np.array_equal(order[n:2 * n].astype(np.int64), masks)
    assert np.array_equal(np.sort(perm), np.arange(n))
    sect = masks[perm]
    assert (sect[:n - nonzero] == 0).all() and (sect[n - nonzero:] != 0).all()
    assert (np.diff(perm[:n - nonzero]) > 0).all()      # rows without neighbours stay in their order
    keys = _keys(sect[n - nonzero:])
    assert (np.diff(keys) >= 0).all()
    rec_at = (2 * n + TAIL + 3) // 4 * 4
    rec = order[rec_at:rec_at + 4 * n].reshape(n, 4)[n - nonzero:].astype(np.int64)
    rows, m = perm[n - nonzero:], sect[n - nonzero:]
    rest = m & (m - 1)
    assert np.array_equal(rec[:, 0], rows) and np.array_equal(rec[:, 1], m)
    assert np.array_equal(rec[:, 2], nbr[_low(m), rows])
    assert np.array_equal(rec[:, 3], np.where(rest == 0, -1, nbr[_low(np.where(rest == 0, 1, rest)), rows]))
    if nonzero - single <= n // 8 + 32:
        at = rec_at + 4 * n
        shared = order[at:at + 32 * (nonzero - single)].reshape(-1, 32)
        rows, m = rows[single:], m[single:]
        assert np.array_equal(shared[:, 0], rows) and np.array_equal(shared[:, 1].astype(np.int64), m)
        for k in range(kv):
            assert np.array_equal(shared[:, 2 + k], np.where((m >> k) & 1, nbr[k, rows], -1))


@pytest.mark.parametrize("n", [1, 255, 65536, 65537, 131073, 196600, 65536 * 17 + 5])
@pytest.mark.parametrize("kv,mid,share", [(27, 13, 0.004), (27, 13, 0.3), (8, -1, 0.5), (8, -1, 0.02)])
def test_order_of_a_table(n, kv, mid, share):
    rng = np.random.default_rng(n + kv)
    nbr = np.where(rng.random((kv, n)) < share, rng.integers(0, n, (kv, n)), -1).astype(np.int32)
    nbr[:, n // 3:n // 2] = -1 if n % 2 else 7       # a run of rows with one pattern
    if mid >= 0:
        nbr[mid] = np.arange(n)
    table = torch.as_tensor(nbr, device=DEV)
    lib = _lib.load()
    order = torch.empty(lib.pce_row_order_elems(n), dtype=torch.int32, device=DEV)
    counts = (_lib.c_int64 * 3)()
    _lib.check(lib.pce_row_order(table.data_ptr(), kv, n, mid, order.data_ptr(), order.numel(), counts, torch.cuda.current_stream().cuda_stream))
    _check(order.cpu().numpy(), nbr, mid, tuple(counts))


def test_order_of_rows_beyond_sixteen_times_the_workgroups():
    """More rows than the places of the counts allow at 16 times 256 rows a workgroup: longer workgroups."""
    kv, n = 8, 256 * 16 * 2040 + 5
    g = torch.Generator(device=DEV).manual_seed(1)
    nbr = torch.where(torch.rand((kv, n), generator=g, device=DEV) < 0.05, 0, -1).int()
    lib = _lib.load()
    order = torch.empty(lib.pce_row_order_elems(n), dtype=torch.int32, device=DEV)
    counts = (_lib.c_int64 * 3)()
    _lib.check(lib.pce_row_order(nbr.data_ptr(), kv, n, -1, order.data_ptr(), order.numel(), counts, torch.cuda.current_stream().cuda_stream))
    masks = torch.zeros(n, dtype=torch.int32, device=DEV)
    pairs = torch.zeros(n, dtype=torch.int32, device=DEV)
    for k in range(kv):
        masks |= (nbr[k] >= 0).int() << k
        pairs += (nbr[k] >= 0).int()
    assert tuple(counts) == (int((pairs >= 3).sum()), int((pairs >= 1).sum()), int((pairs == 1).sum()))
    plain = n - counts[1]
    perm = order[:n].long()
    assert torch.equal(order[n:2 * n], masks) and torch.equal(perm.sort().values, torch.arange(n, device=DEV))
    sect = masks[perm]
    assert bool((sect[:plain] == 0).all()) and bool((sect[plain:] != 0).all()) and bool((perm[:plain].diff() > 0).all())
    assert (np.diff(_keys(sect[plain:].cpu().numpy().astype(np.int64))) >= 0).all()
    at = (2 * n + TAIL + 3) // 4 * 4
    rec = order[at:at + 4 * n].view(n, 4)[plain:]
    assert torch.equal(rec[:, 0], order[plain:n]) and torch.equal(rec[:, 1], sect[plain:]) and bool((rec[:, 2] == 0).all())


@pytest.mark.parametrize("sorted_rows", [True, False])
@pytest.mark.parametrize("cloud", ["lidar", "rooms"])
def test_order_built_with_a_map_of_many_rows(cloud, sorted_rows):
    """A submanifold and a strided map in one batch; unsorted rows take the hash table, whose masks come from the counting pass."""
    c = synth.lidar_cloud(seed=2, azimuths=1100, n_ground=11000, voxel=0.1) if cloud == "lidar" else \
        synth.indoor_batch(scenes=1, n_room=120000, n_box=2500)
    c = c[np.lexsort(c.T[::-1])] if sorted_rows else c[np.random.default_rng(0).permutation(len(c))]
    assert len(c) > 65536
    coords, cmax = dev_coords(c), c[:, 1:].max(0).tolist()
    jobs = [dict(in_coords=coords, ks=(3, 3, 3), stride=(1, 1, 1), pad=(0, 0, 0), cmin=[0, 0, 0], cmax_out=cmax, subm=True, want_csr=True,
                 batchsize=1),
            dict(in_coords=coords, ks=(2, 2, 2), stride=(2, 2, 2), pad=(0, 0, 0), cmin=[0, 0, 0],
                 cmax_out=backend.strided_coords_max(cmax, (2, 2, 2), (2, 2, 2), (0, 0, 0)), subm=False, want_csr=True, want_nbr_in=True,
                 batchsize=1)]
    for km, mid in zip(backend.build_kernel_maps(jobs), (13, -1)):
        nbr = km.nbr_out.cpu().numpy().reshape(km.kv, km.n_out)
        _check(km.order.cpu().numpy(), nbr, mid, (km.order_heavy, km.order_nonzero, km.order_single))
