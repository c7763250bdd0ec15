"""The maps of a cloud built in one library call (``backend.build_pyramid``) against the general path, map by map: the same arrays,
the same cache entries, the same refusals."""
import numpy as np
import pytest
import torch

import pcengine_amd as pe
from pcengine_amd import _lib, backend, spconv, synth
from tests.util import DEV, dev_coords

pytestmark = pytest.mark.gpu

UNET = [(3, 1, 0)] + [(2, 2, 0), (3, 1, 0)] * 4
LISTS = {"unet": UNET, "lean": [(3, 1, 0, True), (2, 2, 0), (3, 1, 0, True), (3, 1, 0)], "one": [(3, 1, 0)], "down": [(2, 2, 0)],
         "threes": [(3, 3, 0), (3, 1, 0), (2, 2, 0)], "padded": [(3, 1, 0), (3, 2, 1), (3, 1, 0)]}
CLOUDS = {"lidar": lambda: synth.lidar_cloud(seed=2, azimuths=700, n_ground=7000, voxel=0.1),
          "rooms": lambda: synth.indoor_batch(scenes=2, n_room=6000, n_box=125),
          "tiny": lambda: synth.random_cloud(seed=1, n=200, extent=24)}


def tensor(c):
    c = c[np.lexsort(c.T[::-1])] if len(c) else c
    return pe.spTensor(torch.zeros((len(c), 1), device=DEV), dev_coords(c), None, [0, 0, 0], c[:, 1:].max(0).tolist(),
                       batchsize=int(c[:, 0].max()) + 1)


def general(monkeypatch):
    def never(*a):
        raise backend.PlanNotApplicable()
    monkeypatch.setattr(backend, "build_pyramid", never)


@pytest.mark.parametrize("cloud", sorted(CLOUDS))
@pytest.mark.parametrize("layers", sorted(LISTS))
def test_same_maps(cloud, layers, monkeypatch):
    c = CLOUDS[cloud]()
    a, b = tensor(c), tensor(c)
    spconv.prebuild_maps(a, LISTS[layers])
    assert any(km.__dict__.get("_arena") is not None for km in a.kmaps.values()) == (layers != "padded")
    general(monkeypatch)
    spconv.prebuild_maps(b, LISTS[layers])
    assert list(a.kmaps) == list(b.kmaps) and set(a.cbook) == set(b.cbook)
    for s in a.cbook:
        assert torch.equal(a.cbook[s], b.cbook[s])
    for key in a.kmaps:
        p, q = a.kmaps[key], b.kmaps[key]
        for name in ("ks", "stride", "pad", "subm", "n_in", "n_out", "kv", "M", "qsum", "order_heavy", "order_nonzero", "order_single", "tag",
                     "has_pairs", "batchsize", "_cmin", "_cmax"):
            assert getattr(p, name) == getattr(q, name), name
        assert list(p.knnz_host) == list(q.knnz_host) and list(p.kpos_host) == list(q.kpos_host) and list(p.qkpos_host) == list(q.qkpos_host)
        assert (p.order is None) == (q.order is None)
        for name in ("knnz", "kpos", "qkpos", "out_coords", "nbr_out", "nbr_in", "icsr", "ocsr", "icode", "ocode", "islot", "oslot", "imap", "omap"):
            x, y = getattr(p, name), getattr(q, name)
            assert (x is None) == (y is None), name
            assert x is None or torch.equal(x.reshape(-1), y.reshape(-1)), name
        assert [torch.equal(u, v) for u, v in zip(p._as_list()[:4], q._as_list()[:4])] == [True] * 4
        assert all(torch.is_tensor(p[i]) and torch.equal(p[i], q[i]) for i in range(4)) and p[4] == q[4] and p[5] == q[5] and p[-1] == q[-1]
        if p.order is not None:
            n = p.n_out
            assert torch.equal(p.order[n:2 * n], q.order[n:2 * n])                     # patterns
            assert torch.equal(p.order[:n].sort().values, q.order[:n].sort().values)   # (rows of one pattern lie as they came)


@pytest.mark.parametrize("kind", ["unsorted", "far", "outside the box"])
def test_what_it_does_not_take(kind, monkeypatch):
    c = CLOUDS["lidar"]()
    x = tensor(c)
    if kind == "unsorted":
        x.coords = x.coords[torch.randperm(len(c), device=DEV)].contiguous()
    elif kind == "far":
        x.coords[-1, 1] = 40000
    else:
        x.coords_max = [v // 2 for v in x.coords_max]
    def outcome():
        y = pe.spTensor(x.feats, x.coords.clone(), None, [0, 0, 0], list(x.coords_max), batchsize=1)
        try:
            spconv.prebuild_maps(y, UNET)
        except Exception as e:
            return type(e), str(e)
        return [(k, m.M, m.imap.clone(), m.omap.clone()) for k, m in y.kmaps.items()]
    got = outcome()
    general(monkeypatch)
    want = outcome()
    assert type(got) is type(want)
    if isinstance(got, tuple):
        assert got == want
    else:
        for (k, m, i, o), (k2, m2, i2, o2) in zip(got, want):
            assert k == k2 and m == m2 and torch.equal(i, i2) and torch.equal(o, o2)


def counted(monkeypatch):
    """Calls of the chained output coordinates and the maps that were built one by one, from here on."""
    chains, singles = [], []
    chain, build = backend.build_out_coords_chain, backend.build_kernel_maps
    monkeypatch.setattr(backend, "build_out_coords_chain", lambda *a: (chains.append(1), chain(*a))[1])
    monkeypatch.setattr(backend, "build_kernel_maps", lambda jobs, *a, **k: (singles.extend(jobs), build(jobs, *a, **k))[1])
    return chains, singles


def test_a_kernel_too_large_for_a_plan_costs_no_second_chain(monkeypatch):
    x = tensor(CLOUDS["lidar"]())
    chains, singles = counted(monkeypatch)
    spconv.prebuild_maps(x, [(5, 1, 0), (2, 2, 0), (3, 1, 0), (2, 2, 0), (3, 1, 0)])
    assert len(chains) == 1 and len(singles) == 5 == len(x.kmaps)


@pytest.mark.parametrize("call", ["pce_outcoords_chain", "pce_pyramid_plan_levels", "pce_pyramid_maps"])
@pytest.mark.parametrize("status", [_lib.PCE_EHIP, _lib.PCE_EWORKSPACE])
def test_a_failed_launch_is_an_error(call, status, monkeypatch):
    """What is not the cloud's fault is raised and nothing is built again (the status is made up on the host, no launch fails)."""
    x = tensor(CLOUDS["lidar"]())
    chains, singles = counted(monkeypatch)
    monkeypatch.setattr(_lib.load(), call, lambda *a: status)
    with pytest.raises(_lib.PCEError, match=f"pce status {status}"):
        spconv.prebuild_maps(x, UNET)
    assert len(chains) == 1 and not singles and not x.kmaps


@pytest.mark.parametrize("call", ["pce_outcoords_chain", "pce_pyramid_plan_levels", "pce_pyramid_maps"])
@pytest.mark.parametrize("status", [_lib.PCE_ECOORD, _lib.PCE_ECAPACITY])
def test_a_refused_cloud_is_built_map_by_map(call, status, monkeypatch):
    x = tensor(CLOUDS["lidar"]())
    real, done = getattr(_lib.load(), call), []
    monkeypatch.setattr(_lib.load(), call, lambda *a: (done.append(1), status if len(done) == 1 else real(*a))[1])
    spconv.prebuild_maps(x, UNET)
    assert len(x.kmaps) == 9 and not any(km.__dict__.get("_arena") is not None for km in x.kmaps.values())


@pytest.mark.parametrize("kind", ["too empty", "refused maps"])
def test_the_chain_of_a_declined_cloud_is_not_asked_again(kind, monkeypatch):
    """The general path goes on from the levels' coordinates, or from the answer that the chain does not take the cloud."""
    c = CLOUDS["lidar"]() if kind == "refused maps" else synth.lidar_cloud(seed=2, azimuths=40, n_ground=400, voxel=0.1)
    a, b = tensor(c), tensor(c)
    with monkeypatch.context() as m:
        chains, singles = counted(m)
        if kind == "refused maps":
            m.setattr(_lib.load(), "pce_pyramid_maps", lambda *args: _lib.PCE_ECAPACITY)
        spconv.prebuild_maps(a, UNET)
        assert len(chains) == 1 and len(singles) == 9
    general(monkeypatch)
    spconv.prebuild_maps(b, UNET)
    assert list(a.kmaps) == list(b.kmaps)
    for key in a.kmaps:
        p, q = a.kmaps[key], b.kmaps[key]
        assert p.M == q.M and torch.equal(p.out_coords, q.out_coords) and torch.equal(p.imap, q.imap) and torch.equal(p.omap, q.omap)


@pytest.mark.parametrize("kind", ["unsorted", "outside the box"])
@pytest.mark.parametrize("layers", ["unet", "lean", "one", "down", "threes"])
def test_rows_that_the_column_grid_refuses(kind, layers, monkeypatch):
    """They go through the hash table, and nothing that has been built is built again on the general path."""
    c = CLOUDS["lidar"]()
    cmax = c[:, 1:].max(0).tolist()
    if kind == "unsorted":
        c = c[np.random.default_rng(0).permutation(len(c))]
    else:
        cmax[0] //= 2
    make = lambda: pe.spTensor(torch.zeros((len(c), 1), device=DEV), dev_coords(c), None, [0, 0, 0], list(cmax), batchsize=1)
    a, b = make(), make()
    with monkeypatch.context() as m:
        chains, singles = counted(m)
        spconv.prebuild_maps(a, LISTS[layers])
        assert len(chains) <= 1 and not singles
    general(monkeypatch)
    spconv.prebuild_maps(b, LISTS[layers])
    assert list(a.kmaps) == list(b.kmaps) and set(a.cbook) == set(b.cbook)
    for s in a.cbook:
        assert torch.equal(a.cbook[s], b.cbook[s])
    for key in a.kmaps:
        p, q = a.kmaps[key], b.kmaps[key]
        for name in ("n_in", "n_out", "kv", "M", "qsum", "order_heavy", "order_nonzero", "order_single", "tag", "has_pairs", "batchsize", "_cmin", "_cmax"):
            assert getattr(p, name) == getattr(q, name), name
        assert list(p.kpos_host) == list(q.kpos_host) and list(p.qkpos_host) == list(q.qkpos_host)
        for name in ("knnz", "kpos", "qkpos", "out_coords", "nbr_out", "nbr_in", "icsr", "ocsr", "icode", "ocode", "islot", "oslot"):
            x, y = getattr(p, name), getattr(q, name)
            assert (x is None) == (y is None), name
            assert x is None or torch.equal(x.reshape(-1), y.reshape(-1)), name
        if p.has_pairs:
            assert torch.equal(p.imap, q.imap) and torch.equal(p.omap, q.omap)
        if p.order is not None:
            n = p.n_out
            assert torch.equal(p.order[n:2 * n], q.order[n:2 * n])
            assert torch.equal(p.order[:n].sort().values, q.order[:n].sort().values)
        spans = [(t.untyped_storage().data_ptr(), t.untyped_storage().nbytes()) for t in p.device_tensors()]
        for name in ("nbr_out", "out_coords", "kpos"):
            at = getattr(p, name).data_ptr()
            assert any(lo <= at < lo + size for lo, size in spans), name


def test_memory_of_maps_built_on_another_stream_is_told():
    x = tensor(CLOUDS["lidar"]())
    spconv.prebuild_maps(x, UNET)
    for km in x.kmaps.values():
        spans = [(t.untyped_storage().data_ptr(), t.untyped_storage().nbytes()) for t in km.device_tensors()]
        for name in ("imap", "nbr_out", "order", "out_coords", "kpos"):
            at = getattr(km, name).data_ptr()
            assert any(lo <= at < lo + n for lo, n in spans), name


def test_arrays_are_cut_natively():
    """The arrays of a map are parts of its allocation; what the extension does not take is sliced."""
    whole = torch.arange(1000, dtype=torch.int32, device=DEV)
    for array, first, count in ((whole, 0, 1000), (whole, 0, 0), (whole, 1000, 0), (whole, 3, 17), (whole[100:], 5, 895), (whole, 999, 1)):
        part = _lib.host().cut(array, first, count)
        want = array[first:first + count]
        assert torch.equal(part, want) and part.shape == want.shape and part.stride() == want.stride() and part.data_ptr() == want.data_ptr()
        assert part.untyped_storage().data_ptr() == whole.untyped_storage().data_ptr() and not part.requires_grad
    for array, first, count in ((whole, 1, 1000), (whole, 1001, 0), (whole[::2], 0, 5), (whole.view(10, 100), 0, 5), (whole.long(), 0, 5), (whole.cpu(), 0, 5)):
        assert _lib.host().cut(array, first, count) is None
        assert torch.equal(backend._cut(array, first, count), array[first:first + count])
    for array, first, count in ((whole, -3, 2), (whole, 3, -1), (whole, 2 ** 62, 2 ** 62)):
        assert _lib.host().cut(array, first, count) is None
    with pytest.raises(TypeError):
        _lib.host().cut(whole, 1)
    with pytest.raises(OverflowError):
        _lib.host().cut(whole, 2 ** 70, 1)
    with torch.inference_mode():
        other = torch.arange(10, dtype=torch.int32, device=DEV)
        assert torch.equal(backend._cut(other, 2, 3), other[2:5])
    x = tensor(CLOUDS["lidar"]())
    spconv.prebuild_maps(x, UNET)
    for km in x.kmaps.values():
        assert km.imap.numel() == km.omap.numel() == km.M and km.imap is km.imap and km.nbr_out.numel() == km.kv * km.n_out
