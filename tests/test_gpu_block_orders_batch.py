"""Block orders of several tables in one call: the same arrays as one by one, whatever stands beside them."""
import numpy as np
import pytest
import torch

import pcengine_amd as pe
from pcengine_amd import _lib, backend, nets, synth
from tests.util import DEV, dev_coords, gpu_map

pytestmark = pytest.mark.gpu


def _problems(tables):
    lib, probs, orders = _lib.load(), (_lib.OsbOrderProblem * len(tables))(), []
    for p, (nbr, mask, mid) in zip(probs, tables):
        kv, n = nbr.shape
        p.order_elems = lib.pce_osb_order_elems(n)
        orders.append(torch.full((p.order_elems,), -7, dtype=torch.int32, device=DEV))
        p.nbr, p.mask, p.mid, p.kv, p.n_rows, p.order = nbr.data_ptr(), None if mask is None else mask.data_ptr(), mid, kv, n, orders[-1].data_ptr()
    return probs, orders


@pytest.mark.parametrize("rows", [(1, 2), (700, 63, 7168), (8192, 5), (8191, 8193, 100, 16384, 16385, 1, 20011, 129)])
def test_same_as_one_by_one(rows):
    rng = np.random.default_rng(len(rows))
    tables = []
    for i, n in enumerate(rows):
        kv, mid = ((27, 13), (8, -1), (27, -1))[i % 3]
        nbr = np.where(rng.random((kv, n)) < 0.3, 0, -1).astype(np.int32)
        mask = ((nbr >= 0).astype(np.int64) << np.arange(kv)[:, None]).sum(0).astype(np.int32) if i % 2 else None
        tables.append((torch.as_tensor(nbr, device=DEV), None if mask is None else torch.as_tensor(mask, device=DEV), mid))
    lib, s = _lib.load(), torch.cuda.current_stream().cuda_stream
    probs, got = _problems(tables)
    _lib.check(lib.pce_osb_order_batch(probs, len(rows), s))
    probs, want = _problems(tables)
    for p in probs:
        _lib.check(lib.pce_osb_order(p.nbr, p.mask, p.mid, p.kv, p.n_rows, p.order, p.order_elems, s))
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_refused():
    nbr = torch.zeros((27, 50), dtype=torch.int32, device=DEV)
    probs, orders = _problems([(nbr, None, 13)] * 2)
    lib, s = _lib.load(), torch.cuda.current_stream().cuda_stream
    for count in (0, -1, _lib.OSB_ORDER_MAX + 1):
        assert lib.pce_osb_order_batch(probs, count, s) == _lib.PCE_EINVAL
    probs[1].order_elems -= 1
    assert lib.pce_osb_order_batch(probs, 2, s) == _lib.PCE_EWORKSPACE
    torch.cuda.synchronize()
    assert bool((orders[0] == -7).all())        # nothing ran


def test_kept_as_if_built_alone():
    maps = [gpu_map(synth.random_cloud(seed=s, n=n, extent=24), (3, 3, 3), batchsize=1) for s, n in ((1, 9000), (2, 700))]
    alone = [backend.block_order(m).clone() for m in maps]
    for m in maps:
        m.__dict__.pop("_blocks")
    backend.block_orders([(m, False) for m in maps] + [(maps[0], True)])     # (no input-major table: not built)
    for m, order in zip(maps, alone):
        assert list(m._blocks) == [False] and m._blocks[False][1] == torch.cuda.current_stream().cuda_stream
        assert torch.equal(backend.block_order(m), order)


@pytest.mark.parametrize("planned", [False, True])
def test_network_builds_its_orders_ahead(planned, monkeypatch):
    """Every order a forward uses is there before its first layer, and the logits do not change."""
    torch.manual_seed(3)
    model = nets.SparseResUNet(4, 20).to(DEV).eval().fuse_bn().half()
    if planned:
        model.use_planner()
    coords = synth.random_cloud(seed=5, n=40000, extent=40)
    f = torch.as_tensor(synth.features(4, len(coords), 4), device=DEV).half()
    make = lambda: pe.spTensor(f, dev_coords(coords), None, [0, 0, 0], coords[:, 1:].max(0).tolist(), batchsize=1)
    single = []
    real = backend._build_kept
    monkeypatch.setattr(backend, "_build_kept", lambda km, kept, what, *a: (single.append(what), real(km, kept, what, *a))[1])
    with torch.no_grad():
        x = make()
        got = model(x).feats.clone()
        assert "blocks" not in single and any(km.__dict__.get("_blocks") for km in x.kmaps.values())
        monkeypatch.setattr(nets.SparseResUNet, "_prebuild_block_orders", lambda self, x: None)
        want = model(make()).feats
        assert "blocks" in single and torch.equal(got, want)


@pytest.mark.parametrize("change", ["dataflows", "a stage", "a width"])
def test_orders_follow_the_modules(change):
    """Layers that are set to another dataflow, or replaced, after a forward: no order is built that none of them reads, and those
    that they read are there ahead of them."""
    torch.manual_seed(3)
    model = nets.SparseResUNet(4, 20).to(DEV).eval().half()
    coords = synth.random_cloud(seed=5, n=40000, extent=40)
    f = torch.as_tensor(synth.features(4, len(coords), 4), device=DEV).half()
    make = lambda: pe.spTensor(f, dev_coords(coords), None, [0, 0, 0], coords[:, 1:].max(0).tolist(), batchsize=1)

    def orders():
        x = make()
        with torch.no_grad():
            model(x)
        return {key for key, km in x.kmaps.items() if km.__dict__.get("_blocks")}

    first = orders()
    deep = [key for key in first if key[1] == max(k[1] for k in first)]
    assert len(first) > 1 and len(deep) >= 1
    if change == "dataflows":
        for m in model.modules():
            if isinstance(m, pe.conv3d):
                m.dataflow = "fds"
        assert orders() == set()
        for m in model.modules():
            if isinstance(m, pe.conv3d):
                m.dataflow = "auto"
        assert orders() == first
    elif change == "a stage":
        model.enc[-1] = torch.nn.Sequential(nets.ResidualBlock(128, 256, "fds"), nets.ResidualBlock(256, 256, "fds")).to(DEV).eval().half()
        assert orders() == first - set(deep)
    else:
        model.dec[-1][1].b.conv = pe.conv3d(96, 96, 3).to(DEV).half()
        assert orders() == first
