"""Arrays that layers build on first use and keep on their map (the block order): they live as long as the map, other
streams wait for them, and a capture leaves nothing behind that has not run."""
import pytest
import torch

import pcengine_amd as pe
from pcengine_amd import backend, nets, synth
from pcengine_amd.backend import DATAFLOW_OS
from pcengine_amd.spconv import MapPlanner, prebuild_maps
from tests.util import DEV, dev_coords, gpu_map

pytestmark = pytest.mark.gpu


def _tensor(coords, c=4):
    f = torch.as_tensor(synth.features(4, len(coords), c), device=DEV).half()
    return pe.spTensor(f, dev_coords(coords), None, [0, 0, 0], coords[:, 1:].max(0).tolist(), batchsize=1)


def _planned_map(coords):
    planner = MapPlanner()
    x = _tensor(coords)
    prebuild_maps(x, [(3, 1, 0)], planner)
    assert planner.plans
    return next(iter(x.kmaps.values())), planner


def test_the_order_of_a_planned_map_lies_in_its_plan():
    """Not in the arena of the forward that built it: that is handed out again by the next forward, while the map's
    plan holds the map until its next cloud."""
    km, planner = _planned_map(synth.random_cloud(seed=9, n=6000, extent=24))
    arena = backend.ForwardArena(torch.device(DEV))
    for _ in range(2):          # the first pass measures what the arena needs, in the second it has memory
        km.__dict__.pop("_blocks", None)
        with backend.allocate_from(arena):
            backend._new(1 << 20, torch.uint8, torch.device(DEV))
            order = backend.block_order(km)
    plan = next(iter(planner.plans.values())).arena
    assert plan.data_ptr() <= order.data_ptr() and order.data_ptr() + 4 * order.numel() <= plan.data_ptr() + plan.numel()
    assert backend.block_order(km).data_ptr() == order.data_ptr()


def test_a_tensor_goes_through_a_planned_network_again():
    """a, b, b: the second pass over b finds b's maps, and their block orders, where the first one left them."""
    torch.manual_seed(6)
    model = nets.SparseResUNet(4, 20).to(DEV).eval().fuse_bn().half()
    clouds = [synth.random_cloud(seed=s, n=40000, extent=40) for s in (1, 2)]
    with torch.no_grad():
        want = [model(_tensor(c)).feats.clone() for c in clouds]
        model.use_planner()
        a, b = (_tensor(c) for c in clouds)
        for _ in range(2):
            assert torch.equal(model(a).feats, want[0])
            a = _tensor(clouds[0])
        for _ in range(3):
            assert torch.equal(model(b).feats, want[1])
        assert any("_blocks" in km.__dict__ for km in b.kmaps.values())


@pytest.mark.parametrize("on_default", [False, True])
@pytest.mark.parametrize("planned", [False, True])
def test_another_stream_waits_for_the_order(planned, on_default):
    coords = synth.random_cloud(seed=9, n=60000, extent=44)
    km = _planned_map(coords)[0] if planned else gpu_map(coords, (3, 3, 3), batchsize=1)
    f = torch.as_tensor(synth.features(1, km.n_out, 128), device=DEV).half()
    w = torch.as_tensor(synth.weights(2, 27, 128, 128), device=DEV).half()
    packed = backend.pack_weights(w)
    first, second = torch.cuda.default_stream() if on_default else torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        torch.cuda._sleep(20000000)          # the order is far from ready when the layer is queued
        backend.block_order(km)
    assert km._blocks[False][1] == first.cuda_stream
    with torch.cuda.stream(second):
        got = backend.conv_forward(f, w, km, DATAFLOW_OS, packed=packed)
        queued = torch.cuda.Event()
        queued.record()
    assert not queued.query()                # it waits on the GPU, the host did not
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        torch.cuda._sleep(20000000)
    with torch.cuda.stream(second):          # later layers do not wait for what the builder's stream does by then
        again = backend.conv_forward(f, w, km, DATAFLOW_OS, packed=packed)
        second.synchronize()
    assert not first.query()
    assert torch.equal(again, got)
    assert torch.equal(got, backend.conv_forward(f, w, km, DATAFLOW_OS, packed=packed))


@pytest.mark.parametrize("warm", [False, True])
def test_capture_of_a_wide_layer(warm):
    """A layer captured on the graph's stream, its order built before on another stream or inside the capture: every
    replay gives the eager result, and eager calls before the first replay do not read what only the graph computes."""
    km = gpu_map(synth.random_cloud(seed=9, n=20000, extent=32), (3, 3, 3), batchsize=1)
    f = torch.as_tensor(synth.features(1, km.n_out, 128), device=DEV).half()
    w = torch.as_tensor(synth.weights(2, 27, 128, 128), device=DEV).half()
    packed = backend.pack_weights(w)
    out = torch.zeros((km.n_out, 128), dtype=torch.float16, device=DEV)
    other = gpu_map(synth.random_cloud(seed=9, n=20000, extent=32), (3, 3, 3), batchsize=1)
    want = backend.conv_forward(f, w, other, DATAFLOW_OS, packed=packed)
    if warm:
        backend.conv_forward(f, w, km, DATAFLOW_OS, packed=packed)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        backend.conv_forward(f, w, km, DATAFLOW_OS, packed=packed, out=out)
    assert (False in km.__dict__.get("_blocks", {})) == warm
    assert torch.equal(backend.conv_forward(f, w, km, DATAFLOW_OS, packed=packed), want)
    for _ in range(3):
        out.fill_(float("nan"))
        (f * 2).sum().item()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_the_routes_of_a_planned_map_lie_in_its_plan():
    coords = synth.random_cloud(seed=9, n=6000, extent=24)
    planner, x = MapPlanner(), _tensor(coords)
    prebuild_maps(x, [(2, 2, 0)], planner)
    km = next(iter(x.kmaps.values()))
    plan = next(iter(planner.plans.values())).arena
    spans = []
    with backend.allocate_from(backend.ForwardArena(torch.device(DEV))):
        for transposed in (False, True):
            route = backend.pair_route(km, transposed)
            assert plan.data_ptr() <= route.data_ptr() and route.data_ptr() + 4 * route.numel() <= plan.data_ptr() + plan.numel()
            assert (km.route_t if transposed else km.route) is route and backend.pair_route(km, transposed) is route
            spans.append((route.data_ptr(), route.data_ptr() + 4 * route.numel()))
    assert spans[0][1] <= spans[1][0] or spans[1][1] <= spans[0][0]
