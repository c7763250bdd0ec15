"""The native host side of a layer against the general path: the same results for every layout either takes, the same errors."""
import pytest
import torch

from pcengine_amd import _lib, backend, synth
from pcengine_amd.backend import BLOCKS_LEAD, DATAFLOW_FDS, DATAFLOW_OS, DATAFLOW_OSO
from tests.util import DEV, gpu_map

pytestmark = pytest.mark.gpu


def general(monkeypatch, fn):
    with monkeypatch.context() as m:
        for name in _lib._NATIVE:
            m.setattr(_lib, name, lambda *args: None)
        return fn()


@pytest.fixture
def answers(monkeypatch):
    """What the native calls answer, by name, in the order of the calls."""
    _lib.host()
    seen = {name: [] for name in _lib._NATIVE}

    def record(name, fn):
        def call(*args):
            seen[name].append(fn(*args))
            return seen[name][-1]
        return call
    for name in _lib._NATIVE:
        monkeypatch.setattr(_lib, name, record(name, getattr(_lib, name)))
    return seen


def outcome(fn):
    try:
        return fn().clone()
    except Exception as e:         # (the ordered rows refuse odd pointers)
        return type(e), str(e)


def matrix(n, c, dtype, layout, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    f = torch.randn((n, c), generator=g, device=DEV).to(dtype)
    if layout == "slice":
        wide = torch.zeros((n, c + 24), dtype=dtype, device=DEV)
        wide[:, 8:8 + c] = f
        return wide[:, 8:8 + c]
    if layout == "columns":        # neither dense rows nor a slice of them
        return f.t().contiguous().t()
    if layout == "odd":            # not on a 16-byte boundary
        return torch.empty(n * c + 1, dtype=dtype, device=DEV)[1:].view(n, c).copy_(f)
    return f


@pytest.mark.parametrize("layout", ["dense", "slice", "columns", "odd"])
@pytest.mark.parametrize("dtype,df,c_in,c_out,ks,stride,transposed", [
    (torch.float16, DATAFLOW_OSO, 32, 48, (3, 3, 3), (1, 1, 1), False),
    (torch.float32, DATAFLOW_OSO, 16, 16, (3, 3, 3), (1, 1, 1), False),
    (torch.float16, BLOCKS_LEAD, 128, 192, (3, 3, 3), (1, 1, 1), False),
    (torch.float16, DATAFLOW_OS, 128, 192, (2, 2, 2), (2, 2, 2), True),
    (torch.float32, DATAFLOW_OS, 64, 40, (3, 3, 3), (1, 1, 1), False),
    (torch.float16, DATAFLOW_FDS, 64, 96, (2, 2, 2), (2, 2, 2), True),
    (torch.float16, DATAFLOW_FDS, 64, 96, (2, 2, 2), (2, 2, 2), False),
    (torch.float32, DATAFLOW_FDS, 20, 24, (3, 3, 3), (1, 1, 1), False)])
def test_layer(monkeypatch, answers, layout, dtype, df, c_in, c_out, ks, stride, transposed):
    km = gpu_map(synth.random_cloud(seed=3, n=1500, extent=14), ks, stride)
    n_in, n_out = (km.n_out, km.n_in) if transposed else (km.n_in, km.n_out)
    x = matrix(n_in, c_in, dtype, layout, 1)
    w = matrix(km.kv * c_in, c_out, dtype, "dense", 2).view(km.kv, c_in, c_out) * 0.1
    b, r = matrix(1, c_out, dtype, "dense", 3)[0], matrix(n_out, c_out, dtype, layout, 4)
    packed = backend.pack_weights(w)

    def run(**kw):
        return backend.conv_forward(x, w, km, df, transposed=transposed, packed=packed, **kw)
    for kw in (dict(), dict(bias=b, act="relu"), dict(bias=b, residual=r, act=("leaky_relu", 0.1)),
               dict(out=torch.zeros((n_out, c_out + 16), dtype=dtype, device=DEV)[:, 8:8 + c_out])):
        answers["layer"].clear()
        got, want = outcome(lambda: run(**kw)), general(monkeypatch, lambda: outcome(lambda: run(**kw)))
        # dense rows and slices of wider ones (of whole 16-byte pieces, as a residual dense rows) are taken; on odd pointers the
        # output-stationary layers are not asked for, and what the ordered rows refuse is the library's answer
        took = [type(a) for a in answers["layer"]]
        if layout == "columns" or (layout == "slice" and ("residual" in kw or c_in % 8)):
            assert took == [type(None)]
        elif layout == "odd" and df == DATAFLOW_OS:
            assert took == []
        else:
            assert took == [torch.Tensor if torch.is_tensor(got) else int]
        assert torch.equal(got, want) if torch.is_tensor(got) else (got == want and layout == "odd" and df == DATAFLOW_OSO), (sorted(kw), got, want)
    for bad, error in ((dict(bias=b[:-1]), ValueError), (dict(residual=r[:-1]), ValueError), (dict(act="tanh"), ValueError),
                       (dict(out=torch.zeros((n_out, c_out + 1), dtype=dtype, device=DEV)), ValueError)):
        with pytest.raises(error):
            run(**bad)
    with pytest.raises(ValueError):
        backend.conv_forward(x[:-1], w, km, df, transposed=transposed)
    with pytest.raises(TypeError):
        backend.conv_forward(x.to(torch.float16 if dtype == torch.float32 else torch.float32), w, km, df, transposed=transposed)


@pytest.mark.parametrize("dtype,df,c_in,c_out,ks,stride,transposed,arrays", [
    (torch.float16, DATAFLOW_OSO, 32, 48, (3, 3, 3), (1, 1, 1), False, ("nbr_out", "order")),
    (torch.float16, BLOCKS_LEAD, 128, 192, (3, 3, 3), (1, 1, 1), False, ("nbr_out",)),
    (torch.float32, DATAFLOW_OS, 64, 40, (3, 3, 3), (1, 1, 1), False, ("nbr_out",)),
    (torch.float16, DATAFLOW_FDS, 64, 96, (2, 2, 2), (2, 2, 2), True, ("imap", "omap", "islot", "icsr", "kpos", "qkpos")),
    (torch.float32, DATAFLOW_FDS, 20, 24, (3, 3, 3), (1, 1, 1), False, ("imap", "omap", "oslot", "ocsr", "kpos", "qkpos"))])
def test_kept_layouts_follow_the_maps_arrays(answers, dtype, df, c_in, c_out, ks, stride, transposed, arrays):
    """Later calls over a map take the layout of the first; none reads an array that the map does not hold any more."""
    km = gpu_map(synth.random_cloud(seed=3, n=1500, extent=14), ks, stride)
    x = matrix(km.n_out if transposed else km.n_in, c_in, dtype, "dense", 1)
    w = matrix(km.kv * c_in, c_out, dtype, "dense", 2).view(km.kv, c_in, c_out) * 0.1
    packed = backend.pack_weights(w)
    run = lambda: backend.conv_forward(x, w, km, df, transposed=transposed, packed=packed).clone()
    want = run()
    kept = list(km._calls.values())
    assert len(kept) == 1 and torch.equal(run(), want) and list(km._calls.values())[0] is kept[0]
    for name in arrays:
        old = getattr(km, name)
        setattr(km, name, old.clone())
        assert torch.equal(run(), want)
        assert not any(v is old for call in km._calls.values() for v in call[1]) and any(v is getattr(km, name) for call in km._calls.values() for v in call[1])
    assert [type(a) for a in answers["layer"]] == [torch.Tensor] * (2 + len(arrays))


@pytest.mark.parametrize("layout", ["dense", "columns", "odd"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_dense_norm_and_kernel_gradient(monkeypatch, answers, dtype, layout):
    n, c, c_out = 700, 40, 24
    km = gpu_map(synth.random_cloud(seed=3, n=1500, extent=14), (3, 3, 3))
    x, dy = matrix(n, c, dtype, layout, 1), matrix(n, c, dtype, layout, 2)
    w, b = matrix(c, c_out, dtype, "dense", 3), matrix(1, c_out, dtype, "dense", 4)[0]
    run = lambda: backend.dense_forward(x, w, backend.pack_weights(w), bias=b, act="relu")
    assert torch.equal(run(), general(monkeypatch, run))
    weight, bias = torch.rand(c, device=DEV), torch.rand(c, device=DEV)

    def norm():
        mean, var = torch.zeros(c, device=DEV), torch.ones(c, device=DEV)
        y, m, s = backend.bn_forward(x, weight, bias, mean, var, True, 0.1, 1e-5, act="relu", residual=dy)
        return [y, m, s, mean, var, *backend.bn_backward(x, dy, weight, m, s, True, y_act=y, act="relu")]
    assert all(torch.equal(p, q) for p, q in zip(norm(), general(monkeypatch, norm)))
    f, g = matrix(km.n_in, c, dtype, layout, 5), matrix(km.n_out, c_out, dtype, layout, 6)
    p, q = backend.conv_wgrad(f, g, km), general(monkeypatch, lambda: backend.conv_wgrad(f, g, km))
    # one kernel both times: its fp32 atomics add in another order, 2^-24 of a sum of 1500 products each
    assert p.shape == q.shape and ((p - q).norm() / q.norm()).item() <= 2 ** -24 * 1500 ** 0.5
    # one native call of each (the general path's are not recorded)
    kind = type(None) if layout == "columns" else torch.Tensor
    taken = {"layer": kind, "wgrad": kind, "bn_forward": type(None) if layout == "columns" else tuple,
             "bn_backward": type(None) if layout == "columns" else tuple}
    assert {name: [type(a) for a in seen] for name, seen in answers.items()} == {name: [t] for name, t in taken.items()}
    with pytest.raises(ValueError):
        backend.conv_wgrad(f[:-1], g, km)
    with pytest.raises(ValueError):
        backend.bn_forward(x, weight, bias, torch.zeros(c + 1, device=DEV), None, True, 0.1, 1e-5)


@pytest.mark.parametrize("df,c_in,c_out,ks,stride,transposed", [
    (DATAFLOW_FDS, 64, 96, (2, 2, 2), (2, 2, 2), False), (DATAFLOW_FDS, 32, 48, (3, 3, 3), (1, 1, 1), False),
    (DATAFLOW_OS, 32, 48, (3, 3, 3), (1, 1, 1), False), (DATAFLOW_OS, 64, 40, (2, 2, 2), (2, 2, 2), True)])
def test_no_memory_is_taken_without_packed_weights(monkeypatch, df, c_in, c_out, ks, stride, transposed):
    """fp16 layers that were given an output and a buffer, but no packed kernel: nothing is packed for them."""
    km = gpu_map(synth.random_cloud(seed=3, n=1500, extent=14), ks, stride, want_nbr_in=transposed)
    n_in, n_out = (km.n_out, km.n_in) if transposed else (km.n_in, km.n_out)
    x, out = matrix(n_in, c_in, torch.float16, "dense", 1), torch.empty((n_out, c_out), dtype=torch.float16, device=DEV)
    w = matrix(km.kv * c_in, c_out, torch.float16, "dense", 2).view(km.kv, c_in, c_out) * 0.1
    buffer = torch.empty(km.M * c_out, dtype=torch.float16, device=DEV)
    run = lambda: backend.conv_forward(x, w, km, df, transposed=transposed, out=out, buffer=buffer)
    run()
    taken = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    before = taken()
    got = run()
    assert taken() == before
    assert torch.equal(got.clone(), general(monkeypatch, run))


def test_a_declined_call_leaves_the_arena_as_it_was(monkeypatch):
    """Layers that the general path takes in the end ask the forward's arena for one output, as without the native call."""
    km = gpu_map(synth.random_cloud(seed=3, n=1500, extent=14), (3, 3, 3))
    x, wide = matrix(km.n_in, 64, torch.float16, "dense", 1), matrix(km.n_in, 64, torch.float16, "slice", 1)
    w, w1 = matrix(27 * 64, 48, torch.float16, "dense", 2).view(27, 64, 48), matrix(64, 48, torch.float16, "dense", 3)
    residual = matrix(km.n_out, 48, torch.float16, "slice", 4)
    arena = backend.ForwardArena(DEV)

    def run():
        p, p1 = backend.pack_weights(w), backend.pack_weights(w1)
        with backend.allocate_from(arena):
            outs = [backend.conv_forward(x, w, km, DATAFLOW_OSO, packed=p, residual=residual), backend.dense_forward(wide, w1, p1),
                    backend.conv_forward(x, w, km, DATAFLOW_OSO, packed=p)]
        return arena.need, outs

    run()
    for _ in range(2):
        (need, outs), (plain, same) = run(), general(monkeypatch, run)
        assert need == plain == 3 * (-(-km.n_out * 48 * 2 // 256) * 256)
