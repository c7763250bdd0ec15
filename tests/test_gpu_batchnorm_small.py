"""The batch normalisation of few rows in one launch: its edges against fp64, and bit for bit against the passes of many rows (which a
call whose output lies in an operand's memory takes)."""
import pytest
import torch

from pcengine_amd import _lib, backend
from tests.util import DEV

pytestmark = pytest.mark.gpu
CODE = {torch.float16: _lib.PCE_F16, torch.float32: _lib.PCE_F32}
# rel-L2: fp16 outputs are rounded once (2^-11 at most, 2.8e-4 rms); fp32 sums over 8 rows and one rounding of the coefficients
BAR = {torch.float16: 6e-4, torch.float32: 1e-6}


def rel(a, b):
    return ((a.double() - b).norm() / b.norm().clamp_min(1e-30)).item()


def data(n, c, dtype):
    g = torch.Generator(device=DEV).manual_seed(n * 1000 + c)
    r = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    return (r(n, c) * 2 + 0.5).to(dtype), r(n, c).to(dtype), r(n, c).to(dtype), r(c).abs() + 0.5, r(c)


def forward(x, res, y, w, b, act, batches=None):
    n, c = x.shape
    lib = _lib.load()
    mean, var, s = torch.zeros(c, device=DEV), torch.ones(c, device=DEV), torch.empty(2, c, device=DEV)
    ws = torch.empty(lib.pce_bn_workspace_bytes(n, c), dtype=torch.uint8, device=DEV)
    ptr = lambda t: None if t is None else t.data_ptr()
    _lib.check(lib.pce_bn_forward_counted(x.data_ptr(), ptr(res), y.data_ptr(), CODE[x.dtype], n, c, w.data_ptr(), b.data_ptr(), mean.data_ptr(),
                                          var.data_ptr(), ptr(batches), 1, 0.1, 1e-5, s[0].data_ptr(), s[1].data_ptr(), ws.data_ptr(),
                                          ws.numel(), act, 0.1, torch.cuda.current_stream().cuda_stream))
    return mean, var, s


def backward(x, dy, y, w, s, act, dx, masked=None):
    n, c = x.shape
    lib = _lib.load()
    g = torch.empty(2, c, device=DEV)
    ws = torch.empty(lib.pce_bn_workspace_bytes(n, c), dtype=torch.uint8, device=DEV)
    _lib.check(lib.pce_bn_backward_masked(x.data_ptr(), dy.data_ptr(), y.data_ptr(), act, 0.1, None if masked is None else masked.data_ptr(),
                                          dx.data_ptr(), CODE[x.dtype], n, c, w.data_ptr(), s[0].data_ptr(), s[1].data_ptr(), 1,
                                          g[0].data_ptr(), g[1].data_ptr(), ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    return g


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n,c", [(2, 8), (63, 8), (64, 24), (257, 40), (1000, 16), (2047, 96), (2048, 128), (2049, 128), (1024, 384), (1025, 384),
                                 (1536, 256), (1537, 256), (4096, 64), (4096, 256), (4097, 256), (300, 2056)])
@pytest.mark.parametrize("act", [_lib.ACT_NONE, _lib.ACT_RELU, _lib.ACT_LEAKY_RELU])
def test_against_fp64_and_the_passes_of_many_rows(n, c, dtype, act):
    x, dy, res, w, b = data(n, c, dtype)
    y, count = torch.empty_like(x), torch.full((), 6, dtype=torch.int64, device=DEV)
    mean, var, s = forward(x, res, y, w, b, act, count)
    assert int(count) == 7
    xd = x.double()
    m, v = xd.mean(0), xd.var(0, unbiased=False)
    xh = (xd - m) * (v + 1e-5).rsqrt()
    want = xh * w.double() + b.double() + res.double()
    want = {_lib.ACT_NONE: want, _lib.ACT_RELU: want.relu(), _lib.ACT_LEAKY_RELU: torch.where(want > 0, want, want * 0.1)}[act]
    if n > 2:    # (two rows: eps decides)
        assert rel(y, want) <= BAR[dtype] and rel(s[0], m) <= 1e-6 and rel(s[1], (v + 1e-5).rsqrt()) <= 1e-6
        assert rel(mean, 0.1 * m) <= 1e-6 and rel(var, 0.9 + 0.1 * v * n / (n - 1)) <= 1e-6
    # in place: the passes of many rows
    y2 = x.clone()
    mean2, var2, s2 = forward(y2, res, y2, w, b, act)
    for p, q in ((y, y2), (mean, mean2), (var, var2), (s, s2)):
        assert torch.equal(p, q)

    g_exact = dy.double() * torch.where(y > 0, 1.0, {_lib.ACT_NONE: 1.0, _lib.ACT_RELU: 0.0, _lib.ACT_LEAKY_RELU: 0.1}[act]).double()
    dx = torch.empty_like(x)
    g = backward(x, dy, y, w, s, act, dx)
    if n > 2:
        gb, gw = g_exact.sum(0), (g_exact * xh).sum(0)
        want = w.double() * (v + 1e-5).rsqrt() * (g_exact - gb / n - xh * gw / n)
        scale = g_exact.abs().sum(0).norm()       # (gradients of a channel may cancel)
        assert rel(dx, want) <= 2 * BAR[dtype]
        assert (g[0].double() - gw).norm() <= 1e-6 * scale and (g[1].double() - gb).norm() <= 1e-6 * scale
    dx2 = dy.clone()
    g2 = backward(x, dx2, y, w, s, act, dx2)
    assert torch.equal(dx, dx2) and torch.equal(g, g2)
    if act == _lib.ACT_NONE:
        return
    # the masked gradient: torch's own values, and the norm's gradients from them
    dm, dx3 = torch.empty_like(x), torch.empty_like(x)
    g3 = backward(x, dy, y, w, s, act, dx3, dm)
    if act == _lib.ACT_RELU:
        assert torch.equal(dm, torch.ops.aten.threshold_backward(dy, y, 0.0))
    else:   # a product in fp32 rounded to fp16, or rounded to it at once: one unit in the last place apart at most, 2^-10 of the value
        want = torch.where(y > 0, dy, dy * 0.1)
        assert ((dm.double() - want.double()).abs() <= (2.0 ** -10 if dtype == torch.float16 else 0) * want.double().abs() + 2.0 ** -24).all()
    dx4 = dm.clone()
    g4 = backward(x, dx4, y, w, s, _lib.ACT_NONE, dx4)
    assert torch.allclose(dx3.double(), dx4.double(), rtol=2e-3 if dtype == torch.float16 else 1e-5, atol=1e-3 if dtype == torch.float16 else 1e-6)
    assert torch.allclose(g3, g4, rtol=1e-5, atol=1e-5 * float(g_exact.abs().sum(0).max()))


@pytest.mark.parametrize("n", [500, 5000])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_masked_gradient_where_values_are_not_finite(n, dtype):
    x, dy, res, w, b = data(n, 32, dtype)
    y = torch.relu(res)
    y[3, 4], y[7, 5], dy[11, 6], dy[12, 6], dy[13, 7] = float("nan"), float("inf"), float("inf"), float("nan"), float("-inf")
    s = torch.ones(2, 32, device=DEV)
    dm, dx = torch.empty_like(x), torch.empty_like(x)
    backward(x, dy, y, w, s, _lib.ACT_RELU, dx, dm)
    assert torch.equal(torch.nan_to_num(dm, 77.0), torch.nan_to_num(torch.ops.aten.threshold_backward(dy, y, 0.0), 77.0))
    assert torch.isfinite(dx[:, 8:]).all()


def test_module_counts_its_batches_on_the_device():
    import pcengine_amd as pe
    coords = torch.zeros((100, 4), dtype=torch.int32, device=DEV)
    for momentum in (0.1, None):
        bn = pe.BatchNorm(16, momentum=momentum).to(DEV)
        x = pe.spTensor(torch.randn(100, 16, device=DEV, requires_grad=True), coords, None, [0, 0, 0], [1, 1, 1])
        for _ in range(3):
            bn(x)
        assert int(bn.num_batches_tracked) == 3
        bn.eval()
        bn(x)
        assert int(bn.num_batches_tracked) == 3
    with pytest.raises(ValueError):
        backend.bn_backward(x.feats.detach(), x.feats.detach(), None, torch.zeros(16, device=DEV), torch.ones(16, device=DEV), True, masked=True)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("n,c", [(1, 8), (1025, 8), (1025, 5), (5003, 64), (20001, 33), (70001, 20), (60000, 24)])
def test_rows_behind_the_last_one_add_nothing(n, c, dtype):
    """Sums and maps of many rows, by full vectors and single columns: the last row, which stands in for rows that are not there, counts
    once, also where it is infinite."""
    x, dy, _, w, b = data(n, c, dtype)
    x[-1, 0], dy[-1, 0] = float("inf"), 1.0
    x[-1, 1], dy[-1, 1] = 3.0, float("inf")
    s = backend.col_sums(x, dy).double()
    want = torch.stack([x.double().sum(0), (x.double() * dy.double()).sum(0)])
    scale = torch.stack([x.double().abs().sum(0), (x.double() * dy.double()).abs().sum(0)])
    assert torch.equal(torch.isnan(s.view(2, c)), torch.isnan(want)) and torch.equal(torch.isinf(s.view(2, c)), torch.isinf(want))
    ok = torch.isfinite(want)
    # fp32 sums over eight rows, fp64 above, one rounding to fp32: at most 2^-24 (8 + 1 + 1) of the terms' sum
    assert ((s.view(2, c) - want).abs()[ok] <= 10 * 2.0 ** -24 * scale[ok]).all()
    y = torch.empty_like(x)
    k = torch.randn(3, c, device=DEV)
    lib = _lib.load()
    for d, kd in ((None, None), (dy, k[2])):
        whole = torch.full((n + 2, c), 7.0, device=DEV).to(dtype)
        y = whole[1:-1]
        if y.data_ptr() % 16 and c % 8 == 0:
            continue
        _lib.check(lib.pce_col_affine(x.data_ptr(), None if d is None else d.data_ptr(), y.data_ptr(), CODE[dtype], n, c, k[0].data_ptr(),
                                      None if kd is None else kd.data_ptr(), k[1].data_ptr(), _lib.ACT_NONE, 0.0,
                                      torch.cuda.current_stream().cuda_stream))
        want = x.double() * k[0].double() + k[1].double() + (0 if d is None else d.double() * kd.double())
        assert rel(y[:-1], want[:-1]) <= BAR[dtype] and rel(y[-1:, 2:], want[-1:, 2:]) <= 3 * BAR[dtype]
        assert bool((whole[0] == 7).all()) and bool((whole[-1] == 7).all())
