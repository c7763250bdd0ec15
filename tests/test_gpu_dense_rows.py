"""fp16 layers of 33 to 64 columns on large clouds with many neighbours: four wavefronts that share an offset's weights."""
import numpy as np
import pytest
import torch

import pcengine_amd as pe
from pcengine_amd import backend, synth
from pcengine_amd.spconv import prebuild_maps
from tests.util import DEV, gpu_map

pytestmark = pytest.mark.gpu


def _map(n, density, seed):
    coords = torch.as_tensor(synth.random_cloud(seed=seed, n=n, extent=max(2, round((n / density) ** (1 / 3)))), device=DEV).int()
    x = pe.spTensor(torch.zeros((len(coords), 1), device=DEV), coords, None, [0, 0, 0], coords[:, 1:].max(0).values.tolist(), batchsize=1)
    prebuild_maps(x, [(3, 1, 0)])
    return next(iter(x.kmaps.values()))


# rows just beyond the line of the selection (more than 3072 groups of 32 rows with two neighbours), dense ones, and of a
# cloud whose rows with none or one are more than half
@pytest.mark.parametrize("n,density", [(125001, 0.25), (190011, 0.9), (250003, 0.06)])
@pytest.mark.parametrize("c_in,c_out,slices", [(16, 40, False), (32, 64, True), (48, 48, False), (64, 64, False), (64, 56, True)])
def test_sums_of_rows_that_share_weights(n, density, c_in, c_out, slices):
    km = _map(n, density, seed=11)
    backend.row_order(km)
    rows, split = km.n_out, km.order_nonzero - km.order_single
    assert split > 3072 * 32 and 3 * split >= rows
    gen = torch.Generator(device=DEV).manual_seed(c_in * 100 + c_out)
    wide = torch.randn((rows, c_in + (8 if slices else 0)), generator=gen, device=DEV).half()
    x = wide[:, :c_in]
    w = (torch.randn((27, c_in, c_out), generator=gen, device=DEV) * 0.1).half()
    bias = torch.randn(c_out, generator=gen, device=DEV).half()
    residual = torch.randn((rows, c_out), generator=gen, device=DEV).half()
    out = torch.full((rows, c_out + (8 if slices else 0)), 7.0, dtype=torch.float16, device=DEV)
    backend.conv_forward(x, w, km, backend.DATAFLOW_OSO, bias=bias, residual=residual, act="relu", out=out[:, :c_out])
    nbr = km.nbr_out.view(27, rows).long()
    nbr[13] = torch.arange(rows, device=DEV)
    want = torch.zeros((rows, c_out), dtype=torch.float64, device=DEV)
    size = torch.zeros((rows, c_out), dtype=torch.float64, device=DEV)
    for k in range(27):
        at = torch.nonzero(nbr[k] >= 0)[:, 0]
        f = x[nbr[k][at]].double()
        want[at] += f @ w[k].double()
        size[at] += f.abs() @ w[k].double().abs()
    want = want + bias.double() + residual.double()
    size = size + bias.double().abs() + residual.double().abs()
    # one rounding to fp16 of the result, and of every fp32 addition at most half a unit of what is summed
    bound = 2.0 ** -11 * want.abs() + (27 * c_in + 2) * 2.0 ** -24 * size + 2.0 ** -24
    got = out[:, :c_out].double()
    assert ((got - want.clamp(min=0)).abs() <= bound).all()
    if slices:
        assert (out[:, c_out:] == 7.0).all()


# four copies of a cloud, none near another: each has too few rows for the shared weights by itself, together they take them
@pytest.mark.parametrize("n,density", [(30001, 0.25), (44007, 0.9), (62003, 0.06)])
@pytest.mark.parametrize("c_in,c_out", [(32, 40), (32, 64), (48, 48), (64, 64)])
def test_same_bits_as_the_rows_alone(n, density, c_in, c_out):
    one = synth.random_cloud(seed=5, n=n, extent=round((n / density) ** (1 / 3)))
    one = one[np.lexsort(one[:, ::-1].T)]
    step = np.array([0, int(one[:, 1].max()) + 3, 0, 0], one.dtype)
    alone, four = (gpu_map(c, (3, 3, 3), batchsize=1) for c in (one, np.concatenate([one + k * step for k in range(4)])))
    split = [km.order_nonzero - km.order_single for km in (alone, four)]
    assert split[0] <= 3072 * 32 < split[1] and 3 * split[1] >= four.n_out and 2 * alone.order_nonzero > alone.n_out
    rows = alone.n_out
    gen = torch.Generator(device=DEV).manual_seed(c_in * 100 + c_out)
    x = torch.randn((rows, c_in), generator=gen, device=DEV).half()
    w = (torch.randn((27, c_in, c_out), generator=gen, device=DEV) * 0.1).half()
    bias = torch.randn(c_out, generator=gen, device=DEV).half()
    want = backend.conv_forward(x, w, alone, backend.DATAFLOW_OSO, bias=bias)
    got = backend.conv_forward(x.repeat(4, 1), w, four, backend.DATAFLOW_OSO, bias=bias)
    assert all(torch.equal(part, want) for part in got.view(4, rows, c_out))


@pytest.mark.parametrize("ks,density", [((3, 3, 1), 0.6), ((1, 3, 3), 0.6), ((2, 2, 2), 0.6)])
def test_kernels_of_fewer_offsets(ks, density):
    n, c_in, c_out = 165001, 48, 40
    km = gpu_map(synth.random_cloud(seed=6, n=n, extent=round((n / density) ** (1 / 3))), ks, batchsize=1)
    backend.row_order(km)
    rows, split = km.n_out, km.order_nonzero - km.order_single
    assert split > 3072 * 32 and 3 * split >= rows and rows <= 1024 * 128
    gen = torch.Generator(device=DEV).manual_seed(2)
    x = torch.randn((rows, c_in), generator=gen, device=DEV).half()
    w = (torch.randn((km.kv, c_in, c_out), generator=gen, device=DEV) * 0.1).half()
    out = torch.full((rows, c_out), float("nan"), dtype=torch.float16, device=DEV)
    backend.conv_forward(x, w, km, backend.DATAFLOW_OSO, out=out)
    kpos, mid = km.kpos.cpu().tolist(), backend._mid(km.ks)
    want = x.double() @ w[mid].double()
    size = x.double().abs() @ w[mid].double().abs()
    for k in range(km.kv):
        i, o = km.imap[kpos[k]:kpos[k + 1]].long(), km.omap[kpos[k]:kpos[k + 1]].long()
        want.index_add_(0, o, x[i].double() @ w[k].double())
        size.index_add_(0, o, x[i].double().abs() @ w[k].double().abs())
    # as above: one rounding to fp16, half a unit of what is summed per fp32 addition
    bound = 2.0 ** -11 * want.abs() + km.kv * c_in * 2.0 ** -24 * size + 2.0 ** -24
    assert ((out.double() - want).abs() <= bound).all()


def test_odd_pointers_of_a_selected_layer():
    """110 k rows at seven pairs or more: the selector's answer takes features, bias and output on any boundary."""
    km = gpu_map(synth.random_cloud(seed=3, n=110003, extent=62), (3, 3, 3), batchsize=1)
    rows = km.n_out
    assert rows > 73728 and 6 < km.M / rows <= 12
    df = backend._lib.load().pce_select_dataflow(rows, rows, km.M, 48, 40, 27, 13, 0, backend.PCE_F16)
    assert df == backend.select_dataflow(km, 48, 40, torch.float16) == backend.DATAFLOW_OS
    gen = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn((rows, 48), generator=gen, device=DEV).half()
    w = (torch.randn((27, 48, 40), generator=gen, device=DEV) * 0.1).half()
    bias = torch.randn(40, generator=gen, device=DEV).half()
    want = backend.conv_forward(x, w, km, df, bias=bias)

    def odd(t):
        return torch.empty(t.numel() + 4, dtype=t.dtype, device=DEV)[4:].view(t.shape).copy_(t)

    for feats, b, out in ((odd(x), bias, None), (x, odd(bias), None), (x, bias, odd(torch.full_like(want, 7.0)))):
        assert torch.equal(backend.conv_forward(feats, w, km, df, bias=b, out=out), want)
