"""The kernel gradient into an array that another launch has cleared: the launch that transposes the kernel clears all of it and
nothing else, and the sums are those of the call that clears for itself."""
import pytest
import torch

from pcengine_amd import _lib, backend, synth
from tests.util import DEV, gpu_map

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("src,dst", [(torch.float32, torch.float32), (torch.float32, torch.float16), (torch.float16, torch.float16)])
@pytest.mark.parametrize("shape", [(27, 32, 32), (27, 31, 33), (8, 4, 70), (1, 1, 1), (3, 65, 8), (40, 24)])
@pytest.mark.parametrize("transpose,flip", [(True, True), (True, False), (False, False)])
def test_the_launch_clears_the_array_and_nothing_else(src, dst, shape, transpose, flip):
    w = torch.randn(shape, device=DEV).to(src)
    whole = torch.full((w.numel() + 128,), 7.0, device=DEV)
    zero = whole[64:64 + w.numel()].view(shape)
    got = backend.prepare_weights(w, dst, transpose, flip and w.dim() == 3, zero=zero)
    want = backend.prepare_weights(w, dst, transpose, flip and w.dim() == 3)
    assert torch.equal(got[0], want[0]) and (got[1] is None) == (want[1] is None) and (got[1] is None or torch.equal(got[1], want[1]))
    assert bool((zero == 0).all()) and bool((whole[:64] == 7).all()) and bool((whole[-64:] == 7).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("c_in,c_out", [(16, 16), (40, 72), (128, 128), (4, 32)])
@pytest.mark.parametrize("dense_rows", [True, False])
def test_sums_go_to_what_is_there(dtype, c_in, c_out, dense_rows):
    km = gpu_map(synth.random_cloud(seed=3, n=1200, extent=14), (3, 3, 3), batchsize=1)
    f, g = torch.randn((km.n_in, c_in), device=DEV).to(dtype), torch.randn((km.n_out, c_out), device=DEV).to(dtype)
    if not dense_rows:      # the general path
        f = torch.cat([f, f], dim=1)[:, :c_in]
    want = backend.conv_wgrad(f, g, km)
    zeros = torch.zeros((27, c_in, c_out), device=DEV)
    assert backend.conv_wgrad(f, g, km, zeros=zeros) is zeros
    scale = float(want.abs().max())
    assert float((zeros - want).abs().max()) <= 2e-6 * scale        # fp32 atomics in another order
    backend.conv_wgrad(f, g, km, zeros=zeros)
    assert float((zeros - 2 * want).abs().max()) <= 4e-6 * scale
    with pytest.raises(ValueError):
        backend.conv_wgrad(f, g, km, zeros=zeros[:26])


@pytest.mark.parametrize("need_feats,need_weight", [(True, True), (False, True), (True, False)])
def test_backward_twice_gives_the_same(need_feats, need_weight):
    km = gpu_map(synth.random_cloud(seed=3, n=1200, extent=14), (3, 3, 3), batchsize=1)
    f, g, w = torch.randn((km.n_in, 32), device=DEV).half(), torch.randn((km.n_out, 48), device=DEV).half(), torch.randn((27, 32, 48), device=DEV).half()
    one, two = (backend.conv_backward(f, w, km, g, need_feats=need_feats, need_weight=need_weight, weight_dtype=torch.float32) for _ in range(2))
    for a, b in zip(one, two):
        assert (a is None) == (b is None) and (a is None or torch.allclose(a, b, rtol=1e-5, atol=1e-4))
    if need_weight:
        want = backend.conv_wgrad(f, g, km)
        assert torch.allclose(one[1], want, rtol=1e-5, atol=1e-5 * float(want.abs().max())) and one[1].data_ptr() != two[1].data_ptr()
