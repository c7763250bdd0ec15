"""Column slabs of fp32 products: whatever their width, the sums of a row are the same."""
import pytest
import torch

from pcengine_amd import backend
from tests.util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c_in,c_out", [(2000, 128, 128), (16000, 256, 256), (16500, 256, 256), (32000, 128, 128), (32000, 96, 96), (33000, 96, 128),
                                          (57000, 64, 64), (57500, 64, 64), (65000, 16, 48), (60000, 16, 96), (127, 29, 35)])
def test_width_of_the_slabs_does_not_show(n, c_in, c_out):
    g = torch.Generator(device=DEV).manual_seed(n + c_in)
    x = torch.randn((70000, c_in), generator=g, device=DEV)          # 547 tiles: the widest slabs for any width
    w = torch.randn((c_in, c_out), generator=g, device=DEV)
    got = backend.dense_forward(x[:n], w)
    assert torch.equal(got, backend.dense_forward(x, w)[:n])
    want = x[:n].double() @ w.double()
    # c_in products, each rounded in fp32 and added: 2^-24 * sqrt(2 c_in) in the mean
    assert ((got - want).norm() / want.norm()).item() <= 2 ** -24 * (2 * c_in) ** 0.5
