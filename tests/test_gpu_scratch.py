"""Memory of a call over a map whose arrays are built: none with ``out`` and a large enough ``buffer``, and no partial sums
where no tile is cut."""
import pytest
import torch

from pcengine_amd import _lib, backend, synth
from pcengine_amd.backend import DATAFLOW_OS
from tests.util import DEV, gpu_map

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,extent,cuts", [(3000, 200, False), (30000, 34, True)])
def test_block_layer_allocates_nothing(n, extent, cuts):
    km = gpu_map(synth.random_cloud(seed=5, n=n, extent=extent), (3, 3, 3), batchsize=1)
    lib, c = _lib.load(), 256
    need = lib.pce_conv_osb_scratch_bytes(km.n_out, km.M, c, c, 27)
    assert need == (lib.pce_conv_osb_workspace_bytes(km.n_out, c) if cuts else 0)
    f = torch.as_tensor(synth.features(1, km.n_out, c), device=DEV).half()
    w = torch.as_tensor(synth.weights(2, 27, c, c), device=DEV).half()
    packed = backend.pack_weights(w)
    want = backend.conv_forward(f, w, km, DATAFLOW_OS, packed=packed)
    out = torch.empty_like(want)
    buffer = torch.empty(need // 4, device=DEV) if cuts else None
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    before = count()
    backend.conv_forward(f, w, km, DATAFLOW_OS, packed=packed, out=out, buffer=buffer)
    assert count() == before
    assert torch.equal(out, want)
    if cuts:                    # a buffer that is too small, or not aligned, does not serve
        for other in (buffer[1:], torch.empty(need // 4 - 1, device=DEV)):
            backend.conv_forward(f, w, km, DATAFLOW_OS, packed=packed, out=out, buffer=other)
            assert torch.equal(out, want)


def test_entry_point_needs_a_workspace_only_where_tiles_are_cut():
    lib = _lib.load()
    n, c = 30000, 256
    assert lib.pce_conv_osb_scratch_bytes(n, 9 * n, c, c, 27) > 0
    # null where it is needed: refused before anything is launched
    assert lib.pce_conv_fwd_osb(16, 16, 16, _lib.PCE_F16, n, n, 9 * n, c, c, 27, 16, 16, None, 0, None, None) == _lib.PCE_EWORKSPACE
    assert lib.pce_conv_osb_scratch_bytes(n, 0, 64, 96, 27) == 0 and lib.pce_conv_osb_scratch_bytes(0, 0, c, c, 27) == 0
