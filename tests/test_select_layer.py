"""The selector with the block kernel among its answers, and what a layer takes whose rows or pointers that kernel does not."""
import pytest
import torch

import pcengine_amd as pe
from pcengine_amd import _lib, backend, synth
from tests.util import DEV


def test_block_kernel_is_answered_where_it_leads_and_can_run():
    lib = _lib.load()
    F16, F32, OSB = _lib.PCE_F16, _lib.PCE_F32, _lib.DATAFLOW_OSB
    for n, rho in ((3000, 8), (25000, 9), (66000, 9), (90000, 3), (680000, 5), (950000, 1.2), (950000, 0.1)):
        m = int(n * rho)
        for ci in (16, 48, 64, 96, 128, 192, 256, 512):
            for co in (32, 64, 72, 96, 128, 256, 512, 1024):
                for kv, mid in ((27, 13), (27, -1), (8, 3), (8, -1), (125, 62)):
                    for tr in (0, 1):
                        for dt in (F16, F32):
                            got = lib.pce_select_layer(n, n, m, ci, co, kv, mid, tr, dt)
                            leads = lib.pce_conv_osb_leads(n, m, ci, co, kv, mid, dt) and (not tr or kv % 2)
                            assert got == (OSB if leads else lib.pce_select_dataflow(n, n, m, ci, co, kv, mid, tr, dt))
    # features beyond what its gathers address: 2 bytes of 5.3 M rows x 384 channels
    n = 5300000
    assert lib.pce_conv_osb_leads(n, 6 * n, 384, 384, 27, 13, F16) == 1
    assert lib.pce_select_layer(n, n, 6 * n, 384, 384, 27, 13, 0, F16) == lib.pce_select_dataflow(n, n, 6 * n, 384, 384, 27, 13, 0, F16) == _lib.DATAFLOW_FDS


@pytest.mark.gpu
def test_layer_the_block_kernel_cannot_read():
    """An odd pointer, or rows too far apart for it: deferred scatter as for any layer it does not lead on, not the tile
    kernel that multiplies every offset."""
    coords = synth.random_cloud(seed=5, n=30000, extent=42)
    layer = pe.conv3d(128, 192, 3, 1, bias=True).to(DEV).half().eval()
    layer.bias.data = torch.randn(192, device=DEV).half()

    def through(feats):
        x = pe.spTensor(feats, torch.as_tensor(coords, device=DEV).int(), None, [0, 0, 0], coords[:, 1:].max(0).tolist(), batchsize=1)
        with torch.no_grad():
            y = layer(x).feats
        return y, next(iter(x.kmaps.values()))

    n = len(coords)
    f = torch.randn((n, 128), device=DEV).half()
    want, km = through(f)
    assert "_blocks" in km.__dict__ and backend.select_dataflow(km, 128, 192, torch.float16) is backend.BLOCKS_LEAD
    assert {backend.DATAFLOW_OS: "os"}[backend.BLOCKS_LEAD] == "os"      # what a caller compares or looks up
    assert _lib.load().pce_select_dataflow(n, n, km.M, 128, 192, 27, 13, 0, _lib.PCE_F16) == backend.DATAFLOW_FDS
    odd = torch.empty(n * 128 + 4, dtype=torch.float16, device=DEV)[4:].view(n, 128).copy_(f)
    assert odd.data_ptr() % 16 == 8
    far = torch.empty((n, 0xF0000000 // (2 * n) // 8 * 8 + 8), dtype=torch.float16, device=DEV)[:, :128]
    far.copy_(f)
    for feats in (odd, far):
        got, km = through(feats)
        assert "_blocks" not in km.__dict__ and km.has_csr
        assert ((got.float() - want.float()).norm() / want.float().norm()).item() < 2e-3


def test_selector_on_measured_wide_layers():
    """fp16 layers timed with every dataflow; us in brackets: block kernel, the one it stands against."""
    lib = _lib.load()
    FDS, OSO, OSB = _lib.DATAFLOW_FDS, _lib.DATAFLOW_OSO, _lib.DATAFLOW_OSB
    for n, rho, c_in, c_out, want in [
            (12036, 7.5, 384, 384, FDS),       # random clouds: 112, 76
            (11437, 9.4, 512, 512, FDS),       # 155, 123
            (18729, 9.8, 384, 256, FDS),       # 114, 94
            (20202, 7.2, 256, 128, FDS),       # 51, 43
            (32025, 5.4, 192, 128, FDS),       # 58, 45
            (113177, 2.9, 256, 128, FDS),      # 111, 82
            (199899, 3.7, 384, 384, FDS),      # 1.13 of it
            (82198, 4.2, 96, 96, OSO),         # 1.22 of it
            (66200, 8.9, 96, 96, OSO),         # a level of a scan: 58, 55
            (12063, 11.6, 512, 512, FDS),      # a level of indoor scenes: 3 to 5 % behind
            (155843, 3.6, 256, 1024, FDS),     # 1260, 1084
            (302352, 7.7, 768, 512, FDS),      # 4814, 3833
            (16369, 12.1, 64, 192, _lib.DATAFLOW_OS),   # 36, 30 for the dense tiles
            (821, 6.5, 192, 192, OSB),         # 0.81 of it
            (12036, 7.5, 128, 192, OSB),       # equal
            (28103, 10.1, 256, 256, OSB),      # 0.87 of it
            (60159, 7.7, 192, 192, OSB),       # 0.68
            (66200, 8.9, 256, 256, OSB),       # a level of a scan: 0.67
            (679728, 5.2, 192, 192, OSB),      # indoor scenes: 0.42
            (276205, 8.7, 384, 256, OSB),      # 0.42
            (69431, 9.9, 512, 512, OSB),       # 0.52
            (69431, 9.9, 768, 512, OSB),       # 0.60
            (16455, 10.9, 256, 512, OSB),      # 0.73
            (806, 13.1, 256, 256, OSB),        # 0.83
            (261532, 7.8, 64, 96, OSB),        # 0.84 of the ordered rows
            (106646, 5.5, 64, 128, OSB)]:      # 0.82
        assert lib.pce_select_layer(n, n, round(n * rho), c_in, c_out, 27, 13, 0, _lib.PCE_F16) == want, (n, rho, c_in, c_out)
