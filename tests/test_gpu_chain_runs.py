"""The occupancy map of the chained strided levels: rows that share a word, across wavefronts and gaps."""
import numpy as np
import pytest
import torch

from pcengine_amd import backend, synth
from tests.util import DEV, dev_coords

pytestmark = pytest.mark.gpu


def test_runs_of_a_word_across_wavefronts_and_gaps():
    """Output coordinates of strided levels where consecutive rows share a word of the occupancy map, a few of them or many, with
    clipped rows between."""
    rows = [(0, x, y, z) for x in range(7) for y in range(9) for z in range(0, 130, 1 + (x * y) % 3)]
    c = torch.tensor(rows, dtype=torch.int32, device=DEV)
    for cmax in ([6, 8, 129], [6, 5, 70]):       # the second box clips rows in the middle of runs
        chain = [backend.Geom.make((2, 2, 2), (2, 2, 2), (0, 0, 0), [0, 0, 0], m, False)
                 for m in (lambda a: [a, backend.strided_coords_max(a, (2, 2, 2), (2, 2, 2), (0, 0, 0))])(
                     backend.strided_coords_max(cmax, (2, 2, 2), (2, 2, 2), (0, 0, 0)))]
        outs = backend.build_out_coords_chain(c, chain, 1)
        assert outs is not None
        want = c
        for out, g in zip(outs, chain):
            want = torch.cat([want[:, :1], want[:, 1:] // 2], dim=1)
            top = torch.tensor(list(g.cmax), device=DEV)
            want = torch.unique(want[(want[:, 1:] <= top).all(dim=1)], dim=0)
            assert torch.equal(out, want.int())


@pytest.mark.parametrize("order", ["sorted", "random"])
@pytest.mark.parametrize("n,extent", [(800, 33), (9000, 34), (40000, 45), (40000, 70)])
def test_levels_with_many_rows_a_word(n, extent, order):
    """Below and above the density from which the runs of a wavefront are combined, down to a level of one word."""
    c = synth.random_cloud(seed=n, n=n, extent=extent)
    c = c[np.lexsort(c.T[::-1])] if order == "sorted" else c[np.random.default_rng(0).permutation(len(c))]
    chain, m = [], c[:, 1:].max(0).tolist()
    for _ in range(5):
        m = backend.strided_coords_max(m, (2, 2, 2), (2, 2, 2), (0, 0, 0))
        chain.append(backend.Geom.make((2, 2, 2), (2, 2, 2), (0, 0, 0), [0, 0, 0], m, False))
    want = dev_coords(c)
    for out, g in zip(backend.build_out_coords_chain(want, chain, 1), chain):
        want = torch.cat([want[:, :1], want[:, 1:] // 2], dim=1)
        want = torch.unique(want[(want[:, 1:] <= torch.tensor(list(g.cmax), device=DEV)).all(dim=1)], dim=0)
        assert torch.equal(out, want.int())
