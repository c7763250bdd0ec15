"""The one-launch weight preparation of a training step and the kernel gradient over every kind of pair list."""
import pytest
import torch

from pcengine_amd import backend

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("src,dst", [(torch.float32, torch.float16), (torch.float16, torch.float16), (torch.float32, torch.float32)])
@pytest.mark.parametrize("shape", [(27, 4, 32), (8, 96, 33), (1, 31, 65), (125, 8, 8), (20, 7), (27, 256, 192)])
def test_prepare_weights(src, dst, shape):
    w = torch.randn(shape, device="cuda").to(src)
    w.view(-1)[:3] = torch.tensor([float("inf"), float("nan"), -0.0])
    for transpose in (False, True):
        for flip in (False, True):
            if flip and w.dim() == 2:
                continue
            want = w.to(dst)
            want = want.transpose(-2, -1) if transpose else want
            want = (want.flip(0) if flip else want).contiguous()
            got, packed = backend.prepare_weights(w, dst, transpose, flip)
            assert got.shape == want.shape and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))
            if dst == torch.float16:
                ref = backend.pack_weights(want).view(torch.float16)
                assert torch.equal(packed.view(torch.float16).nan_to_num(7.0), ref.nan_to_num(7.0))
            else:
                assert packed is None
    # a kernel that is not contiguous is taken as it reads
    t = torch.randn(shape, device="cuda").to(src).transpose(-2, -1)
    assert torch.equal(backend.prepare_weights(t, dst)[0], t.to(dst))


class _Pairs:
    """A map of given pair lists, as much of one as the kernel gradient reads."""

    def __init__(self, counts, n, centre):
        g = torch.Generator().manual_seed(len(counts) + sum(counts))
        self.kv, self.n_in, self.n_out, self.subm = len(counts), n, n, centre
        self.ks = [3, 3, 3] if centre else [len(counts), 1, 1]
        self.imap = torch.randint(n, (max(1, sum(counts)),), generator=g, dtype=torch.int32)
        self.omap = torch.randint(n, (max(1, sum(counts)),), generator=g, dtype=torch.int32)
        pos, q = [0], [0]
        for c in counts:
            pos.append(pos[-1] + c)
            q.append(q[-1] + -(-c // 128) * 128)
        self.kpos, self.qkpos, self.qsum = torch.tensor(pos, dtype=torch.int32), torch.tensor(q, dtype=torch.int32), q[-1]


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("counts,n,centre,ci,co", [
    ([1] * 13 + [0] + [1] * 13, 1, True, 16, 16),               # a single row
    ([0] * 27, 129, True, 72, 40),                              # only the centre
    ([0, 127, 128, 129, 0, 1, 1030, 0], 300, False, 64, 96),    # edges of tiles, empty offsets, fewer tiles than XCDs
    ([300 + 37 * i for i in range(13)] + [0] + [700] * 13, 5000, True, 130, 257),   # several blocks of channels
    ([40] * 125, 500, False, 24, 8),                            # more offsets than lanes
    ([300000, 5, 0, 260000], 3000, False, 32, 32),              # runs of many tiles
    ([90000, 5, 0, 130, 180000, 0, 1], 3000, False, 72, 24),    # empty and one-tile offsets among long ones
    ([20000] * 13 + [0] + [20000] * 13, 20001, True, 16, 100),  # ... with a centre
    ([3000] * 130, 4000, False, 72, 16),                        # more offsets than any kernel map of the networks
])
def test_kernel_gradient_covers_every_pair(dtype, counts, n, centre, ci, co):
    km = _Pairs(counts, n, centre)
    g = torch.Generator().manual_seed(3)
    x = torch.randint(-3, 4, (n, ci), generator=g).to(dtype)
    d = torch.randint(-3, 4, (n, co), generator=g).to(dtype)
    want = torch.zeros(km.kv, ci, co)
    for w in range(km.kv):
        i, o = km.imap[km.kpos[w]:km.kpos[w + 1]].long(), km.omap[km.kpos[w]:km.kpos[w + 1]].long()
        want[w] = x[i].float().t() @ d[o].float()
    if centre:
        want[13] += x.float().t() @ d.float()
    for name in ("imap", "omap", "kpos", "qkpos"):
        setattr(km, name, getattr(km, name).cuda())
    # sums of whole numbers below 2^24: exact in any order
    assert torch.equal(backend.conv_wgrad(x.cuda(), d.cuda(), km).cpu(), want)
