"""The sort of the block order (``pce_osb_order``): stable, the same in every run, and no entry from behind the last row."""
import numpy as np
import pytest
import torch

from pcengine_amd import _lib
from tests.util import DEV

pytestmark = pytest.mark.gpu

WINDOW = 8192


def sort_keys(pattern, kv):
    """Sort keys of int64 patterns: for a 3x3x3 kernel the offsets' bits by distance from the centre, corners first, else
    the pattern; then the rank in the reflected Gray code (the exclusive-or of all higher bits)."""
    if kv == 27:
        dist = [sum(v != 1 for v in (k // 9, k // 3 % 3, k % 3)) for k in range(27)]
        rank = sorted(range(27), key=lambda k: (-dist[k], k))
        key = np.zeros_like(pattern)
        for pos, k in enumerate(rank):
            key |= ((pattern >> k) & 1) << (26 - pos)
    else:
        key = pattern.copy()
    for shift in (1, 2, 4, 8, 16):
        key ^= key >> shift
    return key


def block_order(pattern, kv, mid=-1, known=False):
    lib, n = _lib.load(), len(pattern)
    table = np.where((pattern[None] >> np.arange(kv)[:, None]) & 1, 0, -1).astype(np.int32)
    nbr = torch.as_tensor(table, device=DEV).contiguous()
    mask = torch.as_tensor(pattern.astype(np.int32), device=DEV) if known else None
    elems = lib.pce_osb_order_elems(n)
    order = torch.full((elems,), -7, dtype=torch.int32, device=DEV)
    _lib.check(lib.pce_osb_order(nbr.data_ptr(), mask.data_ptr() if known else None, mid, kv, n, order.data_ptr(), elems,
                                 torch.cuda.current_stream().cuda_stream))
    return order.cpu().numpy()


def test_the_pattern_of_offset_0_alone_has_the_last_key():
    # what the entries behind the last row hold as well: only a stable sort keeps them there
    assert sort_keys(np.array([1], dtype=np.int64), 27)[0] == (1 << 27) - 1


@pytest.mark.parametrize("n", [1, 63, 65, 1000, 8191, 8193, 20011])
@pytest.mark.parametrize("kind", ["offset 0 alone", "few", "any"])
@pytest.mark.parametrize("kv,mid", [(27, -1), (27, 13), (8, -1)])
def test_order_is_the_stable_sort(n, kind, kv, mid):
    rng = np.random.default_rng(n)
    if kind == "offset 0 alone":
        pattern = np.ones(n, dtype=np.int64)
    elif kind == "few":
        pattern = rng.choice(np.array([0, 1, 1, 1, 2, 5], dtype=np.int64), size=n)
    else:
        pattern = rng.integers(0, 1 << kv, size=n)
    full = pattern | (1 << mid if mid >= 0 else 0)
    key = sort_keys(full, kv)
    want = np.concatenate([lo + np.argsort(key[lo:lo + WINDOW], kind="stable") for lo in range(0, n, WINDOW)])
    for known in (False, True):
        order = block_order(pattern, kv, mid, known)
        assert np.array_equal(order[:n], want)
        at = (n + 63) // 64 * 64
        blocks = np.concatenate([full[want], np.zeros(-n % 16, np.int64)]).reshape(-1, 16)
        assert np.array_equal(order[at:at + len(blocks)], np.bitwise_or.reduce(blocks, axis=1))
