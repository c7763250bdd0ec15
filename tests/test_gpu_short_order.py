"""The block order of clouds of one window that is not full: fewer entries per thread, the same stable sort."""
import numpy as np
import pytest

from tests.test_gpu_block_order import block_order, sort_keys

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1024, 1025, 2047, 6145, 7168, 7169])
@pytest.mark.parametrize("kv,mid", [(27, 13), (8, -1)])
def test_stable_sort_at_the_edges_of_a_threads_entries(n, kv, mid):
    rng = np.random.default_rng(n)
    pattern = (rng.integers(0, 1 << kv, n) & rng.integers(0, 1 << kv, n)).astype(np.int64)
    full = pattern | (1 << mid if mid >= 0 else 0)
    want = np.argsort(sort_keys(full, kv), kind="stable")
    got = block_order(pattern, kv, mid)
    assert np.array_equal(got[:n], want)
    at = (n + 63) // 64 * 64
    blocks = np.bitwise_or.reduce(np.concatenate([full[want], np.zeros(-n % 16, np.int64)]).reshape(-1, 16), axis=1)
    assert np.array_equal(got[at:at + len(blocks)].astype(np.int64), blocks)
