"""Host-issued batches: sizes around the chunk of 2^19 queries and the three
slots, and calls from several threads on one tree, each with its own
staging buffers."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHUNK = 1 << 19


@pytest.fixture(scope="module")
def tree():
    from ecl_wavelet_amd import WaveletTree
    rng = np.random.default_rng(11)
    text = rng.integers(0, 20, 300_001).astype(np.uint8)
    text[::7] = 3
    prefix = np.zeros((20, len(text) + 1), np.uint64)
    for c in range(20):
        prefix[c, 1:] = np.cumsum(text == c)
    return WaveletTree(text, np.arange(20, dtype=np.uint8)), text, prefix


def _check(tree, m, seed):
    wt, text, prefix = tree
    rng = np.random.default_rng(seed)
    n = len(text)
    idx = rng.integers(0, n, m).astype(np.uint64)
    assert np.array_equal(wt.access(idx), text[idx])
    pos = rng.integers(0, n + 1, m)
    sym = rng.integers(0, 20, m)
    assert np.array_equal(wt.rank(wt.make_queries(pos, sym)), prefix[sym, pos])
    # the occurrence at a position is the (rank + 1)-th of its symbol
    at = rng.integers(0, n, m)
    k = prefix[text[at], at] + np.uint64(1)
    assert np.array_equal(wt.select(wt.make_queries(k, text[at])), at.astype(np.uint64))


@pytest.mark.parametrize("m", [1, 2, 63, CHUNK - 1, CHUNK, CHUNK + 1, 3 * CHUNK, 3 * CHUNK + 1,
                               5 * CHUNK + 77])
def test_batch_sizes(gpu, tree, m):
    _check(tree, m, m)


def test_threads_and_released_buffers(gpu, tree):
    from ecl_wavelet_amd import release_cached_memory
    failed = []

    def work(i):
        try:
            for m in (5, 1000 + i, CHUNK // 2 + i):
                _check(tree, m, 100 * i + 1)
        except BaseException as e:  # noqa: BLE001 - reported below
            failed.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed[0]
    release_cached_memory()
    _check(tree, 1000, 5)
