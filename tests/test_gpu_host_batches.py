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


def test_threads_over_two_trees_and_long_batches(gpu, tree):
    """Callers at once on two trees of different element width, each with
    batches of more chunks than slots (collected by a second thread) between
    batches of one: the staging sets pass from tree to tree."""
    from ecl_wavelet_amd import WaveletTree
    rng = np.random.default_rng(21)
    n = 200_003
    alphabet = (np.arange(300) * 11 + 5).astype(np.uint32)
    sym = rng.integers(0, 300, n)
    wide_text = alphabet[sym]
    wide = WaveletTree(wide_text, alphabet)
    order = np.argsort(sym, kind="stable")
    nth = np.empty(n, np.int64)
    nth[order] = np.arange(n) - np.searchsorted(sym[order], np.arange(300))[sym[order]]

    def check_wide(m, seed):
        r = np.random.default_rng(seed)
        at = r.integers(0, n, m)
        assert np.array_equal(wide.access(at.astype(np.uint64)), wide_text[at])
        got = wide.rank(wide.make_queries(at, wide_text[at]))
        assert np.array_equal(got, nth[at].astype(np.uint64))
        got = wide.select(wide.make_queries(nth[at] + 1, wide_text[at]))
        assert np.array_equal(got, at.astype(np.uint64))

    failed = []

    def work(i):
        try:
            for m in (3 * CHUNK + 7 + i, 300 + i, 5 * CHUNK - i, 1):
                if (i + m) % 2:
                    _check(tree, m, 7 * i + m)
                else:
                    check_wide(m, 7 * i + m)
        except BaseException as e:  # noqa: BLE001 - reported below
            failed.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed[0]


@pytest.mark.parametrize("stage", ["directory", "query lines", "quad", "hex"])
@pytest.mark.parametrize("dt", [np.uint8, np.uint16, np.uint64])
def test_access_past_the_text_gives_zero(gpu, dt, stage):
    """An index past the text has no symbol: its answer is 0, whatever batch
    of another tree the shared staging slots held before.  Batch sizes of
    every access kernel (16, 8, 2 and 1 lanes per query) and of a pipelined
    batch."""
    from ecl_wavelet_amd import WaveletTree
    rng = np.random.default_rng(5)
    n, sigma = 70_003, 16
    alphabet = np.arange(3, 3 + sigma).astype(dt)  # no symbol is 0
    text = alphabet[rng.integers(0, sigma, n)]
    wt = WaveletTree(text, alphabet)
    {"directory": lambda: None, "query lines": wt.buildQueryLines, "quad": wt.buildQuadLines,
     "hex": wt.buildHexLines}[stage]()
    other = WaveletTree(np.full(5000, 1, np.uint8), np.arange(2, dtype=np.uint8))
    for m in (1, 500, 8193, 40_000, 4 * CHUNK + 3):
        # every staged output byte of the other tree's batch is not 0
        q = other.make_queries(np.full(m, 4369), np.full(m, 1))
        assert np.all(other.rank(q) == 4369)
        idx = rng.integers(0, n, m).astype(np.uint64)
        past = rng.random(m) < 0.3
        past[m // 2] = True
        idx[past] = rng.choice(np.array([n, n + 1, 1 << 40, 2**64 - 1], np.uint64), past.sum())
        want = np.where(past, dt(0), text[np.where(past, 0, idx).astype(np.int64)])
        assert np.array_equal(wt.access(idx), want), m


@pytest.mark.parametrize("m", [1, 1000, CHUNK, CHUNK + 1])
def test_refused_batch_launches_nothing(gpu, tree, m):
    """A host batch is refused for device memory before its kernels run,
    whatever its size, and its output is untouched."""
    import ctypes as C

    from ecl_wavelet_amd import Profiler, _lib, set_device_memory_cap
    wt, text, _ = tree
    idx = np.zeros(m, np.uint64)
    q = wt.make_queries(np.ones(m), np.full(m, 3))
    calls = {"access": (idx, np.full(m, 0xA5, np.uint8), 2 * m * 9),
             "rank": (q, np.full(m, 0xA5, np.uint64), 2 * m * 24),
             "select": (q, np.full(m, 0xA5, np.uint64), 2 * m * 24)}
    try:
        Profiler.enable()
        for kind, (src, out, need) in calls.items():
            args = (f"ecl_wavelet_tree_{kind}", wt._h, src.ctypes.data_as(C.c_void_p), m,
                    out.ctypes.data_as(C.c_void_p), 0)
            set_device_memory_cap(0, need - 1)
            Profiler.reset()
            with pytest.raises(_lib.EclError) as e:
                _lib.call(*args)
            assert e.value.status == _lib.ECL_ERROR_OUT_OF_MEMORY_QUERIES
            assert Profiler.get("wt_" + kind)[0] == 0
            assert np.all(out == 0xA5)
            set_device_memory_cap(0, need)  # just enough
            _lib.call(*args)
            assert Profiler.get("wt_" + kind)[0] >= 1
    finally:
        Profiler.enable(False)
        set_device_memory_cap(0, 0)
