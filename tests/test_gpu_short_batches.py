"""Short batches over the binary levels run 16 or 8 lanes per query: batch
sizes around the changes of kernel, over the directory, the query lines with
hints and the select lines, for alphabets with short and long codes and
symbols too rare or too dense for a select line."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = (1, 15, 8192, 8193, 16384, 16385, 32768, 32769)


@pytest.mark.parametrize("dt,sigma", [(np.uint8, 2), (np.uint8, 20), (np.uint8, 256),
                                      (np.uint16, 300), (np.uint32, 7)])
def test_short_batches(gpu, dt, sigma):
    from ecl_wavelet_amd import WaveletTree
    rng = np.random.default_rng(sigma)
    n = 250_007
    sym = np.minimum(rng.geometric(min(0.5, 8 / sigma), n) - 1, sigma - 1)
    sym[: n // 3] = rng.integers(0, sigma, n // 3)
    text = sym.astype(dt)
    order = np.argsort(sym, kind="stable")          # positions by symbol, in order
    first = np.searchsorted(sym[order], np.arange(sigma + 1))
    nth = np.empty(n, np.int64)                     # occurrence number of each position
    nth[order] = np.arange(n) - first[sym[order]]
    wt = WaveletTree(text, np.arange(sigma, dtype=dt))
    for stage in ("directory", "query lines", "select lines"):
        if stage == "query lines":
            wt.buildQueryLines()
        elif stage == "select lines":
            wt.buildSelectLines()
        for m in SIZES:
            at = rng.integers(0, n, m)
            at[0] = n - 1
            assert np.array_equal(wt.access(at.astype(np.uint64)), text[at]), (stage, m)
            # the symbol at a position has nth occurrences before it
            got = wt.rank(wt.make_queries(at, sym[at]))
            assert np.array_equal(got, nth[at].astype(np.uint64)), (stage, m)
            got = wt.select(wt.make_queries(nth[at] + 1, sym[at]))
            assert np.array_equal(got, at.astype(np.uint64)), (stage, m)
        c = np.arange(sigma)
        cnt = np.diff(first)
        assert np.array_equal(wt.rank(wt.make_queries(np.full(sigma, n), c)), cnt.astype(np.uint64))
        assert np.array_equal(wt.select(wt.make_queries(cnt + 1, c)), np.full(sigma, n, np.uint64))
        assert np.array_equal(wt.select(wt.make_queries(np.zeros(sigma), c)),
                              np.full(sigma, n, np.uint64))


@pytest.mark.parametrize("n", [(1 << 24) - 8, 1 << 24, (1 << 29) + 72])
def test_short_batches_over_long_directories(gpu, n):
    """Access and rank over the directory take 16 lanes per query from sizes
    of batch and tree that the trees above do not have: batches around each
    change of kernel, at the tree sizes around each."""
    from ecl_wavelet_amd import WaveletTree
    rng = np.random.default_rng(n)
    period = 1_000_003  # the text repeats a block, so ranks are known
    block = rng.integers(0, 256, period).astype(np.uint8)
    text = np.resize(block, n)
    prefix = np.zeros((256, period + 1), np.uint32)
    for c in range(256):
        prefix[c, 1:] = np.cumsum(block == c)
    wt = WaveletTree(text, np.arange(256, dtype=np.uint8))
    for m in (1, 127, 128, 512, 513, 4096, 4097, 8192, 8193):
        at = rng.integers(0, n, m)
        at[0] = n - 1
        assert np.array_equal(wt.access(at.astype(np.uint64)), text[at]), m
        at[0] = n
        sym = rng.integers(0, 256, m)
        want = at // period * prefix[sym, period].astype(np.int64) + prefix[sym, at % period]
        assert np.array_equal(wt.rank(wt.make_queries(at, sym)), want.astype(np.uint64)), m
