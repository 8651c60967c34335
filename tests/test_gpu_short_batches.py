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
