"""Construction at the edges of its tiles: text lengths around whole chunks
and tiles, and symbol counts that put the ends of many, few, empty and tiny
groups inside the 16-byte chunks of a level.  Every level's bits, count and
node rank equals the oracle's tree over the same text."""
import numpy as np
import pytest

from test_gpu_wavelet_tree import _check_structure_vs_oracle

pytestmark = pytest.mark.gpu


def _text(kind, n, sigma, rng):
    if kind == "uniform":
        return rng.integers(0, sigma, n)
    if kind == "rare":  # one symbol takes nearly everything, the others a few places
        t = np.full(n, sigma // 2)
        at = rng.integers(0, n, min(n, 3 * sigma))
        t[at] = rng.integers(0, sigma, at.size)
        return t
    if kind == "sorted":  # whole tiles of one symbol
        return np.sort(rng.integers(0, sigma, n))
    return np.arange(n) * 7 % sigma  # "cycle": every group the same length


@pytest.mark.parametrize("kind", ["uniform", "rare", "sorted", "cycle"])
@pytest.mark.parametrize("dt,sigma", [(np.uint8, 2), (np.uint8, 4), (np.uint8, 20),
                                      (np.uint8, 129), (np.uint8, 256), (np.uint16, 300),
                                      (np.uint16, 1024), (np.uint32, 70000)])
def test_tile_and_chunk_edges(gpu, dt, sigma, kind):
    from ecl_wavelet_amd import WaveletTree
    rng = np.random.default_rng(sigma)
    tile = 32768 // np.dtype(dt).itemsize
    for n in (1, 15, 16, 17, 33, tile - 1, tile, tile + 1, 2 * tile + 17):
        if sigma > 65536 and n > tile:
            continue
        text = _text(kind, n, sigma, rng).astype(dt)
        wt = WaveletTree(text, np.arange(sigma, dtype=dt))
        _check_structure_vs_oracle(wt, text, sigma)


@pytest.mark.parametrize("kind", ["uniform", "rare", "sorted"])
@pytest.mark.parametrize("dt,sigma", [(np.uint16, 65536), (np.uint32, 70000), (np.uint32, 1 << 17),
                                      (np.uint64, 300), (np.uint64, 70000)])
def test_later_passes_over_many_tiles(gpu, dt, sigma, kind):
    """Two- and three-pass builds whose nodes span several tiles of every
    pass, with codes that get narrower from pass to pass (4, 2, 1 bytes), and
    8-byte alphabets."""
    from ecl_wavelet_amd import WaveletTree
    rng = np.random.default_rng(sigma)
    for n in (4 * 32768 - 1, 6 * 32768 + 77):
        text = _text(kind, n, sigma, rng).astype(dt)
        wt = WaveletTree(text, np.arange(sigma, dtype=dt))
        _check_structure_vs_oracle(wt, text, sigma)


@pytest.mark.parametrize("span", [1, 2, 4])
def test_span_edges(gpu, span):
    """Text lengths around whole spans of tiles, where a workgroup's carried
    words meet the next one's."""
    from ecl_wavelet_amd import WaveletTree, set_build_span
    rng = np.random.default_rng(span)
    set_build_span(span)
    try:
        for dt, sigma in ((np.uint8, 4), (np.uint8, 20), (np.uint8, 256), (np.uint16, 1024)):
            tile = 32768 // np.dtype(dt).itemsize
            for n in (span * tile - 1, span * tile, span * tile + 1, 2 * span * tile + 31):
                for kind in ("uniform", "rare"):
                    text = _text(kind, n, sigma, rng).astype(dt)
                    wt = WaveletTree(text, np.arange(sigma, dtype=dt))
                    _check_structure_vs_oracle(wt, text, sigma)
    finally:
        set_build_span(0)


@pytest.mark.parametrize("sigma", [4, 20, 75, 200])
def test_mapped_bytes_edges(gpu, sigma):
    """Byte alphabets that are not 0..sigma-1 are mapped by table while the
    tiles are counted: whole and partial chunks, and batches of four chunks."""
    from ecl_wavelet_amd import WaveletTree
    rng = np.random.default_rng(sigma)
    alphabet = np.sort(rng.permutation(256)[:sigma]).astype(np.uint8)
    for n in (1, 15, 17, 8191, 8192, 8193, 32768 + 16 * 512 * 3 + 5):
        sym = rng.integers(0, sigma, n)
        wt = WaveletTree(alphabet[sym], alphabet)
        _check_structure_vs_oracle(wt, sym.astype(np.uint8), sigma)
