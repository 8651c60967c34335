"""Builds of the quad and hex lines at the edges of their workgroups (28672
positions for quad lines, 8192 for hex lines) and of the nodes inside them:
every position's symbol, and the rank of every line's first position."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

QUAD_WG, HEX_WG = 64 * 448, 64 * 128


@pytest.mark.parametrize("layout", ["quad", "hex"])
@pytest.mark.parametrize("sigma", [16, 256])
@pytest.mark.parametrize("n", [1, 447, 448, HEX_WG - 1, HEX_WG, HEX_WG + 1, QUAD_WG - 1, QUAD_WG,
                               QUAD_WG + 1, 5 * QUAD_WG + 33])
def test_layout_workgroup_edges(gpu, n, sigma, layout):
    from ecl_wavelet_amd import WaveletTree
    rng = np.random.default_rng(n + sigma)
    # half uniform, half one symbol: nodes far longer than a workgroup and
    # nodes that start and end inside one
    text = rng.integers(0, sigma, n).astype(np.uint8)
    text[rng.random(n) < 0.5] = sigma // 3
    wt = WaveletTree(text, np.arange(sigma, dtype=np.uint8))
    wt.buildQuadLines() if layout == "quad" else wt.buildHexLines()
    assert np.array_equal(wt.access(np.arange(n, dtype=np.uint64)), text)
    at = np.arange(0, n + 1, 448 if layout == "quad" else 128, dtype=np.uint64)
    for c in (0, sigma // 3, sigma - 1):
        cs = np.full(len(at), c, dtype=np.uint64)
        assert np.array_equal(wt.rank(wt.make_queries(at, cs)), O.scan_rank_batch(text, at, cs))


@pytest.mark.parametrize("sigma,lengths,fits", [(4, [448 * 64 * 300 - 1], 82573088),
                                                (16, [448 * 64 * 150], 86837808),
                                                (256, [1_000_000, 2_345_678], 97918880)])
def test_forest_quad_layouts_memory_limit(gpu, sigma, lengths, fits):
    """Free device memory that these texts' quad layouts have been accepted
    with (lines, tables, 64 MiB to spare and 6 words of scratch per 64 quad
    lines) stays enough for them."""
    from ecl_wavelet_amd import DeviceBuffer, Forest, set_device_memory_cap
    lengths = np.array(lengths, np.uint64)
    starts = np.concatenate([[0], np.cumsum((lengths + 15) // 16 * 16)[:-1]]).astype(np.uint64)
    text = (np.arange(int(starts[-1] + lengths[-1])) * 7 % sigma).astype(np.uint8)
    d = DeviceBuffer.from_array(text)
    forest = Forest(d, starts, lengths, np.full(len(lengths), sigma, np.uint64))
    try:
        set_device_memory_cap(0, fits)
        forest.buildQuadLayouts()
    finally:
        set_device_memory_cap(0, 0)
