"""The measured work of this library: what its users have it do, from one
small tree to the full-size texts, through the public entry points.

Every output is a whole number (bits, directory entries, positions, counts,
symbols), so results are compared bit for bit and there is no rounding to
bound.  A case is a dict; its "kind" names the path:

  session  a host text: build the tree, then ask it from host memory
  build    a tree over a text that is already on the device
  index    the same, then the query structures, then a first batch over them
  query    device-resident batches of access, rank and select over a tree
  host     host-to-host batches over a tree (copies included)
  binary   the directory of one bit array into the caller's buffers, then
           rank1 and select1 batches
  forest   many texts built together, then one mixed batch over all trees
  serve    mixed requests against the resident trees of a query server
"""
import ctypes as C
import math

import numpy as np
import torch

import ecl_wavelet_amd as E
from ecl_wavelet_amd import _lib
from ecl_wavelet_amd.api import MIXED_DTYPE

BYTE_SIGMAS = (4, 16, 20, 64, 75, 256)
WORD_SIGMAS = (1024, 65536)
LINE = 128  # bytes a random read costs


class TensorBuffer(E.DeviceBuffer):
    """The library's view of a torch tensor's memory."""

    def __init__(self, tensor):
        self.device = 0
        self.nbytes = tensor.numel() * tensor.element_size()
        self.ptr = C.c_void_p(tensor.data_ptr())
        self._owner = tensor


class _Span:
    """Device memory of a library object as a torch tensor (no copy); the
    owner lives as long as the tensor."""

    def __init__(self, owner, address, count, typestr):
        self._owner = owner
        self.__cuda_array_interface__ = {
            "shape": (count,), "typestr": typestr, "data": (address, False),
            "strides": None, "version": 2}


def _span(owner, address, count, typestr):
    if count == 0:
        kind = {"<i2": torch.int16, "<i4": torch.int32, "<i8": torch.int64}[typestr]
        return torch.empty(0, dtype=kind, device="cuda")
    return torch.as_tensor(_Span(owner, address, count, typestr), device="cuda")


# ---------------------------------------------------------------------------
# the cases
def listed():
    return [
        # a first use: a short text from host memory and 10^5 questions of each kind
        dict(name="session_u8_sigma4", kind="session", n=1 << 20, sigma=4, m=100_000),
        # a residue-like alphabet: 20 symbols that are not 0..19, an odd length
        dict(name="build_u8_sigma20", kind="build", n=123_456_789, bytes=1, sigma=20, spread=True,
             zipf=0.0),
        # the full-size byte text
        dict(name="build_u8_sigma256", kind="build", n=6_000_000_000, bytes=1, sigma=256,
             spread=False, zipf=0.0),
        # word tokens: 16 levels, skewed counts, lines for the binary levels
        dict(name="index_u16_zipf", kind="index", n=500_000_000, bytes=2, sigma=65536,
             spread=False, zipf=1.1, layout="lines", m=2_500_000),
        # a byte text made ready for the fastest queries
        dict(name="index_u8_sigma256", kind="index", n=2_000_000_000, bytes=1, sigma=256,
             spread=False, zipf=0.0, layout="quad", m=10_000_000),
        # short batches, where launches count
        dict(name="query_few", kind="query", n=(1 << 26) + 13, bytes=1, sigma=64, spread=False,
             zipf=0.0, layout="quad", m=1000),
        # large batches over the directory alone, and over the quad and hex layouts
        dict(name="query_directory", kind="query", n=6_000_000_000, bytes=1, sigma=256,
             spread=False, zipf=0.0, layout="none", m=10_000_000),
        dict(name="query_layouts", kind="query", n=6_000_000_000, bytes=1, sigma=256,
             spread=False, zipf=0.0, layout="quad", m=10_000_000),
        # the queries of a program that keeps them in host memory
        dict(name="host_batch", kind="host", n=1 << 30, sigma=64, layout="none", m=10_000_000),
        # one long bit array
        dict(name="binary", kind="binary", bits=1 << 34, p=0.5, lines=True, m=10_000_000),
        # thousands of short texts
        dict(name="forest", kind="forest", texts=2000, longest=1 << 21, m=10_000_000,
             layout="none"),
        # a server's resident trees under a burst of requests
        dict(name="serve", kind="serve", trees=8, longest=1 << 26, requests=48,
             largest=200_000, layout="lines"),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(("session", "build", "build", "index", "index", "query", "query", "query",
                       "host", "binary", "forest", "serve"))
    if kind == "session":
        return dict(kind=kind, n=_log(rng, 1 << 10, 1 << 22), sigma=rng.choice(BYTE_SIGMAS),
                    m=_log(rng, 1, 100_000))
    if kind in ("build", "index", "query"):
        width = rng.choice((1, 1, 1, 2))
        sigma = rng.choice(BYTE_SIGMAS if width == 1 else WORD_SIGMAS)
        spread = rng.random() < 0.3 and sigma not in (256, 65536)
        top = 500_000_000 if width == 2 else 2_000_000_000 if kind == "index" else 6_000_000_000
        if kind == "build" and (spread or sigma in (20, 75)):
            top = min(top, 4_000_000_000)  # mapped to codes first
        case = dict(kind=kind, n=_log(rng, 1 << 18, top), bytes=width, sigma=sigma,
                    spread=spread, zipf=1.1 if width == 2 else rng.choice((0.0, 0.0, 1.0)))
        if kind != "build":
            even = sigma in (4, 16, 64, 256, 1024, 65536)
            layouts = ["lines"] + (["quad"] if even else []) + (["none"] if kind == "query" else [])
            case.update(layout=rng.choice(layouts),
                        m=_log(rng, 1000 if kind == "index" else 1,
                               1_000_000 if width == 2 else 10_000_000))
        return case
    if kind == "host":
        return dict(kind=kind, n=_log(rng, 1 << 18, 1 << 30), sigma=rng.choice(BYTE_SIGMAS),
                    layout=rng.choice(("none", "lines")), m=_log(rng, 1, 10_000_000))
    if kind == "binary":
        return dict(kind=kind, bits=_log(rng, 1 << 18, 1 << 34), p=rng.choice((0.5, 0.5, 0.05)),
                    lines=rng.random() < 0.6, m=_log(rng, 1000, 10_000_000))
    if kind == "forest":
        return dict(kind=kind, texts=_log(rng, 20, 2000), longest=_log(rng, 1 << 14, 1 << 21),
                    m=_log(rng, 10_000, 10_000_000), layout=rng.choice(("none", "lines", "quad")))
    return dict(kind=kind, trees=rng.randint(1, 8), longest=_log(rng, 1 << 18, 1 << 26),
                requests=rng.randint(4, 48), largest=_log(rng, 1000, 200_000),
                layout=rng.choice(("none", "lines", "quad")))


# ---------------------------------------------------------------------------
# inputs
_TYPES = {1: (torch.uint8, np.uint8), 2: (torch.int16, np.uint16)}


def _alphabet(sigma, width, spread):
    """0 .. sigma-1, or sigma symbols spread over the type's range."""
    top = 1 << (8 * width)
    a = np.arange(sigma, dtype=np.int64)
    if spread:
        a = a * (top // sigma) + 3
    return a.astype(_TYPES[width][1])


def _text(gen, n, width, sigma, spread, zipf):
    """n symbols on the device: uniform, or Zipf over the alphabet's order."""
    out = torch.empty(n, dtype=_TYPES[width][0], device="cuda")
    symbols = torch.from_numpy(_alphabet(sigma, width, spread).astype(np.int64)).cuda()
    symbols = symbols.to(_TYPES[width][0])
    cdf = None
    if zipf:
        w = torch.arange(1, sigma + 1, dtype=torch.float64, device="cuda").pow(-zipf)
        cdf = torch.cumsum(w, 0) / w.sum()
    step = 1 << (26 if zipf else 29)
    for at in range(0, n, step):
        part = out[at:at + step]
        if cdf is not None:
            u = torch.rand(part.numel(), dtype=torch.float64, device="cuda", generator=gen)
            i = torch.searchsorted(cdf, u).clamp_(max=sigma - 1)
            part.copy_(symbols[i] if spread else i)
        elif width == 1:
            part.random_(0, sigma, generator=gen)
            if spread:
                part.copy_(symbols[part.int()])
        else:
            i = torch.randint(0, sigma, (part.numel(),), device="cuda", generator=gen)
            part.copy_(symbols[i])
    return out


def _tree(text, width, sigma, spread):
    return E.WaveletTree(TensorBuffer(text), _alphabet(sigma, width, spread), 0,
                         dtype=_TYPES[width][1], n=text.numel())


def _add_layout(tree, sigma, layout):
    if layout == "lines":
        tree.buildQueryLines()
        tree.buildSelectLines()
    elif layout == "quad":
        tree.buildQuadSelectLines()
        if (sigma.bit_length() - 1) % 4 == 0:
            tree.buildHexLines()


def _random(gen, m, hi):
    return torch.randint(0, hi, (m,), device="cuda", generator=gen)


def _symbols_at(text, at):
    mask = 0xFF if text.element_size() == 1 else 0xFFFF
    return text[at].to(torch.int64) & mask


def _queries(gen, text, width, m):
    """Positions to access, (position, symbol) to rank, (k, symbol) to select
    with 1 <= k <= the symbol's count; symbols as they occur in the text."""
    n = text.numel()
    access = _random(gen, m, n)
    rank = torch.stack([_random(gen, m, n + 1), _symbols_at(text, _random(gen, m, n))], 1)
    counts = torch.zeros(1 << (8 * width), dtype=torch.int64, device="cuda")
    for at in range(0, n, 1 << 28):
        part = text[at:at + (1 << 28)]
        part = part.to(torch.int32) & ((1 << (8 * width)) - 1)
        counts += torch.bincount(part, minlength=counts.numel())
    sym = _symbols_at(text, _random(gen, m, n))
    u = torch.rand(m, dtype=torch.float64, device="cuda", generator=gen)
    k = 1 + torch.minimum((u * counts[sym]).to(torch.int64), counts[sym] - 1)
    return access, rank.contiguous(), torch.stack([k, sym], 1).contiguous()


def _host_queries(rng, text, m):
    n = text.size
    access = rng.integers(0, n, m).astype(np.uint64)
    rank = E.WaveletTree.make_queries(rng.integers(0, n + 1, m), text[rng.integers(0, n, m)])
    counts = np.bincount(text, minlength=256)
    sym = text[rng.integers(0, n, m)]
    k = 1 + np.minimum((rng.random(m) * counts[sym]).astype(np.int64), counts[sym] - 1)
    return access, rank, E.WaveletTree.make_queries(k, sym)


def _mixed(rng, n, sigma, m):
    """A request's queries: every kind, uniform arguments."""
    q = np.zeros(m, MIXED_DTYPE)
    q["kind"] = rng.integers(0, 3, m)
    q["symbol"] = rng.integers(0, sigma, m)
    q["arg"] = np.where(q["kind"] == 2, 1 + rng.integers(0, max(n // sigma, 1), m),
                        rng.integers(0, n, m))
    return q


def _query_buffers(m, width):
    return {"access": torch.zeros(m, dtype=_TYPES[width][0], device="cuda"),
            "rank": torch.zeros(m, dtype=torch.int64, device="cuda"),
            "select": torch.zeros(m, dtype=torch.int64, device="cuda")}


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = dict(case)
    if kind == "session":
        text = rng.integers(0, case["sigma"], case["n"], dtype=np.uint8)
        s["text"] = text
        s["queries"] = _host_queries(rng, text, case["m"])
    elif kind in ("build", "index", "query"):
        width = case["bytes"]
        text = _text(gen, case["n"], width, case["sigma"], case["spread"], case["zipf"])
        if kind != "build":
            s["queries"] = _queries(gen, text, width, case["m"])
            s["out"] = _query_buffers(case["m"], width)
        if kind == "query":
            s["tree"] = _tree(text, width, case["sigma"], case["spread"])
            _add_layout(s["tree"], case["sigma"], case["layout"])
        else:
            s["text"] = text
            s["room"] = {}
    elif kind == "host":
        text = _text(gen, case["n"], 1, case["sigma"], False, 0.0)
        s["tree"] = _tree(text, 1, case["sigma"], False)
        _add_layout(s["tree"], case["sigma"], case["layout"])
        a, r, k = (t.cpu().numpy() for t in _queries(gen, text, 1, case["m"]))
        s["queries"] = (a.astype(np.uint64), E.WaveletTree.make_queries(r[:, 0], r[:, 1]),
                        E.WaveletTree.make_queries(k[:, 0], k[:, 1]))
    elif kind == "binary":
        _prepare_binary(s, case, gen, seed)
    elif kind == "forest":
        _prepare_forest(s, case, gen, rng)
    else:
        _prepare_serve(s, case, gen, rng)
    return s


def _prepare_binary(s, case, gen, seed):
    bits, m = case["bits"], case["m"]
    threshold = min(int(case["p"] * 2.0 ** 64), 2 ** 64 - 1)
    array = E.BitArray([bits])
    array.fillRandom(0, seed, threshold)
    rs = E.RankSelect(array)
    if case["lines"]:
        rs.buildQueryLines()
        rs.buildSelectLines()
    words = C.c_void_p()
    _lib.call("ecl_bit_array_device_pointers", rs.bit_array_._h, C.byref(words), None, None)
    l1, l2, samples = C.c_uint64(), C.c_uint64(), C.c_uint64()
    _lib.call("ecl_rank_select_directory_sizes", bits, C.byref(l1), C.byref(l2),
              C.byref(samples))
    total = rs.getTotalNumVals(0, 1)
    s.update(
        rs=rs, words=words,
        l1=torch.zeros(l1.value, dtype=torch.int64, device="cuda"),
        l2=torch.zeros(l2.value, dtype=torch.int16, device="cuda"),
        samples=torch.zeros(max(samples.value, 1), dtype=torch.int64, device="cuda"),
        ones=torch.zeros(1, dtype=torch.int64, device="cuda"),
        positions=_random(gen, m, bits + 1), kth=1 + _random(gen, m, total),
        rank=torch.zeros(m, dtype=torch.int64, device="cuda"),
        select=torch.zeros(m, dtype=torch.int64, device="cuda"))


def _prepare_forest(s, case, gen, rng):
    count, longest = case["texts"], case["longest"]
    sigmas = rng.choice([4, 20, 64, 256], count).astype(np.uint64)
    lengths = np.exp(rng.uniform(math.log(1 << 10), math.log(longest), count)).astype(np.uint64)
    lengths[0] = longest
    padded = (lengths + np.uint64(15)) // np.uint64(16) * np.uint64(16)
    starts = np.concatenate([[0], np.cumsum(padded)[:-1]]).astype(np.uint64)
    # byte j of a text over sigma symbols: a random byte times sigma / 256,
    # and the last, few symbols of the 20 as likely as the others within 1/13
    text = torch.empty(int(padded.sum()), dtype=torch.uint8, device="cuda")
    text.random_(0, 256, generator=gen)
    per_byte = torch.repeat_interleave(torch.from_numpy(sigmas.astype(np.int16)).cuda(),
                                       torch.from_numpy(padded.astype(np.int64)).cuda())
    for at in range(0, text.numel(), 1 << 28):
        part = text[at:at + (1 << 28)]
        part.copy_((part.to(torch.int32) * per_byte[at:at + (1 << 28)]) >> 8)
    del per_byte
    m = case["m"]
    # queries in the trees' order, as many per tree as its share of the batch
    tree = np.sort(rng.integers(0, count, m)).astype(np.uint64)
    kind = rng.integers(0, 3, m).astype(np.uint64)
    n, sg = lengths[tree], sigmas[tree]
    sym = (rng.random(m) * sg).astype(np.uint64)
    span = np.where(kind == 2, np.maximum(n // sg, 1), n)
    arg = (rng.random(m) * span).astype(np.uint64) + (kind == 2)
    q = np.zeros(m, E.FOREST_QUERY_DTYPE)
    q["arg"], q["symbol"], q["kind"], q["tree"] = arg, sym, kind, tree
    s.update(text=text, starts=starts, lengths=lengths, sigmas=sigmas,
             queries=torch.from_numpy(q.view(np.uint8)).cuda(),
             out=torch.zeros(m, dtype=torch.int64, device="cuda"))


def _prepare_serve(s, case, gen, rng):
    level = {"none": 0, "lines": 2, "quad": 3}[case["layout"]]
    server = E.Server(max_batch=1 << 20, max_inflight=3, query_lines=level)
    shape = np.random.default_rng(case["requests"])  # sizes belong to the case
    trees = []
    for _ in range(case["trees"]):
        sigma = int(shape.choice([4, 20, 64, 256]))
        n = int(math.exp(shape.uniform(math.log(1 << 16), math.log(case["longest"]))))
        text = _text(gen, n, 1, sigma, False, 0.0)
        torch.cuda.synchronize()
        trees.append((server.addTree(TensorBuffer(text), sigma, n), n, sigma))
    requests = []
    for _ in range(case["requests"]):
        tree, n, sigma = trees[int(shape.integers(len(trees)))]
        m = int(math.exp(shape.uniform(0.0, math.log(case["largest"]))))
        requests.append((tree, _mixed(rng, n, sigma, m)))
    s.update(server=server, requests=requests)


# ---------------------------------------------------------------------------
# one pass
def _device_queries(s, tree):
    """The three batches, on the caller's (default) stream."""
    m, out = s["m"], s["out"]
    access, rank, select = s["queries"]
    tree.accessDevice(TensorBuffer(access), m, TensorBuffer(out["access"]))
    tree.rankDevice(TensorBuffer(rank), m, TensorBuffer(out["rank"]))
    tree.selectDevice(TensorBuffer(select), m, TensorBuffer(out["select"]))
    return dict(out)


def _fixed(s, name, got, capacity):
    """`got` in a buffer of the state with room for `capacity` values: what
    is as long as the text's counts make it comes back in a fixed shape."""
    room = s["room"].get(name)
    if room is None:
        room = s["room"][name] = torch.zeros(capacity, dtype=got.dtype, device="cuda")
    room[:got.numel()].copy_(got)
    return room


def _tree_arrays(s, tree):
    """Everything the build made: the level bits, the directory of every
    level, its select samples, the symbol counts and the node ranks."""
    n = s["n"]
    rs = tree.rank_select_
    bits = rs.bit_array_
    words = C.c_void_p()
    _lib.call("ecl_bit_array_device_pointers", bits._h, C.byref(words), None, None)
    d = _lib.RankSelectDevice()
    _lib.call("ecl_rank_select_device_pointers", rs._h, C.byref(d))
    out = {"counts": tree.getCounts().astype(np.int64),
           "node_ranks": tree.nodeRanks()[0].astype(np.int64)}
    l1 = l2 = slot = 0
    levels = bits.numArrays()
    for i in range(levels):
        info = rs.info(i)
        level = _span(tree, words.value + 4 * info.offset_words, (info.size_bits + 31) // 32,
                      "<i4")
        if info.size_bits != n:
            level = _fixed(s, "level%d" % i, level, (n + 31) // 32)
        out["level%d" % i] = level
        slots = info.size_bits // 4096
        ones = _span(tree, d.samples + 8 * slot, info.num_samples_1, "<i8")
        zeros = _span(tree, d.samples + 8 * (slot + slots - info.num_samples_0),
                      info.num_samples_0, "<i8")
        out["ones%d" % i] = _fixed(s, "ones%d" % i, ones, n // 4096)
        out["zeros%d" % i] = _fixed(s, "zeros%d" % i, zeros, n // 4096)
        slot += slots
        l1 += info.num_l1_blocks
        l2 += info.num_l2_blocks
    out["l1"] = _span(tree, d.l1, l1, "<i8")
    out["l2"] = _span(tree, d.l2, l2, "<i2")
    if s["sigma"] & (s["sigma"] - 1):
        out["l1"] = _fixed(s, "l1", out["l1"], levels * ((n + 65535) // 65536))
        out["l2"] = _fixed(s, "l2", out["l2"], levels * ((n + 511) // 512))
    return out


def run(s):
    kind = s["kind"]
    if kind == "session":
        tree = E.WaveletTree(s["text"], _alphabet(s["sigma"], 1, False))
        access, rank, select = s["queries"]
        return {"counts": tree.getCounts().astype(np.int64), "access": tree.access(access),
                "rank": tree.rank(rank).astype(np.int64),
                "select": tree.select(select).astype(np.int64)}
    if kind == "build":
        return _tree_arrays(s, _tree(s["text"], s["bytes"], s["sigma"], s["spread"]))
    if kind == "index":
        tree = _tree(s["text"], s["bytes"], s["sigma"], s["spread"])
        _add_layout(tree, s["sigma"], s["layout"])
        return _device_queries(s, tree)
    if kind == "query":
        return _device_queries(s, s["tree"])
    if kind == "host":
        access, rank, select = s["queries"]
        tree = s["tree"]
        return {"access": tree.access(access), "rank": tree.rank(rank).view(np.int64),
                "select": tree.select(select).view(np.int64)}
    if kind == "binary":
        _lib.call("ecl_rank_select_build_directory_noalloc", 0, s["words"], s["bits"],
                  s["l1"].data_ptr(), s["l2"].data_ptr(), s["samples"].data_ptr(),
                  s["ones"].data_ptr(), None)
        rs, m = s["rs"], s["m"]
        rs.rankDevice(0, TensorBuffer(s["positions"]), m, TensorBuffer(s["rank"]))
        rs.selectDevice(0, TensorBuffer(s["kth"]), m, TensorBuffer(s["select"]))
        return {k: s[k] for k in ("l1", "l2", "samples", "ones", "rank", "select")}
    if kind == "forest":
        forest = E.Forest(TensorBuffer(s["text"]), s["starts"], s["lengths"], s["sigmas"])
        if s["layout"] != "none":
            forest.buildQueryLines()
            forest.buildSelectLines()
        if s["layout"] == "quad":
            forest.buildQuadLayouts()
        forest.queryDevice(TensorBuffer(s["queries"]), s["m"], TensorBuffer(s["out"]))
        return s["out"]
    ids = [s["server"].submit(tree, q) for tree, q in s["requests"]]
    return [s["server"].wait(i)[0].view(np.int64) for i in ids]


# ---------------------------------------------------------------------------
def _tree_bytes(n, sigma):
    """Level bits, directory (2 bytes per 512 bits, 8 per 65536) and select
    samples (8 bytes per 4096 bits) of ceil(log2 sigma) levels."""
    return (sigma - 1).bit_length() * (n / 8 + n / 256 + n / 8192 + n / 512)


def work(case):
    """Inputs read once, outputs written once; a query reads at least one
    random line of the tree.  Integer work only: no floating operations."""
    kind = case["kind"]
    if kind in ("session", "build", "index", "query", "host"):
        n, width = case["n"], case.get("bytes", 1)
        built = n * width + _tree_bytes(n, case["sigma"])
        asked = case.get("m", 0) * (8 + width + 2 * 24 + 3 * LINE)
        moved = {"build": built, "query": asked, "host": asked}.get(kind, built + asked)
    elif kind == "binary":
        bits = case["bits"]
        moved = bits / 8 + bits / 256 + bits / 8192 + bits / 512 + case["m"] * 2 * (16 + LINE)
    elif kind == "forest":
        # lengths are log-uniform over [2^10, longest]
        lo, hi = 1 << 10, case["longest"]
        n = case["texts"] * (hi - lo) / math.log(hi / lo)
        moved = n + _tree_bytes(n, 36) + case["m"] * (24 + 8 + LINE)
    else:
        mean = case["largest"] / max(math.log(case["largest"]), 1.0)
        moved = case["requests"] * mean * (16 + 8 + LINE)
    return {"bytes": moved, "flops": 0}


def tolerance(case):
    return "exact"
