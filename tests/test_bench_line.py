"""The benchmark's result line: one line of JSON short enough for a reader
that keeps only the last 8000 characters of the output, with the headline
fields as they were measured.  Every field below has the length it has in a
full run.  No GPU."""
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402

X = 13515277012.619907 / 7


def _nums(name, n):
    """n fields, rates and times in turn."""
    return {f"{name}_{i}": X if i % 2 else X / 1e8 for i in range(n)}


def _full_result():
    row = {"rate_req_s": 100000.0, "seconds": 0.2, "requests": 20140, "queries": 1475782000,
           "batches": 2307, "p50_ms": 122.909916, "p99_ms": 1231.944345, "queries_per_s": X}
    matched = {"p99_ms": 300.0, "served_qps": X, "plain_qps": X, "ratio": 4.936522491772512}
    layout = {"admit_ms": 1796.3463134765625, "hbm_used_gb": 251.578548224,
              "trees_admitted": 64, "symbols_admitted": 36003186697, "served": [row] * 8,
              "plain": [row] * 8, "matched_p99": [matched] * 7}
    text = "a description of a section's workload, about as long as the longest of them " * 2
    res = {"metric": bench.METRIC, "value": X * 7, "unit": "queries/s", "n_gpus": 1, "steps": 20,
           "warmup": 5, "ms_per_step": 101.31734478473663, "higher_is_better": True,
           "scaling": "weak", "vs_baseline": None, "dtype": "u8", "data": "synthetic",
           "config": {"workload": text * 2, "n": 6 * 10**9, "sigma": 256,
                      "queries_per_kind": 10**7, "levels": 8}}
    res.update(_nums("a_rate_or_time_of_it", 20))
    for name, n in (("plain_directory", 5), ("query_lines_layout", 5), ("quad_lines_layout", 3)):
        res[name] = _nums("a_kind_qps", n)
    res["build_kernels_ms"] = {f"kernel_{i}": {"launches": 12, "ms": X / 1e9} for i in range(5)}
    res["query_roofline"] = {
        "bound": "random dependent 128-byte line reads", "unit": "lines/s", "peak": X,
        "peak_source": text, "peak_half_chains": X, "peak_half_chains_source": text,
        **{k: {"layout": "quad select lines", "lines_per_query": 4, "achieved": X, "peak": X,
               "frac": 0.9139312181435535} for k in ("access", "rank", "select")}}
    res["roofline"] = {"kernel": text[:50], "bound": "hbm", "bytes_basis": text[:100],
                       "traffic_source": "profiles/wt_pass_counters_u8_n6e9_sigma256.txt",
                       "limiter": text[:100], **_nums("number", 8)}
    res["host_to_host"] = {"config": text, **_nums("host_num", 8)}
    res["batched"] = {"config": text, **_nums("a_batched_rate_or_ms", 20)}
    res["binary_rank_select"] = {"config": text, "bits": 1 << 34, "queries": 10**8, **{
        p: _nums("rate_or_time_of", 11) for p in ("p=0.5", "p=0.05")}}
    res["serving"] = {"config": text, "p99_targets_ms": [2.0] * 7,
                      **{k: json.loads(json.dumps(layout)) for k in ("directory", "lines", "quad")}}
    res["full_size_sweep"] = [{"dtype": "uint16", "distribution": "uniform",
                               **_nums("a_sweep_rate_or_time", 17)} for _ in range(4)]
    res["cpu_baseline"] = {"value": 222.5646964288935, "unit": "queries/s", "cores": 16,
                           "kind": "port", "sample": text[:170], "variant_b": {
                               "kind": text[:70], **_nums("a_cpu_number", 7)},
                           **_nums("a_cpu_number", 7)}
    return res


def test_result_line_is_short_and_whole():
    res = _full_result()
    was = json.dumps(res)
    line = bench.result_line(res)
    assert json.dumps(res) == was  # the result itself is not cut
    assert len(was) > 16000 and len(line.encode()) <= bench.LINE_MAX and "\n" not in line
    out = json.loads(line)
    for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step",
              "higher_is_better", "scaling", "vs_baseline", "dtype", "data", "config"):
        assert out[k] == res[k]
    assert set(out) == set(res)
    assert out["cpu_baseline"]["value"] == 222.6
    assert out["serving"]["quad"]["served"][0][2] == 1232.0
    assert out["serving"]["directory"]["matched_p99"][0] == [300.0, 1931000000, 1931000000]
    cols = out["full_size_sweep"]["columns"]
    assert all(len(r) == len(cols) for r in out["full_size_sweep"]["rows"])
