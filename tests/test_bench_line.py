"""bench.py's printed line: the contract's fields as measured and every block's figures, short enough
to survive a capture that keeps the last 8 KB of the output."""
import json

import bench

LONG = 123456.78901234567
KERNEL = "xres_24x24x48_c128_fwd_v1rounds"


def _record():
    """As main() fills it by default: six workloads, two tables of precision variants, six latencies,
    three serving modes of sixteen load points."""
    def measured():
        return {"kernel": KERNEL, "rotate_pairs": 14, "window_ms": [LONG] * 5, "rel_l2_vs_numpy": LONG,
                **{k: LONG for k in ("contract_ms_total", "contract_ms_per_execute", "window_spread",
                                     "ms_per_execute", "transforms_per_s", "us_per_execute_min",
                                     "us_per_execute_max", "achieved_GBs", "roofline_frac")}}
    point = {k: LONG for k in ("rate", "p50_ms", "p99_ms", "mean_ms", "max_ms", "req_per_s", "transforms_per_s")}
    errors = {g: {"rel_l2": LONG, "rel_max": LONG} for g in ("L6", "L8", "L12", "L17")}
    variant = {k: LONG for k in ("us", "GBs", "mfma_tflops", "mfma_util", "rel_l2", "rel_max")}
    precision = {"items": [{"shape": [6, 6, 6], "batch": 65536}] * 4, "bytes_per_launch": 882409472}
    for t in ("one_launch_fft_c64", "one_launch_mfma_bf16x3", "one_launch_mfma_fp16x3"):
        precision[t] = {"kernel": KERNEL, "us": LONG, "GBs": LONG, "mfma_tflops": LONG, "errors": errors}
    for t in ("fft_c64", "mfma_bf16x3", "mfma_fp16x3"):
        precision[t] = {g: dict(variant, kernel=KERNEL, rotate_sets=11) for g in errors}
    replay = {k: LONG for k in ("device_us_per_execute", "round_trip_us_median", "round_trip_us_p99")}
    mode = {"max_rate_req_s": LONG, "at_max": point, "points": [point] * 16,
            "stats": {k: 220000 for k in ("submitted", "completed", "launches", "peak_inflight_bytes")},
            "result_check_rel_l2": {"c128": LONG, "c64": LONG}}
    return {
        "metric": "batched transforms/s + % HBM roofline at L=8/17/36 fp64; serving p99 latency",
        "value": LONG, "unit": "transforms/s", "n_gpus": 1, "steps": 200, "warmup": 10, "ms_per_step": LONG,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic: " + "x" * 60, "config": {"workload": "x" * 90, "kernel": KERNEL, "batch": 1024},
        "gflops_nominal": LONG, "rel_l2_vs_numpy": LONG,
        "roofline": {"achieved": LONG, "peak": 8000.0, "traffic_source": "x" * 160, "frac": LONG},
        "timing": measured(),
        "cpu_baseline": {"value": LONG, "unit": "transforms/s", "cores": 16, "kind": "reference",
                         "sample": "x" * 300, "per_geometry": {f"L{n}": measured() for n in range(8)}},
        "secondary": {f"24x24x48_c128_fwd_b{n}": measured() for n in range(5)},
        "precision_variants": precision,
        "small_batch_latency": {f"{n}x{n}x{n}": {"kernel": KERNEL, "direct": replay, "graph": replay,
                                                 "rel_l2_vs_numpy": LONG} for n in range(6)},
        "host_abi": {"ms_per_execute": LONG, "transforms_per_s": LONG, "rel_l2_vs_numpy": LONG, "note": "x" * 150},
        "serving": {"requests": 20000, "plain": mode, "plain_async": mode, "batched": mode,
                    "throughput_ratio_vs_plain_at_p99_cap": LONG},
    }


def test_line_is_short_and_whole():
    full = _record()
    line = bench.brief(full)
    text = json.dumps(line)
    assert len(json.dumps(full)) > 16000 and len(text) < 7000, len(text)
    assert list(line) == list(full)
    for k in full:
        if k not in bench.BRIEF:
            assert line[k] == full[k], k
    near = float(f"{LONG:.5g}")
    for name in full["secondary"]:
        assert line["secondary"][name]["ms_per_execute"] == near
    assert line["precision_variants"]["mfma_fp16x3"]["L17"]["us"] == near
    assert line["precision_variants"]["one_launch_mfma_bf16x3"]["errors"]["L6"] == {"rel_l2": near}
    assert line["small_batch_latency"]["5x5x5"]["direct"]["device_us_per_execute"] == near
    assert line["serving"]["batched"]["at_max"]["p99_ms"] == near and "points" not in text
    assert full == _record(), "the record is left as it was"


def test_line_without_the_optional_blocks():
    full = {k: None if k in bench.BRIEF else v for k, v in _record().items()}
    assert bench.brief(full) == full
