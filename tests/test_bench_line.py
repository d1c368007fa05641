"""The line that bench.py prints (CPU only: made from the committed record of a run)."""
import json
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_the_line_fits_a_logs_tail():
    """Whole within six kilobytes (with every configuration's full record it was 24 KB, and a tail of 8 KB did not parse),
    with the keys that readers of the line rely on."""
    import bench
    record = json.load(open(os.path.join(ROOT, "profiles", "bench_line.json")))
    text = bench.brief_line(record)
    assert len(text) < 6000 and "\n" not in text
    line = json.loads(text)
    for key in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline",
                "dtype", "data", "config", "roofline", "kernels_ms"):
        assert key in line
    assert abs(line["value"] - record["value"]) <= 1e-5 * record["value"]
    assert set(line["other_configs"]) == set(record["other_configs"])
