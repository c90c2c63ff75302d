"""The benchmark's result line: what it keeps of each configuration stays short enough to be read back whole."""
import importlib.util
import json
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_summaries_keep_the_figures_and_stay_short():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    entry = {"metric": "m" * 80, "value": 1234.56789012345, "unit": "GB/s", "steps": 20, "warmup": 1, "ms_per_step": 1.752839724222819,
             "dtype": "c128", "config": {"workload": "w" * 400}, "cases": {str(i): {"ms": i / 7, "gbs": 1e3 / (i + 1)} for i in range(40)},
             "roofline": {"bound": "hbm", "kernel": "k" * 60, "achieved": 5948.554177613117, "peak": 8000.0, "unit": "GB/s",
                          "frac": 0.7435692722016396, "note": "n" * 300},
             "cpu_baseline": {"value": 1.8157535015494137, "unit": "GB/s", "cores": 1, "kind": "port", "sample": "s" * 200},
             "wall_s": 2.8062326}
    got = bench.summary(entry)
    assert got["value"] == 1234.57 and got["roofline"]["frac"] == 0.743569 and got["cpu_baseline"]["cores"] == 1
    assert "cases" not in got and "note" not in got["roofline"]
    assert len(json.dumps({name: got for name, _ in bench.SECONDARY})) < 6000
    assert bench.summary({"metric": "m", "value": 1, "unit": "u", "roofline": None}) == {"metric": "m", "value": 1, "unit": "u"}
