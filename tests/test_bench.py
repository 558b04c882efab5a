"""bench.py's report where the reference build is not present."""
import importlib.util
import os

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_report_without_the_reference_build(monkeypatch):
    """no CPU baseline, its reason named, and no failure"""
    from oracle import ref
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    monkeypatch.setattr(ref, "available", lambda *a, **k: False)

    class Context:
        def write_tables(self, d):
            raise AssertionError("no tables are needed")
    out = bench.cpu_report(Context(), 1.0, 64, 0, 1)
    assert out["cpu_baseline"] is None and "reference" in out["cpu_baseline_missing"]
    assert "gpu_over_cpu" not in out
