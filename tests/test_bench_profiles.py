"""bench.py reports a committed profile's counters only for the kernels that
it was taken on: the profile names the library sources and their hash."""
import importlib
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
bench = importlib.import_module("bench")


def test_profiles_of_other_sources_are_not_used(tmp_path, monkeypatch):
    for name in os.listdir(os.path.join(ROOT, "profiles")):
        if name.endswith(".json"):
            src = json.load(open(os.path.join(ROOT, "profiles", name)))["sources"]
            assert len(src["sha16"]) == 16
            bench.sources_sha16(src["files"])  # they exist
    csrc = tmp_path / "2023_render_engine_amd" / "csrc"
    csrc.mkdir(parents=True)
    (tmp_path / "profiles").mkdir()
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    (csrc / "k.hip").write_text("int a = 1;  // one\n")
    sha = bench.sources_sha16(["k.hip"])
    p = tmp_path / "profiles" / "p.json"
    p.write_text(json.dumps({"sources": {"files": ["k.hip"], "sha16": sha}, "x": 3}))
    assert bench.load_profile("p.json")["x"] == 3
    (csrc / "k.hip").write_text("/* two */ int a\n  = 1;\n")
    assert bench.load_profile("p.json")["x"] == 3
    (csrc / "k.hip").write_text("int a = 2;\n")
    assert bench.load_profile("p.json") is None
    p.write_text(json.dumps({"x": 3}))
    assert bench.load_profile("p.json") is None and bench.load_profile("none.json") is None
