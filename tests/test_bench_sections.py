"""bench.py prints what it has measured when a later section fails: the section
is named, those after it are listed, those before it are kept."""

import sys
from pathlib import Path

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))
import bench  # noqa: E402


def test_a_failed_section_is_named():
    def fails():
        raise RuntimeError("timed out")

    out = {"value": 1.0}
    bench.run_sections(out, [("a", lambda: 7), ("b", fails), ("c", lambda: 8)])
    assert out == {"value": 1.0, "a": 7, "failed": {"section": "b", "error": "timed out", "not_run": ["c"]}}


def test_all_sections_run():
    out = {}
    bench.run_sections(out, [("a", lambda: 7), ("c", lambda: 8)])
    assert out == {"a": 7, "c": 8}
