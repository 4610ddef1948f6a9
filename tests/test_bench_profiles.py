"""bench.py reports counter figures from profiles/ only while the kernels they were read from are the ones in the tree."""
import json
import os
import shutil

import pytest

import bench
import build

CSRC = os.path.join(bench.ROOT, "realtime-vla_amd", "csrc")


@pytest.mark.parametrize("sources", [bench.GEGLU_SOURCES, bench.FLOW_SOURCES], ids=["geglu", "flow"])
def test_figures_of_another_kernel_are_not_reported(sources, tmp_path, monkeypatch):
    """Same version, same variant name, other code: a kernel whose version was not raised with it."""
    for name in sources:
        shutil.copy(os.path.join(CSRC, name), tmp_path)
    recorded = bench.kernel_digest(sources, tmp_path)
    assert recorded == bench.kernel_digest(sources)
    facts = {"kernel": "k", "workload": "w", "rtvla_version": 12, "digest": recorded, "traffic_bytes_per_launch": 5}
    (tmp_path / "summary.md").write_text("# text\n\nfacts: %s\n" % json.dumps(facts))
    monkeypatch.setattr(bench, "PROFILES", str(tmp_path))
    reported = lambda version=12, kernel="k": bench.profiled_traffic("summary.md", kernel, "w", version, bench.kernel_digest(sources, tmp_path))
    assert reported() == 5 and reported(version=13) is None and reported(kernel="other") is None
    for name in sources:
        whole = (tmp_path / name).read_text()
        (tmp_path / name).write_text("// a comment\n" + whole.replace("\n", "\n\n", 3) + "/* another\n one */\n")
        assert reported() == 5
        (tmp_path / name).write_text(whole + "\nint one_more;\n")
        assert reported() is None
        (tmp_path / name).write_text(whole)
    monkeypatch.setitem(build.EXTRA, sources[0], ["-O1"])
    assert reported() is None


def test_code_inside_strings_is_code(tmp_path):
    digests = []
    for text in ('const char* s = "// one"; int a;', 'const char* s = "// two"; int a;', 'const char* s = "// one"; int b;', 'const char* s = "// one"; /* b */ int a; // c'):
        (tmp_path / "x.hip").write_text(text)
        digests.append(bench.kernel_digest(("x.hip",), tmp_path))
    assert len(set(digests[:3])) == 3 and digests[3] == digests[0]


def test_a_summary_without_a_digest_is_refused(tmp_path, monkeypatch):
    (tmp_path / "summary.md").write_text('facts: {"kernel": "k", "workload": "w", "rtvla_version": 11, "traffic_bytes_per_launch": 5}\n')
    monkeypatch.setattr(bench, "PROFILES", str(tmp_path))
    assert bench.profiled_traffic("summary.md", "k", "w", 11, bench.kernel_digest(bench.FLOW_SOURCES)) is None
