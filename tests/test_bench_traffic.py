"""bench.py's roofline: a committed counter profile counts only for the graph
and the kernel sources it was measured on."""

import json
from types import SimpleNamespace

import bench


def _root(tmp_path, monkeypatch, **profile):
    csrc = tmp_path / "openkhuzdulgraph_amd" / "csrc"
    csrc.mkdir(parents=True, exist_ok=True)
    for name in ("kz_clique.hip", "kz_core.h", "kz_stream.h", "kz_kernels.h"):
        (csrc / name).write_text(f"// {name}\nint x;\n")
    monkeypatch.setattr(bench, "ROOT", tmp_path)
    (tmp_path / "profiles").mkdir(exist_ok=True)
    entry = dict(bytes_per_launch=1000, csr_digest="ab", kernel_sources=bench.kernel_sources_sha(), **profile)
    (tmp_path / "profiles" / "rmat24_k4_persistent_traffic.json").write_text(json.dumps(entry))
    return csrc


def test_traffic_of_the_same_graph_and_sources(tmp_path, monkeypatch):
    csrc = _root(tmp_path, monkeypatch, l2_hit_rate=0.2)
    args = SimpleNamespace(scale=24, k=4)
    assert bench.committed_traffic(args, "ab")["bytes_per_launch"] == 1000
    assert bench.committed_traffic(args, "cd") == {}  # another seed or edge factor
    assert bench.committed_traffic(SimpleNamespace(scale=22, k=4), "ab") == {}
    (csrc / "kz_core.h").write_text("// another comment\n  int x;\n")
    assert bench.committed_traffic(args, "ab") != {}
    (csrc / "kz_core.h").write_text("int y;\n")
    assert bench.committed_traffic(args, "ab") == {}
