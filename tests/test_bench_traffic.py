"""bench.py's figures that belong to one state of a kernel: they go when the kernel's sources change."""
import json
import os

import bench
from quamba_amd import build


def test_a_fingerprint_is_of_the_code_alone(tmp_path):
    a, b = tmp_path / "a.hip", tmp_path / "b.hip"
    a.write_text("int f(int x) { return x; }  // the identity\n/* of\nintegers */\n")
    b.write_text("// the identity\nint f(int x)\n{\n    return x;\n}\n")
    of = lambda *names: bench.source_fingerprint(names, str(tmp_path))
    assert of("a.hip") == of("b.hip")
    b.write_text("int f(int x) { return x + 1; }")
    assert of("a.hip") != of("b.hip") and of("a.hip", "b.hip") != of("a.hip")


def test_traffic_of_changed_kernels_is_not_replayed(tmp_path):
    path = tmp_path / "traffic.json"
    entry = dict(bytes=7, kernel_symbols=["gemm_w8a8_kernel"], sources=["gemm_w8a8.hip"], fingerprint=bench.source_fingerprint(["gemm_w8a8.hip"]))
    gone, changed = dict(entry, kernel_symbols=["no_such_kernel"]), dict(entry, fingerprint="0" * 16)
    path.write_text(json.dumps(dict(head="abc", entries=dict(entry=entry, gone=gone, changed=changed))))
    assert bench.load_traffic(str(path)) == ({"entry": 7}, "abc")
    assert bench.load_traffic(str(tmp_path / "none.json")) == ({}, None)


def test_the_committed_figures_name_existing_sources():
    doc = json.load(open(os.path.join(bench.ROOT, "profiles", "traffic.json")))
    assert set(doc["entries"]) >= {"in_proj_w8a8_gemm", "causal_conv1d_fwd", "sscan_fwd", "out_proj_w8a8_gemm"}
    for entry in doc["entries"].values():
        assert entry["sources"] and all(os.path.exists(os.path.join(build.CSRC, s)) for s in entry["sources"])
