"""The benchmark prints the counter profile of its traversal kernel only beside that kernel's time."""
import json
import os

import bench


def test_fingerprint_follows_code_and_configuration():
    table = {"closest": {"block": 64, "steps": 32, "ms": 5.0, "mrays_s": 1.0}}
    a = bench.kernel_fingerprint(["int a = 1; // one\n/* two\nlines */ int b;\n"], table)
    assert a == bench.kernel_fingerprint(["int a = 1;\n\n  int b; // other words\n"], table)
    assert a == bench.kernel_fingerprint(["int a = 1; int b;"], {"closest": dict(table["closest"], ms=7.0)})
    assert a != bench.kernel_fingerprint(["int a = 2; int b;"], table)
    assert a != bench.kernel_fingerprint(["int a = 1; int b;"], {"closest": dict(table["closest"], steps=16)})


def test_profiles_of_other_kernels_are_not_printed(tmp_path):
    path = tmp_path / "traffic.json"
    assert bench.traffic_profile("x", str(path)) == (None, None, None)
    path.write_text(json.dumps({"hbm_bytes_per_launch": 3, "l2_hit_rate": 0.5, "sq_counters": {"SQ_INSTS_VALU": 7}}))
    assert bench.traffic_profile("x", str(path)) == (None, None, None)  # of no stated kernel
    p = json.loads(path.read_text())
    path.write_text(json.dumps(dict(p, kernel_fingerprint="x")))
    assert bench.traffic_profile("x", str(path)) == (3, 0.5, 7)
    assert bench.traffic_profile("y", str(path)) == (None, None, None)
    assert all(os.path.exists(os.path.join(bench.ROOT, "luisacompute_amd", "csrc", n)) for n in bench.TRACE_SOURCES)
