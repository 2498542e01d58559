"""The rule for captures of HIP graphs among several threads (csrc/gate.hpp, host code): the self-test is compiled and run."""
from __future__ import annotations

import subprocess
from pathlib import Path

REPO = Path(__file__).resolve().parent.parent


def test_gate(tmp_path):
    exe = tmp_path / "gate_selftest"
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-pthread", "-I", str(REPO / "pagerank-cuda-dynamic_amd" / "csrc"),
                    "-o", str(exe), str(REPO / "tests" / "cpp" / "gate_selftest.cpp")], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr


def test_every_entry_that_reaches_the_device_holds_a_call():
    """Each exported function that touches a context's device opens with a Call; the others only read or set fields."""
    import re
    fields = {"prh_default_options", "prh_default_tuning", "prh_context_set_memory_limit", "prh_context_set_tuning",
              "prh_context_get_tuning", "prh_kernel_timing_enable", "prh_kernel_timing_read"}
    seen = set()
    for f in (REPO / "pagerank-cuda-dynamic_amd" / "csrc").glob("*.hip"):
        for name, body in re.findall(r"^(?:int|void) (prh_\w+)\([^{;]*\) \{\n(.*?)^\}", f.read_text(), re.M | re.S):
            seen.add(name)
            assert name in fields or body.startswith("  const Call call;\n"), name
            assert name not in fields or "hip" not in body.replace("hipError", ""), name
    assert {"prh_solve", "prh_stream_update", "prh_ppr_batched", "prh_graph_update"} <= seen
