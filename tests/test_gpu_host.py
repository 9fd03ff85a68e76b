"""Host paths with the runtime's calls watched (tests/cxx/host_check.cpp)."""
import os
import subprocess

import pytest

import gpu_index_test_amd as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", ["pinned_ranges", "stream_failure", "replace_index", "index_bytes", "build_failure",
                                  "pairs_memory", "pairs_failure", "dense_calls", "moved_scratch", "graphs_kept",
                                  "stream_graphs", "stalled_copy"])
def test_host_check(case):
    exe = os.path.join(os.path.dirname(G.__file__), "_lib", "host_check")
    r = subprocess.run([exe, case], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
