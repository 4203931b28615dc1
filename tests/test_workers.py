"""Host threads of the set-up passes, through tests/cpp/test_workers (built by
__graft_entry__.build() / make -C tests/cpp)."""
import os
import subprocess

import pytest

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "test_workers")


def test_workers_pass_exceptions_on_and_do_without_threads():
    if not os.path.exists(BIN):
        pytest.fail(f"{BIN} is not built; run __graft_entry__.build() or make -C tests/cpp")
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
