"""Runs tests/cpp/test_host_memory: what the host call holds in pinned memory and threads."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BINARY = os.path.join(ROOT, "tests", "cpp", "test_host_memory")


@pytest.mark.gpu
def test_host_memory():
    p = subprocess.run([BINARY], cwd=ROOT, capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout + p.stderr


def test_is_built():
    assert os.path.exists(BINARY), "tests/cpp/test_host_memory missing: build() compiles it"
