"""The launchers' scratch memory per stream and per recorded graph, on the host: stream_scratch.hip built by the
host compiler over a runtime that counts (tests/hip_stub), one run of stream_scratch_check.cpp per case."""
import re
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
SOURCE = HERE / "stream_scratch_check.cpp"
CASES = re.findall(r"CASE\((\w+)\)", SOURCE.read_text())[1:]   # the first is the macro's own


@pytest.fixture(scope="session")
def checks(tmp_path_factory):
    exe = tmp_path_factory.mktemp("scratch") / "checks"
    csrc = HERE.parent / "loken_amd" / "csrc"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wno-subobject-linkage", "-pthread", f"-I{HERE / 'hip_stub'}", f"-I{csrc}", str(SOURCE), "-o", str(exe)],
                   check=True)
    return exe


@pytest.mark.parametrize("case", CASES)
def test_scratch(checks, case):
    r = subprocess.run([str(checks), case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
