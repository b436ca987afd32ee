"""Which path the backend takes, and the same results on each, on the CPU:
tests/c/plugin/points-backend.c with the core, the backend and the CPU stand-in for
the kernel library, in a core that answers for backend strides as libCEED's."""

import os
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
C, HOST, ORACLE_LIB = ROOT / "tests" / "c", ROOT / "libceed_amd" / "host", ROOT / "oracle" / "liboracle.so"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not ORACLE_LIB.exists():
        pytest.skip("oracle library not built")
    exe = tmp_path_factory.mktemp("points") / "points-backend"
    res = subprocess.run(["gcc", "-O1", "-std=c11", "-Wall", f"-I{ROOT / 'include'}", f"-I{HOST}", f"-I{ROOT / 'oracle'}", str(C / "plugin" / "points-backend.c"),
                          *map(str, sorted(HOST.glob("*.c"))), str(C / "plugin" / "mi355-cpu-standin.c"),
                          "-Wl,--wrap=CeedElemRestrictionHasBackendStrides", f"-L{ORACLE_LIB.parent}", "-loracle", "-ldl", "-lm",
                          f"-Wl,-rpath,{ORACLE_LIB.parent}", "-o", str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return exe


def run(program, tmp_path, **env):
    log = tmp_path / "calls.log"
    log.unlink(missing_ok=True)
    res = subprocess.run([str(program), str(ROOT / "tests" / "qfunctions" / "t-points.h")], capture_output=True, text=True, timeout=120,
                         env=dict(os.environ, STANDIN_CEED_INCLUDE=str(ROOT / "include"), STANDIN_LOG=str(log), **env))
    assert res.returncode == 0, res.stdout + res.stderr
    return {k: float(v) for k, v in (line.split() for line in res.stdout.splitlines())}, log.read_text().split()


def test_paths_agree(program, tmp_path):
    fused, fused_calls = run(program, tmp_path)
    staged, staged_calls = run(program, tmp_path, CEED_MI355_FUSE_QFUNCTIONS="0")
    assert "PointOperatorApply" in fused_calls and "OperatorCreateHexJitFields" in fused_calls
    assert "PointOperatorCreate" not in staged_calls and "OperatorCreateHexJitFields" not in staged_calls
    assert fused.keys() == staged.keys() and len(fused) == 8
    for k in fused:  # sums of at most 108 values of either path, formed in the same order but for the fused contractions
        assert fused[k] == pytest.approx(staged[k], rel=1e-13), k
