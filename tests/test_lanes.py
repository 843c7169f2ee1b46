"""Device code for one wavefront on the host: 64 lanes as cooperative contexts (tests/lane_runtime.h),
built with the host compiler's undefined-behaviour checks (array bounds among them). The merged list
that a group of lanes forms, over lists of every length, dimensions and both precisions; parity with
the reference's walk (src/PhaseField.cpp:566-615) as tests/gather_driver.cpp repeats it."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
SAN = ["-fsanitize=undefined", "-fno-sanitize-recover=all", "-g"]


def _run(driver, tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text('#include "lane_runtime.h"\n')
    exe = tmp_path / "driver"
    cmd = [gxx, "-std=c++17", "-O1", "-ffp-contract=off", *SAN, f"-I{tmp_path}", f"-I{ROOT / 'tests'}",
           f"-I{ROOT / 'openphase_amd' / 'csrc'}", str(ROOT / "tests" / driver), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0 and "ubsan" in r.stderr:
        pytest.skip("no sanitizer runtime in this toolchain: " + r.stderr[-300:])
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and "runtime error" not in r.stderr, r.stderr[-3000:]
    return r.stdout


def test_merged_list_of_a_group(tmp_path):
    assert "gather ok" in _run("gather_driver.cpp", tmp_path)
