"""The launch shapes of the deferred-cell kernel (openphase_amd/csrc/mpf_device.h), on the host: the
default is one of those the autotuner times, and none is timed twice."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "openphase_amd" / "csrc"

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "mpf_device.h"
int main(int, char** argv)
{
    const long long n = std::atoll(argv[1]);
    int grids[mpf::kDeferredTrials];
    const int k = mpf::deferred_trials(n, grids);
    std::printf("%d", mpf::deferred_blocks(n, mpf::kWideGrid));
    for (int i = 0; i < k; ++i) std::printf(" %d", mpf::deferred_blocks(n, grids[i]));
}
"""


@pytest.mark.parametrize("cells", [1, 64 * 40, 128 * 128, 512 * 512 - 1, 4096 * 32, 4096 * 32 + 1, 6144 * 32, 6144 * 32 + 1,
                                   16384 * 32, 256**3, 2**28 - 1])
def test_autotuner_times_the_default_grid_once(cells, tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no g++")
    src = tmp_path / "shape.cpp"
    src.write_text(SOURCE)
    subprocess.run([gxx, "-std=c++17", "-Wall", "-Wextra", "-Werror", f"-I{CSRC}", str(src), "-o", str(tmp_path / "shape")], check=True)
    default, *tried = map(int, subprocess.run([str(tmp_path / "shape"), str(cells)], capture_output=True, text=True,
                                              check=True).stdout.split())
    assert default in tried
    assert len(set(tried)) == len(tried)
