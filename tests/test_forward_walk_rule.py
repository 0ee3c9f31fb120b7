"""The rule that lets a forward step walk the interior cells only, on the host: a small
program over the library's own header (csrc/common.hpp) prints it for given batches."""
import os
import shutil
import subprocess

import pytest

from elastic_fm_vp_vs_rho_amd import build

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "common.hpp"
using namespace efm;
int main(int argc, char **argv) {
    for (int i = 1; i + 3 < argc; i += 4) {
        EfmDims d{};
        d.nx = atoi(argv[i]); d.ny = atoi(argv[i + 1]); d.nz = atoi(argv[i + 2]); d.nshot = atoi(argv[i + 3]);
        d.ntmax = 1;
        std::printf("%d ", (int)dense_walk(make_geo(d)));
    }
    return 0;
}
"""
CHIP = 14 * 256                     # blocks of 128 lanes


def _blocks(n, S, dense):
    nx, ny, nz = n
    cells = (nz - 4) * (nx - 4) if dense else (nz - 4) * nx - 4 + 31
    return -(-cells // 128) * (ny - 4) * S


def test_dense_where_it_saves_a_round_of_blocks_or_rows_are_short(tmp_path):
    if not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "walk.hip", tmp_path / "walk"
    src.write_text(SOURCE)
    subprocess.run([build._hipcc(), "--offload-host-only", "-std=c++17", "-I", build.INCLUDE, "-I", build.CSRC, str(src),
                    "-o", str(exe)], check=True, capture_output=True, timeout=120)
    cases = [((nx, ny, nz), S) for nx in (5, 28, 41, 63, 64, 65, 76, 128, 200) for nz in (5, 33, 64, 100)
             for ny in (5, 60, 119, 120, 124, 128, 200) for S in (1, 2, 7, 40)]
    args = [str(v) for n, S in cases for v in (*n, S)]
    out = subprocess.run([str(exe), *args], check=True, capture_output=True, text=True, timeout=60).stdout.split()
    assert len(out) == len(cases) and set(out) == {"0", "1"}
    for (n, S), dense in zip(cases, out):
        want = _blocks(n, S, False) > CHIP and (n[0] < 64 or _blocks(n, S, True) <= CHIP)
        assert int(dense) == want, (n, S)
    # a narrow batch of half a million cells, which whole lines push into a second round
    assert _blocks((52, 124, 78), 1, False) > CHIP >= _blocks((52, 124, 78), 1, True)
