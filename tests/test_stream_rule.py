"""Which batches read the forward state with the streaming hint in the adjoint sweep, on the
host: a small program over the library's own header (csrc/common.hpp) prints it."""
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
    for (int i = 1; i + 4 < argc; i += 5) {
        EfmDims d{};
        d.nx = atoi(argv[i]); d.ny = atoi(argv[i + 1]); d.nz = atoi(argv[i + 2]); d.nshot = atoi(argv[i + 3]);
        d.wx_lo = d.wx_hi = d.wy_lo = d.wy_hi = d.wz_lo = d.wz_hi = atoi(argv[i + 4]);
        d.ntmax = 1;
        std::printf("%d ", (int)stream_forward_state(make_geo(d)));
    }
    return 0;
}
"""


def test_hint_while_the_adjoint_state_and_its_sums_are_cached(tmp_path):
    if not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "stream.hip", tmp_path / "stream"
    src.write_text(SOURCE)
    subprocess.run([build._hipcc(), "--offload-host-only", "-std=c++17", "-I", build.INCLUDE, "-I", build.CSRC, str(src),
                    "-o", str(exe)], check=True, capture_output=True, timeout=120)
    cases = [(n, m, k, S, W) for n in (64, 128, 140, 160, 200) for m in (64, 128, 150) for k in (40, 100, 128)
             for S in (1, 2, 9) for W in (0, 10)]
    out = subprocess.run([str(exe), *[str(v) for c in cases for v in c]], check=True, capture_output=True, text=True,
                         timeout=60).stdout.split()
    assert len(out) == len(cases) and set(out) == {"0", "1"}
    for (nx, ny, nz, S, W), got in zip(cases, out):
        N = nx * ny * nz
        psi = 24 * 2 * W * (ny * nz + nz * nx + ny * nx)
        # a shot's 9 adjoint fields, 8 sums and two sets of CPML slabs; lambda, mu and 6 averages
        assert int(got) == (4 * (S * (9 + 8) + 8) * N + 2 * S * psi <= 320e6), (nx, ny, nz, S, W)
