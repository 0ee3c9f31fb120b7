"""The rule that splits a forward batch into groups of shots, on the host: a small program
over the library's own header (csrc/common.hpp) prints the groups of a batch."""
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
// nx ny nz S Lx Ly Lz: the shots of each group of an in-place forward loop
int main(int argc, char **argv) {
    for (int i = 1; i + 6 < argc; i += 7) {
        int v[7];
        for (int k = 0; k < 7; ++k) v[k] = atoi(argv[i + k]);
        EfmDims d{};
        d.nx = v[0]; d.ny = v[1]; d.nz = v[2]; d.nshot = v[3];
        d.wx_hi = v[4]; d.wy_hi = v[5]; d.wz_hi = v[6]; d.ntmax = 1;
        const Geo g = make_geo(d);
        int next = 0;
        for_shot_groups(g, group_shots(g, field_bytes(g) + psi_bytes(g), 12 * g.N), [&](const Geo &gg) {
            if (gg.s0 != next) return 1;
            next += gg.S;
            std::printf("%d ", gg.S);
            return 0;
        });
        std::printf(next == v[3] ? "\n" : "gap\n");
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("groups")
    src, exe = d / "groups.hip", d / "groups"
    src.write_text(SOURCE)
    subprocess.run([build._hipcc(), "--offload-host-only", "-std=c++17", "-I", build.INCLUDE, "-I", build.CSRC, str(src),
                    "-o", str(exe)], check=True, capture_output=True, timeout=120)
    return str(exe)


def _groups(program, *cases):
    args = [str(v) for c in cases for v in c]
    out = subprocess.run([program, *args], check=True, capture_output=True, text=True, timeout=60).stdout
    return [[int(v) for v in line.split()] for line in out.splitlines()]


def _bytes(nx, ny, nz, S, Lx, Ly, Lz):
    N = nx * ny * nz
    return S * (36 * N + 24 * (ny * nz * Lx + Ly * nz * nx + ny * Lz * nx)) + 12 * N


GRIDS = [(73, 64, 37, 12, 12, 12), (64, 64, 64, 20, 20, 20), (36, 138, 89, 16, 16, 8), (96, 96, 96, 20, 20, 20),
         (57, 169, 47, 12, 12, 12), (41, 37, 33, 12, 12, 6), (130, 90, 60, 0, 0, 0)]


def test_a_batch_stays_whole_as_long_as_it_fits_the_cache(program):
    """One threshold, the 256 MB cache, whatever the grid."""
    cases = [(nx, ny, nz, S, *slabs) for nx, ny, nz, *slabs in GRIDS for S in range(1, 160, 1 if nx < 96 else 2)]
    for c, groups in zip(cases, _groups(program, *cases)):
        one = _bytes(*c[:3], 1, *c[4:])
        assert one <= 268e6
        assert (len(groups) == 1) == (c[3] == 1 or _bytes(*c) <= 268e6), c
        assert all(_bytes(*c[:3], k, *c[4:]) <= 268e6 for k in groups), c


def test_shots_beyond_the_cache_stay_together(program):
    assert _groups(program, (256, 256, 128, 4, 20, 20, 20), (200, 200, 200, 3, 0, 0, 0)) == [[4], [3]]


STEPS_SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include "common.hpp"
using namespace efm;
// nx ny nz S Lx Ly Lz nsteps: the shots of each group of a forward call of nsteps steps
int main(int argc, char **argv) {
    for (int i = 1; i + 7 < argc; i += 8) {
        int v[8];
        for (int k = 0; k < 8; ++k) v[k] = atoi(argv[i + k]);
        EfmDims d{};
        d.nx = v[0]; d.ny = v[1]; d.nz = v[2]; d.nshot = v[3];
        d.wx_hi = v[4]; d.wy_hi = v[5]; d.wz_hi = v[6]; d.ntmax = 1;
        const Geo g = make_geo(d);
        for_shot_groups(g, forward_group(g, v[7]), [&](const Geo &gg) { std::printf("%d ", gg.S); return 0; });
        std::printf("\n");
    }
    return 0;
}
"""


@pytest.mark.parametrize("nsteps", [0, 1, 2, 3, 4, 24, 1000])
def test_calls_of_a_step_or_two_keep_their_batch_whole(tmp_path, nsteps):
    """A group gains from its second step on only: loops stepped one call a step (or captured
    in chunks of one) must not pay a round of launches for each group."""
    if not (shutil.which("hipcc") or os.path.exists("/opt/rocm/bin/hipcc")):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "steps.hip", tmp_path / "steps"
    src.write_text(STEPS_SOURCE)
    subprocess.run([build._hipcc(), "--offload-host-only", "-std=c++17", "-I", build.INCLUDE, "-I", build.CSRC, str(src),
                    "-o", str(exe)], check=True, capture_output=True, timeout=120)
    cases = [(96, 96, 96, 32, 20, 20, 20), (64, 64, 64, 24, 20, 20, 20), (57, 169, 47, 20, 12, 12, 12)]
    for c, groups in zip(cases, _groups(str(exe), *[(*c, nsteps) for c in cases])):
        assert sum(groups) == c[3]
        assert (len(groups) == 1) == (nsteps < 3), (c, groups)
