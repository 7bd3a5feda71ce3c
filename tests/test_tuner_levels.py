"""The launch-shape tuners time the numbers of levels per work-group that an
untuned model or ensemble takes, so that tuning a grid never loses them."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

LEVELS = r"""
#include <algorithm>
#include <cstdio>
#include <vector>
namespace ps3d {
int tendency_levels(int tiles, int nz);
int friction_levels(int tiles, int nz, bool mixed, int nz_max);
std::vector<int> tune_levels(int untuned, int nz);
}
int main()
{
    int bad = 0;
    for (int tiles : {1, 3, 8, 24, 30, 72, 128, 300, 512, 2048})
        for (int nz = 2; nz <= 260; ++nz) {
            int rules[4] = {ps3d::tendency_levels(tiles, nz), ps3d::friction_levels(tiles, nz, false, nz),
                            ps3d::friction_levels(tiles, nz, true, nz), ps3d::friction_levels(tiles, nz, false, 260)};
            for (int r : rules) {
                const std::vector<int> c = ps3d::tune_levels(r, nz);
                const bool ok = r >= 1 && r <= nz && std::is_sorted(c.begin(), c.end()) && c.front() == 1 &&
                                c.back() == nz && std::adjacent_find(c.begin(), c.end()) == c.end() &&
                                std::binary_search(c.begin(), c.end(), r);
                if (!ok) ++bad;
            }
        }
    std::printf("%d\n", bad);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_candidates_hold_the_untuned_levels(tmp_path):
    """For the rules of both kernels, alone and in ensembles: 1, the untuned
    number and all levels are among the candidates, each once."""
    from ps3d_amd import _lib
    lib = os.path.join(ROOT, "ps3d_amd", "libps3d.so")
    _lib.load()
    src, exe = tmp_path / "levels.cpp", tmp_path / "levels"
    src.write_text(LEVELS)
    subprocess.run(["g++", "-std=c++17", str(src), lib, f"-Wl,-rpath,{os.path.dirname(lib)}",
                    "-Wl,--unresolved-symbols=ignore-in-shared-libs", "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    assert int(out) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("size,tendency,friction", [
    ((64, 64, 32), {1, 2, 4, 8, 16, 32}, {1, 2, 4, 8, 16, 32}),
    ((96, 96, 48), {1, 2, 3, 4, 8, 16, 32, 48}, {1, 2, 4, 5, 8, 16, 32, 48}),
    ((120, 120, 10), {1, 2, 4, 8, 10}, {1, 2, 4, 8, 10}),
    ((192, 192, 40), {1, 2, 4, 6, 8, 16, 32, 40}, {1, 2, 4, 8, 10, 16, 32, 40}),
])
def test_tuner_times_the_untuned_levels(size, tendency, friction):
    """Launches of the two stages while a model is tuned: three rounds of a
    warm-up and reps launches for each number of levels.  Untuned: 1, 3, 1 and
    6 levels for the tendency, 2, 5, 2 and 10 for friction."""
    from ps3d_amd import configs
    from ps3d_amd.model import Model
    print(f"tuner {size}", flush=True)
    reps = 1
    prm, fields = configs.eddy(*size)
    m = Model(prm)
    for n, a in fields.items():
        m.f[n][...] = a
    m.push()
    m.run(3)
    for stage, levels in (("tendency", tendency), ("friction_ab", friction)):
        m.profile_kernel(stage)
        m.tune(reps=reps)
        n, _ = m.profile_read()
        m.profile_kernel(None)
        chosen = {ln.split()[0]: int(ln.split()[2]) for ln in m.tuning().splitlines()}[stage]
        assert n == 3 * (1 + reps) * len(levels), stage
        assert chosen in levels, stage
    m.close()
