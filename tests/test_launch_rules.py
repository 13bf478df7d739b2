"""The launch layout rules (csrc/launch_rules.h) at and around every size where
they switch and at the largest accepted ray count, compiled for the host."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "cwbvh_amd" / "csrc"


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    """check([(expression, value)]): every expression has its value."""
    if not shutil.which("g++"):
        pytest.skip("no g++")
    path = tmp_path_factory.mktemp("rules")

    def run(cases):
        lines = "\n".join(f'    std::printf("%lld\\n", (long long)({e}));' for e, _ in cases)
        src = path / "rules.cpp"
        src.write_text(f'#include "launch_rules.h"\n#include <cstdio>\nusing namespace cw;\nint main() {{\n{lines}\n}}\n')
        subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(path / "rules")], check=True)
        out = subprocess.run([str(path / "rules")], check=True, capture_output=True, text=True).stdout.split()
        assert [(e, int(v)) for (e, _), v in zip(cases, out)] == [(e, int(w)) for e, w in cases]

    return run


def test_rays_per_wave(check):
    n = 2**31 - 1
    sizes = [(1, 4), (2048, 4), (2049, 8), (32768, 8), (32769, 16), (65536, 16), (65537, 64), (10**9, 64)]
    sizes += [(n - k, 64) for k in range(18)]
    check([(f"team_rays_per_wave({k}, 256)", v) for k, v in sizes])


def test_persistent_lines(check):
    """any hit, rays from surfels, teams of lanes, scene that streams from memory."""
    plain, any_hit, surfels = 3 << 18, 5 << 18, 1 << 21
    lines = {(1, 0, 1, 0): any_hit, (0, 1, 1, 0): surfels, (1, 1, 1, 0): surfels, (0, 1, 1, 1): surfels, (1, 1, 1, 1): surfels}
    every = [tuple(i >> k & 1 for k in range(4)) for i in range(16)]
    check([("auto_persistent_rays(%d, %d, %d, %d)" % k, lines.get(k, plain)) for k in every])


def test_waves_of_a_persistent_grid(check):
    """prefetch, ordered, scene that streams from memory."""
    every = [tuple(i >> k & 1 for k in range(3)) for i in range(8)]
    check([("grid_waves(%d, %d, %d)" % k, 4 if k == (1, 0, 1) else 0) for k in every])


def test_seven_wave_lines(check):
    check([("seven_wave_rays(%d, %d)" % k, 1 << 22 if k == (1, 0) else 3 << 21) for k in ((0, 0), (0, 1), (1, 0), (1, 1))])
