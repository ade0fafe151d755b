"""The line between the product of few rows and the 128 x 128 tiles (neura_amd/csrc/few_rule.hpp), held to both forms as measured on
256 compute units: (element, N, K, packed rows, us of the tiles, us of the product of few rows).  The form the rule picks takes at most
9 % more than the faster one (two timings of one form differ by up to 6 %)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
Q8_0, Q3_K, Q4_K, Q5_K, Q6_K = 8, 11, 12, 13, 14
MEASURED = [
    (Q8_0, 18944, 3584, 512, 154.6, 213.9), (Q8_0, 18944, 3584, 1024, 261.9, 331.1), (Q8_0, 18944, 3584, 128, 65.1, 67.1), (Q8_0, 37888, 3584, 512, 268.3, 418.5),
    (Q8_0, 37888, 3584, 256, 162.9, 216.6), (Q8_0, 3584, 3584, 512, 56.1, 48.4), (Q8_0, 3584, 3584, 1024, 59.0, 76.7), (Q8_0, 4608, 3584, 1024, 105.4, 87.4),
    (Q8_0, 4608, 3584, 768, 59.8, 69.9), (Q8_0, 3584, 18944, 256, 249.7, 128.6), (Q8_0, 3584, 18944, 1024, 254.8, 386.0), (Q8_0, 512, 3584, 1024, 57.5, 25.3),
    (Q8_0, 8960, 1536, 256, 30.7, 32.9), (Q8_0, 8960, 1536, 512, 57.4, 49.9), (Q8_0, 4864, 896, 1024, 46.5, 35.2), (Q8_0, 4864, 896, 768, 27.8, 31.7),
    (Q8_0, 896, 4864, 1024, 70.6, 40.6), (Q8_0, 896, 4864, 4096, 86.8, 118.2), (Q8_0, 3584, 18944, 4096, 1015.3, 1987.1),
    (Q6_K, 18944, 3584, 512, 221.3, 192.6), (Q6_K, 37888, 3584, 2048, 1418.4, 1271.1), (Q6_K, 3584, 18944, 512, 388.7, 195.6), (Q6_K, 4608, 3584, 1024, 150.8, 95.6),
    (Q6_K, 896, 4864, 1024, 106.4, 38.7), (Q6_K, 512, 3584, 8192, 107.3, 116.9), (Q6_K, 37888, 3584, 8192, 5587.9, 4995.3),
    (Q3_K, 18944, 3584, 512, 154.5, 140.4), (Q3_K, 37888, 3584, 512, 252.2, 261.8), (Q3_K, 4608, 3584, 1024, 107.0, 71.4), (Q3_K, 3584, 18944, 4096, 1008.2, 1366.1),
    (Q3_K, 512, 3584, 8192, 85.5, 108.2), (Q3_K, 8960, 1536, 8192, 481.9, 402.4),
    (Q5_K, 18944, 3584, 256, 94.4, 84.2), (Q5_K, 37888, 3584, 512, 241.3, 282.7), (Q5_K, 3584, 3584, 512, 50.8, 40.1), (Q5_K, 4608, 3584, 768, 54.5, 67.3),
    (Q5_K, 8960, 1536, 512, 52.0, 42.4), (Q5_K, 3584, 18944, 1024, 229.0, 286.1),
    (Q4_K, 18944, 3584, 512, 125.4, 147.5), (Q4_K, 3584, 3584, 512, 43.1, 38.7), (Q4_K, 4608, 3584, 1024, 82.1, 77.1), (Q4_K, 3584, 18944, 256, 187.6, 89.4),
    (Q4_K, 8960, 1536, 768, 46.3, 56.9), (Q4_K, 896, 4864, 2048, 60.9, 54.7), (Q4_K, 3584, 3584, 1024, 47.9, 61.3)]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    folder = tmp_path_factory.mktemp("rule")
    source, program = folder / "rule.cpp", folder / "rule"
    source.write_text('#include "%s"\n#include <cstdio>\nint main() {\n    int e;\n    unsigned n, k, rows, units;\n'
                      '    while (std::scanf("%%d %%u %%u %%u %%u", &e, &n, &k, &rows, &units) == 5) std::printf("%%d\\n", (int)nh::few_rows_win(e, n, k, rows, units));\n}\n'
                      % os.path.join(ROOT, "neura_amd", "csrc", "few_rule.hpp"))
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-o", str(program), str(source)], check=True)

    def ask(points):
        done = subprocess.run([str(program)], input="\n".join("%d %d %d %d %d" % point for point in points), capture_output=True, text=True, check=True)
        return [answer == "1" for answer in done.stdout.split()]
    return ask


def test_the_faster_form_is_picked_at_the_measured_points(rule):
    for point, few in zip(MEASURED, rule([(*point[:4], 256) for point in MEASURED])):
        assert point[5 if few else 4] <= 1.09 * min(point[4:]), point


def test_rows_within_a_tile_s_padding_are_few_and_a_grid_s_height_is_kept(rule):
    assert all(rule([(element, n, 256, rows, 256) for element in (Q8_0, Q3_K, Q4_K, Q5_K, Q6_K) for n in (1, 37888) for rows in (1, 96)]))
    assert not any(rule([(element, 32, 256, 65535 * 32 + 1, 256) for element in (Q8_0, Q3_K, Q4_K, Q5_K, Q6_K)]))


def test_the_rule_counts_the_device_s_own_compute_units(rule):
    # 112 tiles leave more than half of 256 units idle, and of 112 none
    assert rule([(Q4_K, 3584, 3584, 512, 256), (Q4_K, 3584, 3584, 512, 112)]) == [True, False]
