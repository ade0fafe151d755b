"""The lines between the product of few rows, the 128 x 128 tiles and the narrow products' own kernels (neura_amd/csrc/few_rule.hpp), held
to the forms as measured on 256 compute units: MEASURED (element, N, K, packed rows, us of the tiles, us of the product of few rows), where
the form the rule picks takes at most 9 % more than the faster one (two timings of one form differ by up to 6 %), and NARROW (element, N,
K, rows, gated, us of the vector and staged kernels, us of the product of few rows), at most 27 % more and 1.5 % on average."""
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

NARROW = [
    (Q8_0, 4608, 3584, 2, False, 19.8, 15.5), (Q8_0, 4608, 3584, 4, False, 31.9, 15.8), (Q3_K, 4608, 3584, 2, False, 14.3, 11.9),
    (Q3_K, 4608, 3584, 4, False, 19.9, 12.2), (Q5_K, 4608, 3584, 2, False, 16.4, 12.5), (Q5_K, 4608, 3584, 4, False, 30.8, 13.0),
    (Q6_K, 4608, 3584, 2, False, 15.2, 15.6), (Q6_K, 4608, 3584, 4, False, 20.1, 16.0), (Q8_0, 3584, 3584, 2, False, 18.5, 13.5),
    (Q8_0, 3584, 3584, 3, False, 26.2, 14.2), (Q8_0, 3584, 3584, 4, False, 25.1, 14.2), (Q3_K, 3584, 3584, 2, False, 8.8, 11.7),
    (Q3_K, 3584, 3584, 3, False, 15.5, 12.2), (Q3_K, 3584, 3584, 4, False, 18.3, 12.2), (Q5_K, 3584, 3584, 2, False, 10.0, 12.3),
    (Q5_K, 3584, 3584, 3, False, 17.2, 12.7), (Q5_K, 3584, 3584, 4, False, 27.2, 12.8), (Q6_K, 3584, 3584, 2, False, 9.5, 15.2),
    (Q6_K, 3584, 3584, 3, False, 15.9, 15.8), (Q6_K, 3584, 3584, 4, False, 18.4, 15.8), (Q8_0, 37888, 3584, 2, True, 110.3, 55.1),
    (Q8_0, 37888, 3584, 4, True, 154.8, 62.6), (Q3_K, 37888, 3584, 2, True, 55.8, 38.3), (Q3_K, 37888, 3584, 4, True, 91.4, 38.7),
    (Q5_K, 37888, 3584, 2, True, 69.5, 39.0), (Q5_K, 37888, 3584, 4, True, 147.7, 40.1), (Q6_K, 37888, 3584, 2, True, 57.0, 52.4),
    (Q6_K, 37888, 3584, 4, True, 94.4, 53.1), (Q8_0, 3584, 18944, 2, False, 60.9, 32.2), (Q8_0, 3584, 18944, 4, False, 89.5, 34.1),
    (Q3_K, 3584, 18944, 2, False, 32.7, 22.5), (Q3_K, 3584, 18944, 4, False, 50.5, 23.7), (Q5_K, 3584, 18944, 2, False, 38.7, 25.1),
    (Q5_K, 3584, 18944, 4, False, 77.6, 26.3), (Q6_K, 3584, 18944, 2, False, 34.1, 29.9), (Q6_K, 3584, 18944, 4, False, 51.5, 31.1),
    (Q8_0, 512, 3584, 2, False, 9.9, 10.6), (Q8_0, 512, 3584, 3, False, 13.7, 11.0), (Q8_0, 512, 3584, 4, False, 13.0, 11.1),
    (Q3_K, 512, 3584, 2, False, 7.2, 11.0), (Q3_K, 512, 3584, 3, False, 13.0, 11.3), (Q3_K, 512, 3584, 4, False, 9.4, 11.3),
    (Q5_K, 512, 3584, 2, False, 8.2, 11.2), (Q5_K, 512, 3584, 3, False, 14.8, 11.4), (Q5_K, 512, 3584, 4, False, 10.0, 11.5),
    (Q6_K, 512, 3584, 2, False, 7.2, 13.3), (Q6_K, 512, 3584, 3, False, 12.8, 13.5), (Q6_K, 512, 3584, 4, False, 9.4, 13.5),
    (Q8_0, 2048, 1536, 2, False, 8.1, 9.3), (Q8_0, 2048, 1536, 3, False, 11.1, 9.5), (Q8_0, 2048, 1536, 4, False, 11.1, 9.4),
    (Q3_K, 2048, 1536, 2, False, 5.5, 8.2), (Q3_K, 2048, 1536, 3, False, 9.8, 8.3), (Q3_K, 2048, 1536, 4, False, 7.4, 8.3),
    (Q5_K, 2048, 1536, 2, False, 6.0, 8.5), (Q5_K, 2048, 1536, 3, False, 10.7, 8.6), (Q5_K, 2048, 1536, 4, False, 8.0, 8.7),
    (Q6_K, 2048, 1536, 2, False, 5.4, 9.5), (Q6_K, 2048, 1536, 3, False, 9.7, 9.6), (Q6_K, 2048, 1536, 4, False, 7.4, 9.7),
    (Q8_0, 1536, 1536, 2, False, 8.1, 9.1), (Q8_0, 1536, 1536, 4, False, 11.2, 9.4), (Q3_K, 1536, 1536, 2, False, 5.4, 8.2),
    (Q3_K, 1536, 1536, 4, False, 7.4, 8.3), (Q5_K, 1536, 1536, 2, False, 6.0, 8.4), (Q5_K, 1536, 1536, 4, False, 7.9, 8.6),
    (Q6_K, 1536, 1536, 2, False, 5.4, 9.4), (Q6_K, 1536, 1536, 4, False, 7.4, 9.7), (Q8_0, 17920, 1536, 2, True, 29.7, 21.4),
    (Q8_0, 17920, 1536, 4, True, 45.3, 21.9), (Q3_K, 17920, 1536, 2, True, 19.6, 15.9), (Q3_K, 17920, 1536, 4, True, 27.3, 16.2),
    (Q5_K, 17920, 1536, 2, True, 23.0, 16.9), (Q5_K, 17920, 1536, 4, True, 44.2, 17.5), (Q6_K, 17920, 1536, 2, True, 20.3, 21.3),
    (Q6_K, 17920, 1536, 4, True, 27.5, 21.9), (Q8_0, 1536, 8960, 2, False, 18.7, 16.1), (Q8_0, 1536, 8960, 4, False, 25.9, 15.5),
    (Q3_K, 1536, 8960, 2, False, 16.0, 13.6), (Q3_K, 1536, 8960, 4, False, 19.7, 14.4), (Q5_K, 1536, 8960, 2, False, 18.2, 14.4),
    (Q5_K, 1536, 8960, 4, False, 30.5, 15.4), (Q6_K, 1536, 8960, 2, False, 16.6, 16.3), (Q6_K, 1536, 8960, 4, False, 20.2, 17.6),
    (Q8_0, 256, 1536, 2, False, 7.6, 8.1), (Q8_0, 256, 1536, 4, False, 10.6, 8.7), (Q3_K, 256, 1536, 2, False, 5.3, 8.1),
    (Q3_K, 256, 1536, 4, False, 7.2, 8.3), (Q5_K, 256, 1536, 2, False, 5.8, 8.3), (Q5_K, 256, 1536, 4, False, 7.8, 8.5),
    (Q6_K, 256, 1536, 2, False, 5.3, 9.1), (Q6_K, 256, 1536, 4, False, 7.2, 9.2), (Q8_0, 1152, 896, 2, False, 7.5, 7.9),
    (Q8_0, 1152, 896, 4, False, 9.9, 8.2), (Q8_0, 896, 896, 2, False, 7.5, 7.9), (Q8_0, 896, 896, 4, False, 9.9, 8.3),
    (Q8_0, 9728, 896, 2, True, 10.3, 11.6), (Q8_0, 9728, 896, 3, True, 13.8, 11.7), (Q8_0, 9728, 896, 4, True, 20.5, 11.7),
    (Q8_0, 896, 4864, 2, False, 11.4, 10.1), (Q8_0, 896, 4864, 4, False, 14.4, 12.1), (Q8_0, 4096, 3584, 2, False, 18.9, 13.8),
    (Q3_K, 4096, 3584, 2, False, 8.9, 11.7), (Q5_K, 4096, 3584, 2, False, 10.2, 12.4), (Q6_K, 4096, 3584, 2, False, 9.8, 15.3),
    (Q8_0, 14592, 1280, 2, False, 25.0, 13.2), (Q5_K, 2944, 256, 2, False, 6.1, 6.8), (Q5_K, 2688, 4096, 4, False, 23.6, 14.1),
    (Q8_0, 2816, 14336, 2, False, 39.8, 28.7), (Q5_K, 20864, 512, 4, False, 45.7, 9.7), (Q6_K, 384, 16384, 4, False, 10.7, 15.5),
    (Q6_K, 3712, 1280, 2, False, 6.0, 9.4), (Q5_K, 384, 5120, 4, False, 10.1, 11.2), (Q5_K, 5376, 16384, 2, False, 45.9, 28.2),
    (Q5_K, 1408, 2048, 4, False, 8.1, 9.9), (Q6_K, 384, 5120, 2, False, 9.1, 11.8), (Q6_K, 5504, 4096, 2, False, 15.4, 16.4),
    (Q6_K, 384, 3072, 2, False, 7.1, 9.5), (Q6_K, 14592, 1280, 2, False, 17.3, 13.8), (Q5_K, 1280, 2048, 2, False, 6.1, 9.7),
    (Q3_K, 2048, 11264, 2, False, 16.7, 14.7), (Q8_0, 640, 14336, 4, False, 25.3, 16.1), (Q3_K, 5760, 1280, 2, False, 9.4, 8.1),
    (Q5_K, 2816, 256, 4, False, 13.8, 7.1), (Q8_0, 384, 256, 2, False, 6.2, 6.9), (Q6_K, 1536, 2048, 4, False, 7.5, 10.2),
    (Q6_K, 6912, 11264, 2, False, 37.1, 28.8), (Q8_0, 20864, 512, 4, False, 19.9, 10.7), (Q5_K, 20864, 512, 2, False, 25.2, 9.4),
    (Q3_K, 768, 256, 4, False, 8.3, 7.0), (Q3_K, 384, 11264, 2, False, 9.4, 10.9), (Q6_K, 2944, 256, 4, False, 7.0, 7.2),
    (Q6_K, 16768, 1024, 4, False, 24.1, 14.6), (Q3_K, 3840, 1280, 4, False, 8.3, 8.1), (Q6_K, 2816, 14336, 2, False, 24.8, 24.2),
    (Q8_0, 768, 256, 2, False, 6.2, 6.8), (Q5_K, 20992, 256, 2, False, 25.8, 7.4), (Q8_0, 1280, 4096, 2, False, 12.1, 12.3),
    (Q3_K, 1152, 8192, 4, False, 16.2, 12.0), (Q6_K, 2816, 256, 2, False, 5.3, 6.9), (Q3_K, 14592, 1280, 2, False, 17.1, 10.7),
    (Q6_K, 640, 14336, 2, False, 11.4, 14.8), (Q6_K, 20864, 512, 2, False, 20.7, 10.7), (Q3_K, 4864, 512, 2, False, 8.6, 6.8),
    (Q8_0, 256, 6144, 4, False, 13.5, 11.6)]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    folder = tmp_path_factory.mktemp("rule")
    source, program = folder / "rule.cpp", folder / "rule"
    source.write_text('#include "%s"\n#include <cstdio>\nint main() {\n    int e, gated;\n    unsigned n, k, rows, units;\n'
                      '    while (std::scanf("%%d %%u %%u %%u %%u %%d", &e, &n, &k, &rows, &units, &gated) == 6)\n'
                      '        std::printf("%%d\\n", (int)(gated < 0 ? nh::few_rows_win(e, n, k, rows, units) : nh::few_narrow_rows_win(e, n, k, rows, gated, units)));\n}\n'
                      % os.path.join(ROOT, "neura_amd", "csrc", "few_rule.hpp"))
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-o", str(program), str(source)], check=True)

    def ask(points):
        done = subprocess.run([str(program)], input="\n".join("%d %d %d %d %d %d" % (point + (-1,))[:6] for point in points), capture_output=True, text=True, check=True)
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


def test_the_faster_form_of_narrow_products_is_picked_at_the_measured_points(rule):
    lost = []
    for point, few in zip(NARROW, rule([(*point[:4], 256, int(point[4])) for point in NARROW])):
        lost.append(point[6 if few else 5] / min(point[5:]))
        assert lost[-1] <= 1.27, point
    assert sum(lost) / len(lost) <= 1.015


def test_narrow_rows_of_more_than_a_pass_are_few_and_q4_k_keeps_its_tiles(rule):
    assert all(rule([(element, 32, 256, rows, 256, 0) for element in (Q8_0, Q3_K, Q5_K, Q6_K) for rows in (3, 5, 6, 7, 8)]))
    assert not any(rule([(Q4_K, 152064, 3584, rows, 256, 0) for rows in range(2, 9)]))
    # one round of the staged kernel's workgroups on 256 compute units is two on 128
    assert rule([(Q3_K, 4096, 3584, 2, 256, 0), (Q3_K, 4096, 3584, 2, 128, 0)]) == [False, True]
