"""The plans of the Q4_K product of several rows (neura_amd/csrc/rows_rule.hpp), every one of them: what a workgroup stages fits the LDS of a
compute unit, its passes reach every row, its slices cover the rows, and the scratch that is set aside holds what the slices leave."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include "%s"
#include <cstdio>
int main() {
    unsigned tiles, blocks, many;
    while (std::scanf("%%u %%u %%u", &tiles, &blocks, &many) == 3) {
        const nh::RowsPlan plan = nh::rows_plan(tiles, blocks, many);
        const unsigned slice = (blocks + plan.splits - 1) / plan.splits;
        std::printf("%%u %%u %%u %%u %%zu %%u %%zu\n", plan.waves, plan.shares, plan.splits, slice, nh::rows_lds(slice, many ? 2 : 1, plan.waves, plan.shares),
                    nh::rows_passes(plan.waves) * nh::rows_hop(plan.waves, slice), nh::rows_scratch_bytes(16 * tiles, 256 * blocks, many ? 16 : 8));
    }
}
"""


def test_every_plan_fits_and_covers_its_rows(tmp_path):
    source, program = tmp_path / "rows.cpp", tmp_path / "rows"
    source.write_text(PROGRAM % os.path.join(ROOT, "neura_amd", "csrc", "rows_rule.hpp"))
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-o", str(program), str(source)], check=True)
    asked = [(tiles, blocks, many) for many in (0, 1) for blocks in list(range(1, 130)) + [208, 512, 4096] for tiles in (1, 2, 85, 86, 128, 129, 256, 257, 511, 512, 1023, 1024, 9504)]
    done = subprocess.run([str(program)], input="\n".join("%d %d %d" % point for point in asked), capture_output=True, text=True, check=True)
    answers = [tuple(map(int, line.split())) for line in done.stdout.splitlines()]
    assert len(answers) == len(asked)
    for (tiles, blocks, many), (waves, shares, splits, slice_, lds, staged, scratch) in zip(asked, answers):
        rows = 16 if many else 8
        assert lds <= 160 * 1024 and waves % shares == 0 and waves <= 16, (tiles, blocks, many)
        assert staged >= rows and slice_ * splits >= blocks > slice_ * (splits - 1), (tiles, blocks, many)
        assert scratch == (4 * splits * rows * (16 * tiles + 1) if splits > 1 else 0), (tiles, blocks, many)
        assert many or splits == 1 or blocks > 16
