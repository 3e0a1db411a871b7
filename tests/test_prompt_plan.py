"""The splits of a prompt's attention (csrc/prompt_plan.hpp, host arithmetic): which pages a row's
pieces cover, and how many launch shapes -- each a HIP graph of its own -- a prompt in chunks meets.
Compiled for the CPU."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAIN = """
#include <stdio.h>
#include "prompt_plan.hpp"
int main() {
  int tiles, heads, span;
  while (scanf("%d %d %d", &tiles, &heads, &span) == 3) {
    const llmk::PromptSplits s = llmk::prompt_splits(tiles, heads, span, 32);
    printf("%d %d\\n", s.num_splits, s.pages_per_split);
  }
}
"""


@pytest.fixture(scope="module")
def splits(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I",
                    os.path.join(ROOT, "cuda-llm-engine_amd", "csrc"), str(d / "main.cpp"), "-o",
                    str(d / "plan")], check=True)

    def run(cases):
        out = subprocess.run([str(d / "plan")], input="\n".join(" ".join(map(str, c)) for c in cases),
                             capture_output=True, text=True, check=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]
    return run


def test_pieces_cover_every_page_and_whole_steps(splits):
    cases = [(t, h, s) for t in (1, 2, 3, 8, 31, 32, 33, 65, 512) for h in (1, 2, 3, 8, 12, 300)
             for s in (1, 7, 8, 9, 16, 17, 63, 64, 65, 66, 127, 129, 1000, 8192)]
    for (tiles, heads, span), (n, pages) in zip(cases, splits(cases), strict=True):
        assert 1 <= n <= 32 and n * pages >= span and pages % 8 == 0
        assert n == 1 or n * tiles * heads <= 256
        exact = -(-span // n)
        assert n == 1 or pages < max(8, exact) * 1.25 + 8


@pytest.mark.parametrize("rows,heads", [(32, 8), (33, 8), (100, 8), (256, 8), (512, 8), (40, 2),
                                        (9, 1), (4096, 1)])
def test_chunks_of_a_long_prompt_share_their_launch_shapes(splits, rows, heads):
    ends = range(rows, 131072 + 1, rows)
    cases = [(-(-rows // 32), heads, (e - 1) // 16 + 1) for e in ends]
    assert len(set(splits(cases))) <= 33
