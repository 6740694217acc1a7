"""The LM head's dispatch (pz_lmtile.h): the cases of test_gpu_lmhead.py launch
every matrix-core kernel that a call can reach, so none can break unseen when
the rule or its times change."""
import os
import subprocess

from test_gpu_lmhead import LARGE_CASES, TILE_CASES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "native", "lm_tile_check.cpp")
INC = os.path.join(ROOT, "project-zero_amd", "csrc")


def paths(tmp_path, cases):
    exe = tmp_path / "lm_tile_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", INC, SRC, "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)] + [str(v) for c in cases for v in c], capture_output=True,
                         text=True, timeout=60, check=True)
    count, *lines = out.stdout.strip().split("\n")
    return int(count), [line.split() for line in lines]


def test_the_gpu_cases_reach_every_tile(tmp_path):
    count, lines = paths(tmp_path, TILE_CASES + LARGE_CASES)
    got = {p for line in lines for p in line}
    # the 256-row batch block (tile 0) never loads W non-temporally
    want = {str(i) for i in range(count)} | {f"{i}nt" for i in range(1, count)} | {"own16", "own32"}
    assert got == want


def test_rows_past_the_workspace_and_chunks(tmp_path):
    _, lines = paths(tmp_path, [(300, 1000, 131072), (4, 1000, 131080), (600, 1000, 512),
                                (33, 128256, 64)])
    assert len(lines[0]) == 19       # 16 batch rows at a time
    assert lines[1] == ["own16"]     # no workspace at all
    assert len(lines[2]) == 3        # 256, 256 and 88
    assert not lines[3][0].startswith("own")  # more than 32 rows: the parts made once
