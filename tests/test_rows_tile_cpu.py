"""The few-rows tile's stage hand-over: what a wave read from a stage is in its registers before another wave may fetch into that stage."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_reads_are_waited_for_ahead_of_the_barrier():
    src = open(os.path.join(ROOT, "aphrodite_engine_amd", "csrc", "dense_rows.h")).read()
    loop = src[src.index("for (int s = 0; s < n; ++s)"):]
    waits = re.findall(r'"(s_waitcnt [^"]*)"', loop[:loop.index("__builtin_amdgcn_s_barrier")])
    assert len(waits) == 2 and all("vmcnt" in w and "lgkmcnt(0)" in w for w in waits), waits
