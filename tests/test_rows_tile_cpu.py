"""The few-rows tile: what a wave read from a stage is in its registers before another wave may fetch into that stage; K is cut over no more
workgroups than run at once."""
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_reads_are_waited_for_ahead_of_the_barrier():
    src = open(os.path.join(ROOT, "aphrodite_engine_amd", "csrc", "dense_rows.h")).read()
    loop = src[src.index("for (int s = 0; s < n; ++s)"):]
    waits = re.findall(r'"(s_waitcnt [^"]*)"', loop[:loop.index("__builtin_amdgcn_s_barrier")])
    assert len(waits) == 2 and all("vmcnt" in w and "lgkmcnt(0)" in w for w in waits), waits


def test_slices_of_tiles_that_have_a_cu_to_themselves():
    from aphrodite_engine_amd import _lib
    slices = _lib.lib().aphro_fp8_gemm_rows_ksplit
    # 64-column tiles times slices: up to 256 from 129 rows on, up to 512 below
    for n, k, few, many in ((6144, 4096, 5, 2), (9216, 1024, 2, 1), (4608, 3584, 7, 3)):
        assert [slices(m, n, k) for m in (128, 129, 192)] == [few, many, many]
