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


def test_wide_weights_that_the_library_serves_better():
    from aphrodite_engine_amd import _lib
    ours = lambda m, n, k: bool(_lib.lib().aphro_dense_rows_preferred(m, n, k))
    assert all(ours(m, n, k) for m in (1, 64) for n, k in ((12288, 4096), (22016, 4096), (57344, 8192)))
    assert not any(ours(m, n, k) for m in (65, 128, 192) for n, k in ((11264, 4096), (12288, 4096), (15360, 5120), (18944, 3584), (37888, 3584)))
    assert all(ours(65, n, 4096) and ours(96, n, 4096) and not ours(97, n, 4096) for n in (22016, 28672))
    assert all(ours(m, n, k) for m in (65, 97, 192) for n, k in ((32000, 4096), (128256, 4096), (4096, 14336), (10240, 8192), (11264, 2048)))
    assert not ours(193, 4096, 4096) and not ours(16, 4096, 4100)


def test_a_workspace_for_many_rows_serves_fewer():
    from aphrodite_engine_amd import _lib
    lib = _lib.lib()
    for n in (1024, 1280, 4096, 4608, 6144, 7168, 9216, 10240, 17408, 28672):
        for k in (1024, 2048, 4096, 8192, 28672):
            sizes = [lib.aphro_fp8_gemm_workspace_bytes(m, n, k) for m in range(1, 301)]
            assert sizes == sorted(sizes)
            assert all(sizes[m - 1] >= 4 * m * n * lib.aphro_fp8_gemm_rows_ksplit(m, n, k) for m in range(33, 193))


def test_a_prompt_workspace_for_many_rows_serves_fewer():
    from aphrodite_engine_amd import _lib
    size = _lib.lib().aphro_scaled_mm_fp8_large_workspace_bytes
    rows = [*range(1, 400), *range(400, 3000, 37), *range(3000, 9000, 211)]
    for n in (128, 1280, 4096, 4224, 6144, 22016, 28672, 37888):
        for k in (128, 1024, 2048, 4096, 11008, 14336):
            sizes = [size(m, n, k) for m in rows]
            assert sizes == sorted(sizes) and sizes[-1] <= 4096 + 256 * 8 * 32 * 1024


def test_int4_products_whose_workspace_is_too_small_for_their_form_stay_refused():
    """(Refused on the host, ahead of any launch.)  Tiles that workgroups share, a copy of bf16 rows that does not fit, slices that a norm sums."""
    from aphrodite_engine_amd import _lib
    lib, p = _lib.lib(), 1 << 20
    size = lambda m, n, k, dt: lib.aphro_wna16_gemm_large_workspace_bytes(m, n, k, k // 128, dt)
    call = lambda m, n, k, dt, ws, room: lib.aphro_wna16_gemm_large(p, p, p, p, p, ws, room, m, n, k, k // 128, k, 1, dt, None)
    refused = -3                                             # APHRO_ERR_WORKSPACE
    for m, n, k, dt, room in ((4096, 28672, 4096, _lib.F16, size(4096, 28672, 4096, _lib.F16) - 1), (150, 4096, 4096, _lib.BF16, 150 * 4096 * 2 - 1),
                              (8192, 4096, 4096, _lib.F16, 1 << 20), (150, 4096, 4096, _lib.BF16, 0)):
        assert call(m, n, k, dt, p if room else None, room) == refused
    assert lib.aphro_wna16_gemm_large_add_norm_supported(150, 4096, 4096, 32, _lib.F16)
    assert lib.aphro_wna16_gemm_large_add_norm(p, p, p, p, p, p, p, 1e-5, p, 160 * 4096 * 4, 150, 4096, 4096, 32, 4096, 1, _lib.F16, 0, None) == refused
