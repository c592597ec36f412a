"""How many runs of keys a decode attention launch cuts a sequence into: none, and none of the scratch that they share, up to 480 keys."""
from aphrodite_engine_amd import _lib


def test_runs_of_keys():
    runs = lambda seqs, longest, kv=8, heads=32, hd=128, block=16: _lib.lib().aphro_paged_attention_runs(seqs, heads, kv, hd, block, longest)
    # whoever overlaps launches of so few keys on several streams may
    assert all(runs(s, n, kv) == 1 for s in (1, 2, 8, 16) for n in (1, 256, 353, 400, 480) for kv in (1, 2, 8))
    assert [runs(1, n) for n in (481, 611, 8192)] == [6, 7, 8] and [runs(8, n) for n in (480, 481, 4096)] == [1, 4, 4]
    assert [runs(16, n) for n in (864, 865)] == [1, 2] and runs(33, 4096) == 1
    assert runs(1, 4096, hd=64) == runs(1, 4096, block=8) == runs(1, 4096, kv=1, heads=32) == 1
    assert runs(0, 4096) == 1


def test_runs_that_are_dealt_out():
    runs = lambda seqs, longest, kv=8: _lib.lib().aphro_paged_attention_runs(seqs, 4 * kv, kv, 128, 16, longest)
    # more than a quarter of the CUs' groups and 2017 keys on: up to eight runs, the launch looks at the lengths; none with a group for every CU
    assert [runs(s, 2017) for s in (8, 9, 17, 31, 32)] == [4, 8, 8, 8, 1] and [runs(s, 2016) for s in (9, 12, 17)] == [3, 2, 1]
    assert [runs(s, 4000, 1) for s in (64, 65, 255, 256)] == [4, 8, 8, 1]
