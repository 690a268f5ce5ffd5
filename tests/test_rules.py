"""The rules that choose sizes and routes (csrc/kernels.hpp), on both sides of each line.  No GPU:
tests/native/rules_check.cpp is compiled with g++ for the host."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT

INC = os.path.join(ROOT, "tr-spmm_zzx_amd", "csrc")
SRC = os.path.join(ROOT, "tests", "native", "rules_check.cpp")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("rules") / "rules_check.so")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                           "-I", INC, SRC, "-o", so])
    lib = ctypes.CDLL(so)
    lib.rule_lds_count_copies.argtypes = [ctypes.c_int64, ctypes.c_int32]
    lib.rule_spmm_route.argtypes = [ctypes.c_void_p, ctypes.c_int32, ctypes.c_int32, ctypes.c_void_p]
    lib.rule_hot_bytes.argtypes = [ctypes.c_void_p, ctypes.c_int32, ctypes.c_int32]
    lib.rule_hot_bytes.restype = ctypes.c_int64
    lib.rule_sddmm_one_pass.argtypes = [ctypes.c_void_p, ctypes.c_int32]
    lib.rule_sddmm_route.argtypes = [ctypes.c_void_p, ctypes.c_int32, ctypes.c_void_p]
    lib.rule_entry_ahead.argtypes = [ctypes.c_uint32, ctypes.c_int32, ctypes.c_int32, ctypes.c_uint32]
    lib.rule_entry_ahead.restype = ctypes.c_uint32
    lib.rule_windows_pay.argtypes = [ctypes.c_int64, ctypes.c_int64]
    lib.rule_task_sizes.argtypes = [ctypes.c_int64, ctypes.c_int64] + [ctypes.c_int32] * 5 + [ctypes.c_void_p]
    return lib


@pytest.mark.parametrize("n", [1, 4096, 32767, 32768, 32769, 60000, 65536, 65537, 250000, 1 << 20])
@pytest.mark.parametrize("total", [1, 8191, 600_000, 31_000_000])
def test_column_count_copies_stay_in_a_small_buffer(rules, total, n):
    c = rules.rule_lds_count_copies(total, n)
    assert c >= 1 and c * 8192 <= max(total, 8192)
    assert c * ((n + 32767) // 32768) <= 256
    # a buffer of 1.75 MB, or of 8 copies (16 past 2^16 columns)
    assert c * n * 4 <= max(7 << 18, (8 if n <= 1 << 16 else 16) * n * 4)
    assert rules.rule_counts_in_lds(n) == 1 and rules.rule_counts_in_lds((1 << 20) + 1) == 0


def sizes(rules, entries, nonempty, longest, spmm, split=False, task=0, piece=0):
    out = (ctypes.c_int32 * 7)()
    rules.rule_task_sizes(entries, nonempty, longest, int(spmm), int(split), task, piece, out)
    return dict(zip(("task", "narrow", "piece", "full_task", "full_piece", "row_task", "even"), out))


TINY, SMALL = 3 << 18, 3 << 20


@pytest.mark.parametrize("spmm", [True, False])
def test_task_sizes_of_even_rows(rules, spmm):
    """Rows no longer than a packed task: 16,384 tasks below 786,432 entries, and no row is cut."""
    for entries, rows, longest in ((278_000, 16384, 42), (483_463, 28439, 40), (552_000, 42440, 32), (740_053, 52861, 36)):
        z = sizes(rules, entries, rows, longest, spmm)
        want = min(z["row_task"], max(16, entries // 16384 if spmm or entries // 16384 >= 20 else 16))
        assert z["even"] and z["task"] == want and z["piece"] >= longest, (entries, z)
        assert z["narrow"] == (want if spmm else 16 if want < 24 else 24), (entries, z)
    for entries, rows in ((TINY, 46000), (1_020_000, 60000), (SMALL - 1, 180_000)):
        z = sizes(rules, entries, rows, 40, spmm)
        assert z["task"] == (min(z["row_task"], max(32, entries // 16384)) if spmm else 64), (entries, z)
    assert sizes(rules, SMALL, 180_000, 40, spmm)["task"] == 4 * SMALL // 180_000


def test_task_and_piece_sizes_of_uneven_rows(rules):
    # SpMM: tasks of 16 and pieces of 32 (tiny), 32 and 64 (small)
    z = sizes(rules, TINY - 1, 40_000, 4000, True, split=True)
    assert not z["even"] and (z["task"], z["piece"]) == (16, 32)
    z = sizes(rules, TINY, 40_000, 4000, True, split=True)
    assert (z["task"], z["piece"]) == (32, 64)
    assert sizes(rules, SMALL - 1, 90_000, 4000, True, split=True)["task"] == 47
    # SDDMM: 16-lane groups take 16,384 tasks (tiny) or tasks of 64, pieces of 64 from 393,216 entries on
    z = sizes(rules, 491_520, 12_000, 4000, False, split=True)
    assert (z["task"], z["narrow"], z["piece"], z["full_task"], z["full_piece"]) == (16, 16, 32, 30, 64)
    z = sizes(rules, 491_520, 12_000, 4000, False)
    assert (z["task"], z["piece"]) == (30, 64)
    z = sizes(rules, (3 << 17) - 1, 12_000, 4000, False)
    assert (z["piece"], z["full_piece"]) == (32, 32)
    z = sizes(rules, 983_040, 40_000, 4000, False, split=True)
    assert (z["task"], z["narrow"], z["piece"], z["full_piece"]) == (64, 32, 64, 128)
    # past 3,145,728 entries: pieces of 128 of short rows up to 5M entries (6,291,456 with split rows), else 256
    for entries, mean, split, want in ((3_194_880, 36, True, 256), (3_932_160, 26, True, 256), (4_915_200, 19.8, True, 128),
                                       (5_898_240, 14.7, True, 128), (5_898_240, 22.5, True, 256), (6 << 20, 15, True, 256),
                                       (4_990_000, 5.5, False, 128), (5_000_000, 5.5, False, 256)):
        z = sizes(rules, entries, int(entries / mean), 20_000, True, split=split)
        assert z["piece"] == want and z["task"] == z["row_task"], (entries, mean, z)
    assert sizes(rules, 3_194_880, 87_000, 14_000, False, split=True)["piece"] == 128
    # a longest row of at most two pieces stays whole
    assert sizes(rules, 200_000, 40_000, 64, True)["piece"] >= 64
    assert sizes(rules, 200_000, 40_000, 65, True)["piece"] == 32


def test_asked_sizes_are_taken(rules):
    for spmm in (True, False):
        z = sizes(rules, 500_000, 20_000, 4000, spmm, task=24, piece=100)
        assert (z["task"], z["narrow"], z["piece"], z["full_piece"]) == (24, 24, 100, 100)
        z = sizes(rules, 2_000_000, 40_000, 4000, spmm, task=512)
        assert (z["task"], z["piece"]) == (512, 512) and z["full_piece"] >= 512


def plan(entries, n, cut=0, split=0, task=64, row_task=64, even=0, hot=0, lanes=0):
    return (ctypes.c_int64 * 9)(entries, n, cut, split, task, row_task, even, hot, lanes)


def spmm(rules, p, K, aligned=True):
    out = (ctypes.c_int32 * 2)()
    rules.rule_spmm_route(p, K, int(aligned), out)
    return tuple(out)


RMAT = dict(entries=7_900_000, n=1 << 18, cut=9000, split=20_000, task=128, row_task=128, hot=16384)


def test_spmm_one_pass_widths(rules):
    short = plan(3_496_630, 349_663, task=44, row_task=44, even=1)
    long_rows = plan(2_400_000, 142_496, task=68, row_task=68, even=1)
    for K in range(100, 257, 4):
        if K % 8 == 0:
            assert spmm(rules, plan(**RMAT), K) == spmm(rules, short, K) == (8, 0)
        elif K < 128:
            assert spmm(rules, short, K) == (4, 32) and spmm(rules, long_rows, K) == spmm(rules, plan(**RMAT), K) == (8, 0)
        else:
            assert spmm(rules, short, K) == (4, 64) and spmm(rules, long_rows, K) == spmm(rules, plan(**RMAT), K) == (8, 32)
            # no staged rows, and no bytes for them
            assert rules.rule_hot_bytes(plan(**RMAT), K, 0) == 0 and rules.rule_hot_bytes(plan(**RMAT), K + 1, 0) > 0
            # a plan that asks for fewer lanes keeps its passes
            assert spmm(rules, plan(**{**RMAT, "lanes": 16}), K) == (8, 0)
            assert rules.rule_hot_bytes(plan(**{**RMAT, "lanes": 16}), K, 0) > 0
    assert spmm(rules, plan((1 << 17) - 1, 20_000, task=16, row_task=36, even=1), 180) == (8, 32)
    assert spmm(rules, plan(TINY - 1, 140_000, cut=64, task=16, row_task=32), 180) == (8, 32)
    assert spmm(rules, plan(TINY, 140_000, cut=64, task=32, row_task=32), 180) == (4, 64)
    assert spmm(rules, short, 260) == (4, 64) and spmm(rules, long_rows, 388) == (8, 32) and spmm(rules, plan(**RMAT), 260) == (8, 0)
    for K in (129, 130, 131, 254, 255, 258, 264):
        assert spmm(rules, short, K) == (8, 0)


def test_spmm_even_rows_of_narrow_widths(rules):
    big = dict(entries=2_400_000, n=142_496, task=68, row_task=68, even=1)
    for K in range(9, 33):
        assert spmm(rules, plan(**big), K) == ((1, 16) if K <= 16 else (2, 16))
        # a cut row, a split part or fewer lanes asked for: as any plan
        for other in (dict(cut=1), dict(split=8), dict(lanes=8), dict(even=0)):
            assert spmm(rules, plan(**{**big, **other}), K) == ((4, 0) if K <= 16 else (8, 0))
        # operands within half an L2, and tiny plans
        small = plan(**{**big, "n": 2_000_000 // (2 * K) - 1})
        tiny = plan(**{**big, "entries": TINY - 1})
        for p in (small, tiny):
            assert spmm(rules, p, K) == ((4, 0) if K <= 16 else (4, 8) if K % 2 else (8, 0))
        assert spmm(rules, plan(**{**big, "entries": (1 << 18) - 1}), K) == ((4, 0) if K <= 16 else (4, 8))


MESH = dict(entries=3_500_000, n=640_000, cut=64, task=32, row_task=32)


def test_spmm_meshes_with_a_few_long_rows(rules):
    for K in range(9, 33):
        small = {**MESH, "entries": (1 << 18) - 1, "n": 47_000}
        assert spmm(rules, plan(**small), K) == ((1, 16) if K <= 16 else (2, 16))
        for n in (640_000, 1_690_000, 4_194_304):
            want = (4, 0) if K <= 16 else (4, 8) if K % 8 and 32 << 20 <= n * K * 2 < 128 << 20 else (8, 0)
            assert spmm(rules, plan(**{**MESH, "n": n}), K) == want
        assert spmm(rules, plan(**{**MESH, "entries": TINY - 1, "n": 140_000}), K) == ((4, 0) if K <= 16 else (4, 8) if K % 2 else (8, 0))
        # long rows that are split, or rows that are not short: no mesh
        for other in (dict(split=9), dict(row_task=40)):
            assert spmm(rules, plan(**{**MESH, **other}), K) == ((4, 0) if K <= 16 else (8, 0))
        assert spmm(rules, plan(**{**small, "split": 9, "row_task": 60}), K) == ((4, 0) if K <= 16 else (4, 8))
    for K in (40, 48, 56, 64):
        assert spmm(rules, plan(**MESH), K) == (8, 0) and spmm(rules, plan(**MESH), K, aligned=False) == (4, 0)
        assert spmm(rules, plan(**MESH), K + 4 if K < 64 else 60) == (4, 0)
        # no cut row (an even graph of short tasks, whatever its longest row), few entries, far past the caches
        for other in (dict(cut=0), dict(cut=0, even=1, task=16), dict(entries=(1 << 18) - 1), dict(n=100_000_000 // K + 1)):
            assert spmm(rules, plan(**{**MESH, **other}), K) == (4, 0)
        assert spmm(rules, plan(**{**MESH, "n": 99_999_999 // K}), K) == (8, 0)


def test_windows_with_few_entries_in_tiles_are_dropped(rules):
    for tiles, entries, want in ((100, 1600, 1), (100, 1601, 0), (161, 491_520, 0), (16_384, 262_144, 1), ((1 << 18) - 1, 30_000_000, 0),
                                 (1 << 18, 30_000_000, 1), (1_030_000, 19_000_000, 1)):
        assert rules.rule_windows_pay(tiles, entries) == want, (tiles, entries)


def test_window_loads(rules):
    want = {4: 1, 5: 2, 8: 2, 9: 4, 16: 4, 17: 8, 23: 8, 25: 4, 28: 8, 32: 8, 33: 4, 34: 8, 36: 4, 40: 8, 44: 4, 48: 8, 52: 8, 63: 4, 65: 8}
    assert {K: rules.rule_window_vec(K) for K in want} == want


def test_sddmm_one_pass(rules):
    one = lambda p, K: rules.rule_sddmm_one_pass(p, K) == 1
    er = dict(entries=15_000_000, n=907_888, task=68, row_task=68, even=1)
    for K in (129, 132, 200, 255, 256):
        assert one(plan(**er), K) and not one(plan(**{**er, "lanes": 16}), K)
        # staged rows or a split part: as long as Y comes from the caches
        mb = 128 if K % 8 == 0 else 64 if K % 2 == 0 else 16
        fits, past = (mb << 20) // (2 * K), (mb << 20) // (2 * K) + 1
        for more in (dict(hot=100), dict(split=100)):
            assert one(plan(**{**er, **more, "n": fits}), K) and not one(plan(**{**er, **more, "n": past}), K)
    for K in (64, 128, 257, 384):
        assert not one(plan(**er), K)


def test_sddmm_routes(rules):
    def route(K, **more):
        out = (ctypes.c_int32 * 2)()
        rules.rule_sddmm_route(plan(**{**dict(entries=15_000_000, n=907_888, task=68, row_task=68, even=1), **more}), K, out)
        return tuple(out)

    for K in (4, 8, 9, 15, 16, 17, 24, 31, 32, 33, 64, 65, 98, 100, 104, 124, 128, 132, 256):
        plain = (1, 0) if K <= 8 else (2, 0) if K <= 16 else (4, 0) if K <= 64 else (8, 0)
        wide = (4, 32) if K in (100, 124) else plain
        assert route(K) == ((1, 16) if 8 < K <= 16 else (2, 16) if 16 < K <= 32 else wide)
        assert route(K, n=11_999_999 // (2 * K) if K <= 16 else 5_999_999 // (2 * K)) == wide
        assert route(K, entries=TINY - 1) == ((1, 16) if 8 < K <= 16 else plain)
        for other in (dict(even=0), dict(split=4), dict(lanes=8)):
            assert route(K, **other) == plain


def test_ragged_sddmm_rows_are_staged_past_48_mb(rules):
    for K in (121, 124, 127):
        fits, past = (48 << 20) // (2 * K), (48 << 20) // (2 * K) + 1
        assert rules.rule_hot_bytes(plan(**{**RMAT, "n": fits - 1}), K, 1) == 0
        assert rules.rule_hot_bytes(plan(**{**RMAT, "n": past}), K, 1) == 16384 * 128 * 2
    assert rules.rule_hot_bytes(plan(**{**RMAT, "n": 4096}), 128, 1) == 16384 * 128 * 2


@pytest.mark.parametrize("e", [1, 64, 513, (1 << 31) - 1])
def test_entries_ahead_stay_in_the_row(rules, e):
    """Also where the last row ends at the 2^31 - 1 entries that a plan may hold."""
    for p0 in (max(e - 700, 0), max(e - 65, 0), e - 1):
        for k in range(8):
            for lane in (0, 63):
                assert rules.rule_entry_ahead(p0, k, lane, e) == min(p0 + 64 * k + lane, e - 1)
