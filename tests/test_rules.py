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
    return lib


@pytest.mark.parametrize("n", [1, 4096, 32767, 32768, 32769, 60000, 65536, 65537, 250000, 1 << 20])
@pytest.mark.parametrize("total", [1, 8191, 600_000, 31_000_000])
def test_column_count_copies_stay_in_a_small_buffer(rules, total, n):
    c = rules.rule_lds_count_copies(total, n)
    assert c >= 1 and c * 8192 <= max(total, 8192)
    assert c * ((n + 32767) // 32768) <= 256
    # a buffer of 2 MB, or of 8 copies (16 past 2^16 columns)
    assert c * n * 4 <= max(2 << 20, (8 if n <= 1 << 16 else 16) * n * 4)
    assert rules.rule_counts_in_lds(n) == 1 and rules.rule_counts_in_lds((1 << 20) + 1) == 0
