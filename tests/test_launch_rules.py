"""The launch rules (csrc/launch_rules.hpp) over sizes up to the operators' limits, built for the host:
every launch they choose fits a dispatch, whose work-items (blocks x threads) count in 32 bits."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
BIG = (1 << 31) - 1


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("clang++") or "/opt/rocm/bin/amdclang++"
    so = str(tmp_path_factory.mktemp("rules") / "rules.so")
    subprocess.run([cxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "launch_rules", "rules_abi.cpp")], check=True)
    lib = ctypes.CDLL(so)
    i64 = ctypes.c_int64
    lib.rule_grid_fits.argtypes = [i64, i64]
    lib.rule_dqsq_blocks.argtypes = [i64, i64]
    lib.rule_dqsq_blocks.restype = i64
    return lib


@pytest.mark.parametrize("threads", [64, 128, 192, 256, 320, 512])
def test_dqsq_grid(rules, threads):
    """The row walk launches at least one workgroup, at most one per row, and never more than a dispatch
    holds, up to the operator's row limit (2^27 rows of 64 threads are one too many at two rows each)."""
    for M in (1, 2, 3, 1000, 16385, 131072, (1 << 27) - 1, 1 << 27, (1 << 27) + 1, 1 << 30, BIG):
        n = rules.rule_dqsq_blocks(M, threads)
        assert 1 <= n <= M
        assert rules.rule_grid_fits(n, threads), (M, n)
    # below the limit: two rows each
    assert rules.rule_dqsq_blocks(131072, threads) == max(65536, 512 * (2048 // threads))
