"""The launch plans' arithmetic (csrc/*_plan.h: plain C++, compiled here with the host
compiler) against its definition in Python's integers."""
import ctypes
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="session")
def plans(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("plans") / "plans.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC",
                    "-I", os.path.join(ROOT, "hyperion_amd", "csrc"), os.path.join(ROOT, "tests", "plans_shim.cc"),
                    "-o", so], check=True)
    return ctypes.CDLL(so)


def test_key_blocks_of_a_split(plans):
    """Chunk attention's split s of S takes blocks [B s / S, B (s + 1) / S) of B, up to the
    2^26 key blocks of the largest position range (2^31) and 256 splits."""
    f = plans.plan_split_first_block
    f.restype = ctypes.c_uint32
    rng = random.Random(5)
    cases = [(1, 1), (5, 4), (1 << 24, 256), ((1 << 24) + 255, 256), (1 << 26, 256), ((1 << 26) - 1, 255)]
    cases += [(rng.randrange(1, 1 << rng.randrange(1, 27)), rng.randrange(1, 257)) for _ in range(200)]
    for blocks, splits in cases:
        for s in {0, 1, splits // 2, splits - 1, splits}:
            assert f(blocks, s, splits) == blocks * s // splits, (blocks, s, splits)
