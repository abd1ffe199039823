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


def gemm(plans, m, ns, k, dual=False, cus=256):
    """(kernel, splits, tiles per wave) of a call; kernel "few", 128 or 256."""
    out = (ctypes.c_uint32 * 3)()
    plans.plan_gemm(m, k, len(ns), (ctypes.c_uint32 * len(ns))(*ns), int(dual), cus, out)
    return ("few", 128, 256)[out[0]], out[1], out[2]


def test_gemm_choice_at_measured_calls(plans):
    """The choice at calls whose alternatives were measured (us, the choice first): q/k/v at 512
    rows 49.1 against 50.0 unsplit (54 on weights read from HBM), at 640 rows 53.5 unsplit; down
    at 2048 rows 208 against 221 unsplit; [3840, 8192] at 700 rows 61.8 against 68.1 (128-row
    tiles, split 2); gate/up at 512 rows 108 unsplit."""
    assert gemm(plans, 512, (4096, 2048, 2048), 3840)[:2] == (128, 2)
    assert gemm(plans, 512, (8192,), 3840)[:2] == (128, 2)
    assert gemm(plans, 640, (4096, 2048, 2048), 3840)[:2] == (128, 1)
    assert gemm(plans, 2048, (3840,), 15360)[:2] == (256, 2)
    assert gemm(plans, 700, (3840,), 8192)[:2] == (256, 5)
    assert gemm(plans, 512, (15360, 15360), 3840, dual=True)[:2] == (256, 1)


def test_gpu_cases_reach_the_kernels_they_name(plans):
    """The paths of the GEMM cases in test_gpu_parity.py and test_zz_no_alloc.py, case by case: a
    rule that moves a case to another kernel or split fails here rather than leave a form
    without a test."""
    from test_gpu_parity import DUAL_CASES, FEW_CASES, TILE_CASES
    few = [gemm(plans, *c) for c in FEW_CASES]
    assert few == [("few", 1, 1), ("few", 2, 1), ("few", 8, 1), ("few", 8, 1), ("few", 4, 4), ("few", 2, 2),
                   ("few", 8, 1), ("few", 2, 2), ("few", 4, 1), (128, 1, 0), ("few", 8, 1)]
    assert [gemm(plans, m, (262144,), 3840) for m in (16, 31)] == [("few", 1, 4)] * 2
    assert [gemm(plans, *c)[:2] for c in TILE_CASES] == [(256, 5), (256, 4), (256, 4), (256, 1), (128, 4), (128, 3), (128, 1)]
    dual = [gemm(plans, m, (n, n), k, dual=True) for n, k, m in DUAL_CASES]
    assert dual == [(256, 1, 0), (256, 1, 0), (128, 2, 0), ("few", 8, 2), ("few", 2, 2), ("few", 4, 2), ("few", 4, 4),
                    ("few", 4, 4), ("few", 4, 4), ("few", 4, 4), ("few", 4, 4), ("few", 8, 4), ("few", 2, 4),
                    (128, 1, 0), (128, 3, 0), (256, 1, 0), (256, 5, 0)]
    qkv = (4096, 2048, 2048)
    assert [gemm(plans, m, qkv, 3840)[:2] for m in (512, 1024, 2048)] == [(128, 2), (128, 1), (256, 1)]
    for m, ns, k, want in ((200, (40, 24, 1000), 4160, (128, 11)), (300, (200,), 4096, (128, 11)),
                           (2000, (8200,), 192, (128, 1)), (2000, (8195,), 320, (128, 1)), (2000, (8200,), 3840, (128, 1)),
                           (1300, (6000,), 4160, (256, 1)), (2000, (1000, 2000), 8256, (128, 1)), (2000, (3000,), 8256, (128, 1)),
                           (2048, (3840,), 15360, (256, 2)), (512, (2048,), 3840, (128, 6)), (1024, (4608,), 65536, (256, 3))):
        assert gemm(plans, m, ns, k)[:2] == want, (m, ns, k)
