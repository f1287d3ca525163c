"""Which plan a product takes and what it uses of its workspace (csrc/fwp_gemm_plan.hpp), on the host."""
import ctypes
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("plan") / "plan.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "host_stub", "plan.cpp"), "-o", so], check=True)
    lib = ctypes.CDLL(so)
    for f in (lib.plan_workspace, lib.plan_used, lib.plan_product_used, lib.plan_product_workspace):
        f.restype = ctypes.c_int64
    return lib


def sizes(n, lo, hi, seed):
    rng = random.Random(seed)
    for _ in range(n):
        yield tuple(int(lo * (hi / lo) ** rng.random()) for _ in range(2)) + (rng.choice((rng.randint(1, 1100), rng.randint(250, 400))),)


def test_gradients_stay_within_their_workspace(plan):
    """Results off a 16-byte boundary get another plan than the one the workspace's size comes from."""
    known = [(10367, 48977, 302), (10240, 32768, 288), (10142, 35166, 258), (32768, 32768, 256)]
    for rows, vocab, dim in known + list(sizes(100000, 4096, 65536, 1)) + list(sizes(20000, 1, 65536, 2)):
        have = plan.plan_workspace(rows, vocab, dim)
        for aligned in (0, 1):
            used = plan.plan_used(rows, vocab, dim, aligned)
            assert used <= have, (rows, vocab, dim, aligned, used, have)
    assert plan.plan_used(32768, 32768, 256, 1) >= 32768 * 256 * 3 // 2 and plan.plan_used(32768, 32768, 256, 0) == 0


def test_products_stay_within_their_workspace(plan):
    for M, N, K in list(sizes(20000, 1, 65536, 3)):
        for m, n, k in ((M, K, N), (M, N, K), (K, M, N)):
            have = plan.plan_product_workspace(m, n, k)
            assert plan.plan_product_used(m, n, k, 1) == have and plan.plan_product_used(m, n, k, 0) == 0, (m, n, k)


def test_a_product_asks_for_no_image_of_its_operand(plan):
    """A weight gradient of a wide layer: its partial results, a few copies of it, and nothing of the size of the 32768 tokens."""
    assert plan.plan_product_workspace(4096, 1024, 32768) <= 4 * 4096 * (1024 + 1)
    assert plan.plan_product_workspace(8192, 2048, 32768) == 0
