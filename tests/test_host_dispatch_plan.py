"""The size rules of the one-launch dispatch, on the CPU: which worlds take it, and with how many tokens a block."""
import os
import subprocess

import pytest

from tests.test_host_runtime_tsan import CSRC, STUB, ROOT, clang


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    """plan(K, hidden, fp8, tokens of every rank) -> (one launch, every wave by itself, tokens of a block)"""
    if clang() is None:
        pytest.skip("no clang on this machine")
    binary = str(tmp_path_factory.mktemp("plan") / "plan_driver")
    subprocess.run([clang(), "-std=c++17", "-O1", "-I", STUB, "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    os.path.join(CSRC, "ep_plan.cpp"), os.path.join(STUB, "plan_driver.cpp"), "-o", binary], check=True)

    def ask(K, hidden, fp8, tokens, fused_small_max=4096, fused_shared_max=16384):
        line = " ".join(map(str, [K, hidden, int(fp8), fused_small_max, fused_shared_max, len(tokens), *tokens]))
        out = subprocess.run([binary], input=line, stdout=subprocess.PIPE, text=True, check=True).stdout
        return tuple(map(int, out.split()))
    return ask


def test_the_cap_on_selections_that_a_program_sets_is_the_cap(plan):
    shared = (8, 2048, True, [640])                    # 5120 selections
    assert plan(*shared) == (1, 0, 4)
    assert plan(*shared, fused_small_max=0)[0] == 0
    assert plan(*shared, fused_small_max=5119)[0] == 0
    assert plan(*shared, fused_shared_max=5119)[0] == 0
    assert plan(8, 2048, True, [64], fused_small_max=0)[0] == 0
    assert plan(8, 2048, True, [64], fused_small_max=512)[0] == 1
    assert plan(8, 2048, True, [64], fused_small_max=511)[0] == 0
