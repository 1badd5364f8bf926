"""The size rules of the one-launch dispatch, on the CPU: which worlds take it, and with how many tokens a block."""
import os
import subprocess

import pytest

from tests.test_host_runtime_tsan import CSRC, STUB, ROOT, clang


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    """plan(K, hidden, fp8, tokens of every rank, experts) -> (one launch, every wave by itself, tokens of a block)"""
    if clang() is None:
        pytest.skip("no clang on this machine")
    binary = str(tmp_path_factory.mktemp("plan") / "plan_driver")
    subprocess.run([clang(), "-std=c++17", "-O1", "-I", STUB, "-I", os.path.join(ROOT, "include"), "-I", CSRC,
                    os.path.join(CSRC, "ep_plan.cpp"), os.path.join(STUB, "plan_driver.cpp"), "-o", binary], check=True)

    def ask(K, hidden, fp8, tokens, experts=64, fused_small_max=4096, fused_shared_max=16384):
        line = " ".join(map(str, [experts, K, hidden, int(fp8), fused_small_max, fused_shared_max, len(tokens), *tokens]))
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


# (tokens, ranks, hidden, top-k, fp8, experts), tokens of a block (0: the separate launches); figures beside plan_small
LINES = [
    # worlds of up to 4096 selections: by how many blocks a CU gets
    ((32, 16, 2048, 8, True, 64), 4), ((32, 16, 2048, 8, True, 1280), 1), ((32, 16, 2048, 8, True, 2560), 4),
    ((32, 16, 2048, 8, False, 1024), 4), ((32, 16, 2048, 8, False, 1280), 1), ((32, 16, 2048, 8, False, 2560), 4),
    ((20, 24, 3072, 8, True, 528), 2), ((20, 20, 3072, 8, True, 80), 2), ((20, 20, 3072, 8, True, 520), 1),
    ((20, 20, 3072, 8, True, 2560), 1), ((16, 24, 1152, 5, True, 72), 4), ((16, 24, 1152, 5, True, 1296), 1),
    ((26, 16, 2048, 8, True, 64), 4), ((26, 16, 2048, 8, False, 64), 1), ((24, 16, 2048, 8, True, 64), 1),
    ((26, 16, 4096, 8, False, 64), 1), ((200, 4, 3072, 4, False, 64), 1), ((96, 8, 2048, 5, True, 64), 4),
    ((55, 12, 4096, 2, True, 96), 1), ((158, 8, 3328, 1, True, 64), 1), ((222, 8, 3456, 1, True, 8), 1),
    ((109, 8, 3968, 2, True, 8), 1), ((51, 16, 3328, 1, True, 256), 2), ((134, 8, 2560, 1, True, 64), 1),
    ((101, 12, 2304, 2, True, 384), 2), ((49, 12, 3072, 2, True, 36), 1),
    ((1024, 1, 768, 4, False, 64), 8), ((1024, 1, 4096, 4, False, 64), 1), ((64, 12, 1024, 1, True, 12), 8),
    # more selections: separate launches where a second block on a CU, or short rows of many ranks, cost more
    ((46, 32, 1024, 8, False, 512), 8), ((46, 32, 1024, 8, False, 640), 0), ((46, 32, 1024, 8, False, 1024), 8),
    ((46, 32, 1024, 8, True, 512), 8), ((46, 32, 1024, 8, True, 640), 0), ((46, 32, 1024, 8, True, 1024), 8),
    ((860, 2, 1024, 8, False, 512), 8), ((860, 2, 1024, 8, True, 512), 0), ((72, 8, 4096, 8, True, 768), 2),
    ((42, 24, 2048, 8, True, 528), 0), ((42, 24, 2048, 8, False, 528), 4),
    ((17, 32, 640, 8, False, 32), 0), ((17, 32, 2048, 8, False, 32), 4), ((17, 32, 640, 8, True, 32), 0),
    ((44, 12, 1024, 12, False, 36), 0), ((17, 32, 896, 12, False, 512), 0), ((53, 12, 1024, 10, False, 24), 0),
    ((92, 8, 1024, 9, False, 72), 8), ((471, 2, 896, 10, False, 16), 8), ((78, 24, 640, 4, False, 384), 0),
    ((251, 8, 640, 6, False, 64), 0), ((37, 24, 1152, 8, False, 192), 0), ((25, 32, 896, 12, True, 64), 0),
    ((57, 16, 768, 9, True, 64), 0), ((71, 16, 640, 8, True, 64), 0), ((19, 32, 896, 7, True, 128), 0),
    ((28, 20, 1024, 8, False, 40), 8), ((33, 32, 640, 4, False, 32), 0), ((40, 32, 1024, 4, False, 32), 8),
]


@pytest.mark.parametrize("world,tokens_of_a_block", LINES, ids=[str(w) for w, _ in LINES])
def test_where_blocks_share_the_lists(plan, world, tokens_of_a_block):
    T, R, hidden, K, fp8, experts = world
    fused, alone, block = plan(K, hidden, fp8, [T] * R, experts)
    assert alone == 0
    assert (block if fused else 0) == tokens_of_a_block
