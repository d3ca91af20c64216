"""The launch rule of the FP8 GEMM (`hy-nomas_amd/csrc/gemm_plan.h`, CPU, no GPU
needed): which kernels the shapes of the GPU tests take on the MI355X's 256 CUs,
and that those tests reach every kernel shape of both modes."""
import subprocess
from pathlib import Path

import pytest

import gemm_shapes as S

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    exe = tmp_path_factory.mktemp("plan") / "gemm_plan_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", str(HERE / "gemm_plan_check.cpp"),
                    "-o", str(exe)], check=True)

    def run(mode, mnk, cus=256):
        text = "".join(f"{mode} {m} {n} {k} {cus}\n" for m, n, k in mnk)
        return subprocess.run([str(exe)], input=text, check=True, capture_output=True, text=True).stdout.splitlines()
    return run


def test_gpu_tests_run_the_kernels_they_name(routes):
    for table in S.ROWCOL_TABLES:
        got = routes(0, [(M, N, K) for M, K, N, *_ in table])
        assert dict(zip(table, got)) == table
    for table in S.BLOCKWISE_TABLES:
        got = routes(1, list(table))
        assert dict(zip(table, got)) == table


@pytest.mark.parametrize("guarded", [False, True])
def test_gpu_tests_reach_every_kernel_shape(guarded):
    """Checked against the oracle, and into guarded buffers."""
    row = (S.GUARD, S.GUARD_TAIL) if guarded else (S.SMALL_ROWCOL, S.PERSISTENT, S.TAIL, S.LIGHT)
    bw = (S.GUARD_BLOCKWISE,) if guarded else (S.SMALL_BLOCKWISE, S.ZERO_FACTORS, S.TAIL_BLOCKWISE)

    def parts(tables):
        seen = set()
        for t in tables:
            for r in t.values():
                i = r.find("tail")
                seen.update([r[i:]] if i == 0 else [r] if i < 0 else [r[:i].strip(), r[i:]])
        return seen
    tails = {"tail 4x1", "tail 4x2", "tail 2x1", "tail 2x2"}
    small = {"64x64", "64x128", "128x128", "128x192", "128x256", "256x192"}
    assert parts(row) >= small | tails | {"256x256", "256x256 edge", "256x256 light"}
    assert parts(bw) >= {"64x64", "128x128", "128x256", "256x256"} | ({"256x256 edge"} if guarded else tails)


def test_workloads_of_the_rule_s_comments(routes):
    """The shapes that the rule's comments and the measured tables speak of."""
    assert routes(0, [(10800, 12288, 3072), (10800, 9216, 3072), (10800, 3072, 12288), (10800, 3072, 3072),
                      (4096, 3072, 3072), (256, 9216, 3072), (256, 3072, 12288)]) == [
        "256x256 light", "256x256 light", "256x256 tail 4x2", "256x256 tail 4x2", "256x192", "128x128", "64x64"]
    assert routes(1, [(10800, 12288, 4096), (1536, 4096, 12288), (256, 4096, 4096)]) == [
        "256x256 tail 2x2", "128x256", "64x64"]
