"""The host rules of the small-batch matrix-core kernel (csrc/small_batch_plan.h), compiled for the host and asked
about many shapes."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = os.environ.get("CXX", "g++")


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    if shutil.which(CXX) is None:
        pytest.skip("needs a host C++ compiler")
    exe = str(tmp_path_factory.mktemp("plan") / "small_batch_plan")
    subprocess.run([CXX, "-std=c++17", "-O2", "-I" + os.path.join(ROOT, "qwen_3.8_27b_optimizations_amd", "csrc"),
                    os.path.join(ROOT, "tests", "arith", "small_batch_plan.cpp"), "-o", exe], check=True)

    def run(lines):
        r = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True)
        out = [[int(x) for x in line.split()] for line in r.stdout.splitlines()]
        assert len(out) == len(lines)
        return out

    return run


def groups():
    for n in list(range(8, 6600, 41)) + [2048, 3072, 4096, 5120, 6144]:
        yield [n, max(1, n // 8), max(1, n // 8)]  # q, k, v
    for n in range(5, 4200, 53):
        yield [n, n]
    for n in range(100, 2500, 97):
        yield [n, n + 13, 2 * n // 3, n // 5]
    for n in range(1, 8300, 67):
        yield [n]


@pytest.mark.parametrize("cus", [256, 304, 128, 64, 37])
def test_one_round_of_workgroups_where_one_is_enough(ask, cus):
    """A launch whose rows fit the CUs at 32 rows per workgroup has no more workgroups than CUs, and the fewest rows
    per workgroup (at least 8) that give that; past it, 32 rows each."""
    cases = list(groups())
    for Ns, (rows, wgs) in zip(cases, ask([f"rows {cus} " + " ".join(map(str, Ns)) for Ns in cases])):
        at = lambda r: sum(-(-n // r) for n in Ns)  # noqa: E731
        assert 8 <= rows <= 32 and wgs == at(rows), Ns
        if at(32) <= cus:
            assert wgs <= cus and (rows == 8 or at(rows - 1) > cus), (Ns, rows, wgs)
        else:
            assert rows == 32, (Ns, rows)
