"""The launchers' host rules (csrc/small_batch_plan.h, csrc/dequant_plan.h), compiled for the host and asked about
many shapes."""
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
    exe = str(tmp_path_factory.mktemp("plan") / "host_plans")
    subprocess.run([CXX, "-std=c++17", "-O2", "-I" + os.path.join(ROOT, "qwen_3.8_27b_optimizations_amd", "csrc"),
                    os.path.join(ROOT, "tests", "arith", "host_plans.cpp"), "-o", exe], check=True)

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


# (N, K, M): the GEMM measured faster there, alone, in a pair or with two eighths of N beside it
SLOWER = [(32768, 1280, 16), (13312, 1536, 20), (28672, 1280, 24), (9216, 2560, 32), (28672, 3072, 32),
          (8192, 1280, 40), (13312, 5120, 40), (28672, 8192, 40), (2048, 768, 48), (8192, 1536, 48),
          (10240, 3328, 48), (28672, 5120, 48), (8192, 2560, 62), (17408, 5120, 49), (17408, 1536, 56),
          (11827, 1536, 57), (13824, 5120, 64), (151936, 4096, 56)]
# and there this kernel, in all three
FASTER = [(17408, 5120, 16), (5120, 17408, 16), (151936, 4096, 16), (151936, 1024, 24), (8192, 2560, 32),
          (12288, 4608, 32), (28672, 8192, 32), (5120, 8192, 33), (17408, 5120, 33), (12288, 4096, 40), (17408, 5120, 48),
          (8192, 5120, 64), (1024, 5120, 64), (5120, 17408, 64)]


def test_routes_by_measured_side(ask):
    """Shapes on both sides of the lines; past the kernel's columns and 32-bit offsets the GEMM."""
    cases = [(c, 0) for c in SLOWER] + [(c, 1) for c in FASTER]
    cases += [((1024, 5120, 65), 0), ((1 << 30, 256, 16), 0), (((1 << 30) - 1, 256, 16), 1),
              ((64, 1 << 24, 16), 0), ((64, (1 << 24) - 256, 16), 1)]
    for (c, want), (got,) in zip(cases, ask([f"small {n} {k} {m}" for (n, k, m), _ in cases])):
        assert got == want, c


def test_q_k_and_v_take_one_route(ask):
    """Up to 8192 rows the route does not depend on N: q, k and v of a grouped call stay in one launch."""
    cases = [(k, m) for k in range(256, 17409, 256) for m in range(9, 66)]
    rows = (8192, 4096, 1024, 1)
    got = ask([f"small {n} {k} {m}" for k, m in cases for n in rows])
    for i, c in enumerate(cases):
        assert len({g[0] for g in got[len(rows) * i:len(rows) * (i + 1)]}) == 1, c


def test_dequantiser_launches_hold_every_accepted_size(ask):
    """Sizes whose threads pass the 2^32 that one launch must stay below (from 2^27 super-blocks, 128 GiB of output)
    are divided; smaller ones stay one launch."""
    sizes = [1, 8, 12345, 2 ** 27 - 9, 2 ** 27 - 8, 2 ** 27 - 7, 2 ** 27, 2 ** 27 + 1, 2 ** 28 - 1, 2 ** 31 - 1]
    for n, got in zip(sizes, ask([f"dequant {n}" for n in sizes])):
        blocks, threads = got[0::2], got[1::2]
        assert sum(blocks) == n and max(threads) < 2 ** 32, n
        assert all(b * 32 <= t for b, t in zip(blocks, threads)), n
        assert len(blocks) == -(-n // (2 ** 27 - 8)), n
