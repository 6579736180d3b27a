"""The GEMM's tiles of 32 tokens, which the planner takes for few tokens and in the tail of a plan: every output bit
for bit what the tiles of 128 tokens give (the debug export runs those), and sampled rows against the oracle."""
import numpy as np
import pytest

from oracle.oracle import LAYOUT_MK, compute_metrics
from test_gpu_parity import NONFINITE_D, check_classes

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def check(pkg, orc, K, N, M, rows):
    dev = torch.device("cuda:0")
    print(f"gemm stages K={K} N={N} M={M}", flush=True)
    W = pkg.synthetic_weights(K, N, seed=300 + K, device=dev)
    X = orc.gen_activations(K * M, seed=301 + M, outliers=True).reshape(M, K)
    ws = pkg.quantize_q8_1(torch.from_numpy(X).to(dev), K, M)
    Y = pkg.mul_mat_q8_1(W, ws, K, N, M)
    Yd = pkg.subblock_sums(W, ws, K, N, M, pkg.PATH_GEMM)[1]
    torch.cuda.synchronize()
    assert torch.equal(Y, Yd)
    T = min(M, 40)  # the last tokens and rows
    AQ = orc.quantize_q8_1_batched(X[M - T:], K, T, LAYOUT_MK)
    Wr = W.view(N, -1)[N - rows:].cpu().numpy().ravel()
    m = compute_metrics(orc.gemm_semantics(Wr, AQ, K, rows, T).T, Y[M - T:, N - rows:].cpu().numpy())
    assert m["rel_l2"] <= 1e-4 and not m["bad"], m


# 40 row tiles and 8 token tiles of 128: one round of 256 workgroups, then 8 row tiles in tiles of 32 tokens
@pytest.mark.parametrize("K,N,M", [(256, 5120, 1000), (1280, 5100, 1024), (1792, 5120, 993)])
def test_tail_of_a_plan(pkg, orc, K, N, M):
    check(pkg, orc, K, N, M, 200)


# 40 row tiles and five tiles of 32 tokens, the last of 2 or 31: four super-blocks per stage, the last stage with
# one to four of them, the first one short as well
@pytest.mark.parametrize("K", [256 * b for b in (1, 2, 3, 4, 5, 6, 7, 8, 9, 13)])
@pytest.mark.parametrize("N,M", [(5120, 130), (5100, 159)])
def test_four_super_blocks_per_stage(pkg, orc, K, N, M):
    check(pkg, orc, K, N, M, 130)


@pytest.mark.parametrize("K", [256 * 4, 256 * 7])
@pytest.mark.parametrize("weights", [False, True])
def test_nonfinite_scales_in_every_slot_of_a_stage(pkg, orc, K, weights):
    """Tokens of different tiles whose Q8_1 scale overflows to +Inf in super-block 0, 1, 2 .. of the row, alone and
    on weights with non-finite scales of their own: every output keeps the reference's class."""
    dev = torch.device("cuda:0")
    N, M, R, bpr = 5120, 130, 150, K // 256
    print(f"non-finite K={K} weights={weights}", flush=True)
    W = orc.gen_weights(K, N, seed=93)
    b = W.reshape(N, bpr, 136)
    if weights:
        for j, r in enumerate(range(N - R, N, 7)):
            b[r, j % bpr, :2] = np.array([NONFINITE_D[j % 3]], np.uint16).view(np.uint8)
    X = orc.gen_activations(K * M, seed=94, outliers=True).reshape(M, K)
    for j in range(bpr):
        X[(21 * j + 3) % M, 256 * j + 40:256 * j + 60] = 3.0e7  # |x| >= 8.3e6: d_x is +Inf in fp16
    AQ = orc.quantize_q8_1_batched(X, K, M, LAYOUT_MK)
    ws = pkg.quantize_q8_1(torch.from_numpy(X).to(dev), K, M, LAYOUT_MK)
    Y = pkg.mul_mat_q8_1(torch.from_numpy(W).to(dev), ws, K, N, M, LAYOUT_MK)
    torch.cuda.synchronize()
    want = orc.gemm_semantics(np.ascontiguousarray(b[N - R:]).ravel(), AQ, K, R, M).T
    check_classes(want, Y[:, N - R:].cpu().numpy(), f"K={K}, non-finite weights {weights}")
