"""The GEMM's tiles of 32 tokens, which the planner takes for few tokens and in the tail of a plan: every output bit
for bit what the tiles of 128 tokens give (the debug export runs those), and sampled rows against the oracle."""
import numpy as np
import pytest

from oracle.oracle import LAYOUT_MK, compute_metrics

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
