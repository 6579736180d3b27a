"""The small-batch matrix-core kernel at the edges of its token blocks, row
blocks and K split: int32 sub-block sums bit for bit against the oracle, fp32
outputs to the path's tolerance (rel-L2 1e-4), every layout, the debug export
and a grouped call bit-identical to the plain one."""
import numpy as np
import pytest

from oracle.oracle import LAYOUT_KM, LAYOUT_MK, compute_metrics

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# K, N, M: the first and last M of each 8-token step (two MFMAs per decode past 32); a row
# block of 1, 20 and 32 rows and a ragged last one; one super-block, fewer than the waves, and a K whose
# super-blocks do not divide among them; both sides of 384 and of 256 row blocks and of 16384 rows
CASES = [(256, 1, 9), (256, 33, 16), (768, 70, 17), (2048, 95, 24), (2304, 64, 25), (5120, 129, 32),
         (8448, 40, 16), (768, 5120 + 7, 12), (512, 32 * 384, 10), (256, 32 * 383 - 5, 31), (512, 2048, 33),
         (768, 2049, 48), (256, 8191, 49), (1280, 2100, 64), (256, 32 * 384, 40), (768, 32 * 383 + 5, 41),
         (3328, 90, 56), (5120, 33, 57), (512, 32 * 384 + 1, 64), (8192, 64, 8),
         (256, 8192, 50), (256, 8193, 34), (256, 16384, 64), (256, 16385, 56), (256, 16385, 57)]


@pytest.mark.parametrize("K,N,M", CASES)
def test_token_and_row_blocks(pkg, orc, K, N, M):
    dev = torch.device("cuda:0")
    print(f"small batch K={K} N={N} M={M}", flush=True)
    W = orc.gen_weights(K, N, seed=7000 + K + N)
    X = orc.gen_activations(K * M, seed=8000 + M, outliers=True).reshape(M, K)
    AQ = orc.quantize_q8_1_batched(X, K, M, LAYOUT_MK)
    Wd = torch.from_numpy(W).to(dev)
    ws = pkg.quantize_q8_1(torch.from_numpy(X).to(dev), K, M, LAYOUT_MK)
    S, Yd = pkg.subblock_sums(Wd, ws, K, N, M, pkg.PATH_GEMM if M > 8 else pkg.PATH_GEMV)
    Y = pkg.mul_mat_q8_1(Wd, ws, K, N, M, LAYOUT_MK)
    Ykm = pkg.mul_mat_q8_1(Wd, ws, K, N, M, LAYOUT_KM)
    n2 = min(N, 100)  # a second matrix of another size in the same call
    Yg = pkg.mul_mat_q8_1_group([Wd, Wd[:n2 * K // 256 * 136]], ws, K, [N, n2], M, LAYOUT_MK)
    Y2 = pkg.mul_mat_q8_1(Wd[:n2 * K // 256 * 136], ws, K, n2, M, LAYOUT_MK)
    torch.cuda.synchronize()
    assert np.array_equal(S.cpu().numpy(), orc.subblock_sums(W, AQ, K, N, M))
    m = compute_metrics(orc.gemm_semantics(W, AQ, K, N, M).T, Y.cpu().numpy())
    assert m["rel_l2"] <= 1e-4 and not m["bad"], m
    assert torch.equal(Yd, Y) and torch.equal(Ykm.T, Y)
    assert torch.equal(Yg[0], Y) and torch.equal(Yg[1], Y2)
