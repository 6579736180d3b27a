"""The small-batch matrix-core kernel at the edges of its token blocks, row
blocks and K split: int32 sub-block sums bit for bit against the oracle, fp32
outputs to the path's tolerance (rel-L2 1e-4), every layout, the debug export
and a grouped call bit-identical to the plain one.  Which calls the kernel
takes is csrc/small_batch_plan.h's use_small_batch (test_host_plans.py)."""
import numpy as np
import pytest

from oracle.oracle import LAYOUT_KM, LAYOUT_MK, compute_metrics

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# K, N, M: the first and last M of each 8-token step that takes short rows (two MFMAs per decode past 32); a row
# block of 1, 20 and 32 rows and a ragged last one; one super-block, fewer than the waves, and a K whose
# super-blocks do not divide among them; then both sides of the lines on which the route to the GEMM lies
CASES = [(256, 1, 9), (256, 33, 16), (768, 70, 17), (2048, 95, 24), (2304, 64, 25), (5120, 129, 32),
         (8448, 40, 16), (768, 5120 + 7, 12), (512, 32 * 384, 10), (256, 32 * 383 - 5, 31), (512, 2048, 33),
         (4096, 2049, 48), (4352, 1000, 49), (4096, 2100, 64), (3328, 90, 40), (5120, 33, 57), (8192, 1024, 8),
         (3840, 300, 41), (4096, 300, 41), (1024, 300, 40), (1280, 300, 40), (1792, 300, 40), (5120, 300, 65)]


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


# K, N, M where every wave has several super-blocks, their counts unequal: each 8-token step with the waves that
# its narrow and its wide matrices get (12 or 8 and 8 or 4), so that the next block's staging and loads, the reuse
# of the two half blocks past 16 tokens and the final sum's reuse of the staging are run in each
SEVERAL = [(6656, 100, 15), (4352, 12300, 16), (7168, 90, 20), (4352, 12289, 24), (8192, 70, 29), (5376, 12300, 32),
           (8192, 100, 33), (4352, 8200, 40), (4352, 16400, 36), (8448, 100, 41), (4352, 8225, 48), (4352, 100, 50),
           (5120, 8191, 56), (8448, 100, 64), (4352, 8192, 57), (8448, 1030, 7)]


@pytest.mark.parametrize("K,N,M", SEVERAL)
def test_several_super_blocks_per_wave(pkg, orc, K, N, M):
    """Sampled rows (first, last and some between) against the oracle; a group with a narrow matrix, whose wave
    count is another one where N is wide, against single calls."""
    dev = torch.device("cuda:0")
    print(f"several super-blocks K={K} N={N} M={M}", flush=True)
    W = pkg.synthetic_weights(K, N, seed=7100 + K + N, device=dev)
    X = orc.gen_activations(K * M, seed=8100 + M, outliers=True).reshape(M, K)
    AQ = orc.quantize_q8_1_batched(X, K, M, LAYOUT_MK)
    ws = pkg.quantize_q8_1(torch.from_numpy(X).to(dev), K, M, LAYOUT_MK)
    S, Yd = pkg.subblock_sums(W, ws, K, N, M, pkg.PATH_GEMM if M > 8 else pkg.PATH_GEMV)
    Y = pkg.mul_mat_q8_1(W, ws, K, N, M, LAYOUT_MK)
    row = K // 256 * 136
    n2 = 60 if M > 8 else 1030  # below 1024 rows 8 columns take another kernel
    Yg = pkg.mul_mat_q8_1_group([W, W[:n2 * row]], ws, K, [N, n2], M, LAYOUT_MK)
    Y2 = pkg.mul_mat_q8_1(W[:n2 * row], ws, K, n2, M, LAYOUT_MK)
    torch.cuda.synchronize()
    assert torch.equal(Yd, Y) and torch.equal(Yg[0], Y) and torch.equal(Yg[1], Y2)
    rows = sorted({*range(0, min(N, 33)), *range(N // 2, min(N, N // 2 + 20)), *range(max(0, N - 40), N)})
    at = torch.tensor(rows, device=dev)
    Wr = np.ascontiguousarray(W.view(N, row)[at].cpu().numpy().ravel())
    assert np.array_equal(S[:, at].cpu().numpy(), orc.subblock_sums(Wr, AQ, K, len(rows), M))
    m = compute_metrics(orc.gemm_semantics(Wr, AQ, K, len(rows), M).T, Y[:, at].cpu().numpy())
    assert m["rel_l2"] <= 1e-4 and not m["bad"], m


def sums_in_sixteen(S, W, AQ, K, N, M):
    """[M][N] fp32 outputs and their fp64 values from the exact sub-block sums, K's super-blocks dealt out to sixteen
    partial sums that are added one after another: acc = fma(sumi, fl(d_w (ls - 32) d_x), acc) per sub-block."""
    b, nsb = W.reshape(N, K // 256, 136), K // 32
    d = b[:, :, :2].copy().view(np.float16)[..., 0].astype(np.float32)
    hi = b[:, :, 2].astype(np.int32) | (b[:, :, 3].astype(np.int32) << 8)
    ls = np.stack([((b[:, :, 4 + i // 2].astype(np.int32) >> (4 * (i % 2))) & 15) | (((hi >> (2 * i)) & 3) << 4)
                   for i in range(8)], -1).reshape(N, nsb) - 32
    sa = np.repeat(d, 8, 1) * ls.astype(np.float32)  # exact
    dx = AQ.reshape(M, nsb, 36)[:, :, :2].copy().view(np.float16)[..., 0].astype(np.float32)
    sumi = np.where(ls == 0, 0, S // np.where(ls == 0, 1, ls))  # exact: S is their product
    term = sumi * (sa[None] * dx[:, None]).astype(np.float64)
    parts = []
    for w in range(16):
        acc = np.zeros((M, N), np.float32)
        for kb in range(w, K // 256, 16):
            for s in range(8 * kb, 8 * kb + 8):
                acc = (acc + term[:, :, s]).astype(np.float32)
        parts.append(acc)
    y = parts[0]
    for p in parts[1:]:
        y = y + p
    return y, term.sum(-1)


# K, N, M: 384 to 511 row blocks (eight waves of two sums each, an odd and an even number of
# super-blocks, fewer than sixteen), and twelve waves at both ends of their range of K
@pytest.mark.parametrize("K,N,M", [(17408, 12288, 8), (8192, 16352, 4), (2304, 12257, 7), (1280, 13000, 5),
                                   (3328, 4096, 8), (3584, 2048, 6), (7936, 5120, 4)])
def test_no_further_from_64_bits_than_sixteen_sums(pkg, orc, K, N, M):
    dev = torch.device("cuda:0")
    print(f"precision K={K} N={N} M={M}", flush=True)
    W = pkg.synthetic_weights(K, N, seed=9000 + K, device=dev)
    X = orc.gen_activations(K * M, seed=9100 + M, outliers=True).reshape(M, K)
    AQ = orc.quantize_q8_1_batched(X, K, M, LAYOUT_MK)
    ws = pkg.quantize_q8_1(torch.from_numpy(X).to(dev), K, M, LAYOUT_MK)
    Y = pkg.mul_mat_q8_1(W, ws, K, N, M, LAYOUT_MK)
    torch.cuda.synchronize()
    R, row = 512, K // 256 * 136  # the last rows: those of a ragged block among them
    Wr = W[(N - R) * row:].cpu().numpy()
    want, exact = sums_in_sixteen(orc.subblock_sums(Wr, AQ, K, R, M), Wr, AQ, K, R, M)
    got = Y[:, N - R:].cpu().numpy()
    err = lambda y: np.linalg.norm(y - exact) / np.linalg.norm(exact)  # noqa: E731
    print(f"  against 64 bits {err(got):.3e}, sixteen sums {err(want):.3e}", flush=True)
    if (N + 31) // 32 >= 384:  # the same sums in the same order
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    assert err(got) <= err(want)
