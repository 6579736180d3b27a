"""The dequantiser on both sides of the output size from which it writes past
the caches: the large call must equal, bit for bit, the same super-blocks
expanded in small calls, and the first and last of them the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_blocks", [1, 7, 192 * 1024, 192 * 1024 + 1, 192 * 1024 + 777])
def test_large_and_small_calls_agree(pkg, orc, n_blocks):
    dev = torch.device("cuda:0")
    W = pkg.synthetic_weights(256, n_blocks, seed=21, device=dev)
    guard = torch.full((n_blocks * 256 + 64,), -1.0, device=dev)  # nothing past the output is written
    got = pkg.dequant(W, n_blocks, out=guard)[:n_blocks * 256]
    step = 100000
    for b in range(0, n_blocks, step):
        n = min(step, n_blocks - b)
        part = pkg.dequant(W[b * 136:(b + n) * 136], n)
        assert torch.equal(got[b * 256:(b + n) * 256].view(torch.int32), part.view(torch.int32)), b
    assert bool((guard[n_blocks * 256:] == -1.0).all())
    n = min(n_blocks, 64)
    Wh = W.cpu().numpy()
    for sl, ours in ((Wh[:n * 136], got[:n * 256]), (Wh[-n * 136:], got[-n * 256:])):
        want = orc.dequant(np.ascontiguousarray(sl), 256, n).ravel()
        assert np.array_equal(ours.cpu().numpy().view(np.uint32), want.view(np.uint32))
