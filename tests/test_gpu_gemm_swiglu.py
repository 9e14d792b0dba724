"""Gate and up with SwiGLU in the projection's epilogue, in both tile shapes, at
the edges of the tiles and of the rule, bit for bit against the separate entry
points (gate, up, SwiGLU, down)."""
import numpy as np
import pytest

from slm_testlib import gen, load_product
from test_gpu_layer import Block, composed_step, dev

P = load_product()
pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# dim, hidden, n, weight scale: the last batches of separate launches and the
# first fused ones (80, 81 tokens of hidden 1024 at 9 blocks, 128, 129 at 17), the
# smallest fused one, 64 x 64 tiles with hidden and tokens cut by a tile, one
# block of nine more than a stage, 128 x 128 tiles whole and cut, and gates large
# enough to saturate
CASES = [
    (288, 1024, 80, 0.3), (288, 1024, 81, 0.3), (544, 1024, 128, 0.3), (544, 1024, 129, 0.3),
    (64, 32, 2, 0.3), (256, 704, 33, 0.3),
    (128, 1024, 128, 0.3), (128, 1024, 129, 0.3), (64, 1056, 193, 0.3), (288, 1568, 160, 0.3),
    (128, 4096, 512, 0.3), (128, 4064, 385, 0.3), (320, 4064, 500, 30.0), (64, 1056, 255, 30.0),
]


@pytest.mark.parametrize("dim,hidden,n,wscale", CASES)
def test_same_as_the_separate_launches(dim, hidden, n, wscale):
    heads = dim // 32
    blk = Block(61, dim, dim, hidden, wscale=wscale)
    try:
        with P.AttentionContext(dim, heads, heads, n, 1, 1e4) as a, \
                P.AttentionContext(dim, heads, heads, n, 1, 1e4) as b:
            x = gen([62, dim, n], (n, dim))
            x[n - 1, 3] = np.inf
            xa, xb = dev(x), dev(x)
            want = composed_step(b, blk, 0, 0, n, xb, 1e-5)
            for _ in range(2):  # the second call finds the first one's buffers
                xa.copy_(xb)
                torch.cuda.synchronize()
                a.layer_forward_dev(0, 0, n, blk.dev, 1e-5, xa.data_ptr())
                a.sync()
                got = xa.cpu().numpy()
                assert np.isfinite(got[:n - 1]).all()
                assert np.array_equal(got, want.cpu().numpy(), equal_nan=True)
    finally:
        blk.close()
