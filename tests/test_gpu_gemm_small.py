"""The Q4_0 GEMM whose blocks are split over the waves, at the edges of its
16 x 16 tiles, its 4-block and 32-block steps and its dispatch, and the tiled
forms, bit for bit against the scalar oracle."""
import numpy as np
import pytest

from oracle import py_oracle as orc
from slm_testlib import assert_bitwise, gen, load_product

P = load_product()
pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    with P.AttentionContext(64, 2, 2, 16, 1) as c:
        yield c


def product(ctx, w, rows, cols, x, res=None):
    batch = x.shape[0]
    with P.Q4Matrix(w, rows, cols) as m:
        xd = torch.from_numpy(x).cuda()
        out = torch.full((batch, rows), float("nan"), device="cuda")
        if res is not None:
            out.copy_(torch.from_numpy(res))
        torch.cuda.synchronize()
        if res is None:
            ctx.gemm_q4_0_dev(m, xd.data_ptr(), batch, out.data_ptr())
        else:  # in place
            ctx.gemm_q4_0_residual_dev(m, xd.data_ptr(), batch, out.data_ptr(), out.data_ptr())
        ctx.sync()
        return out.cpu().numpy()


# rows, cols, batch: ragged row and token tiles; 9, 12, 13, 31 to 33, 64, 65 and
# 512 blocks; the last batches of 1024 rows that are split (64 x 10 workgroups of
# up to 16 blocks, 64 x 16 of more, on 256 CUs) and the first that are tiled;
# rows of 1 to 8 blocks, which are always tiled
CASES = [(20, 288, 16), (33, 384, 15), (24, 416, 5), (7, 992, 17), (48, 1024, 33), (31, 1056, 6),
         (64, 2048, 7), (65, 2080, 48), (96, 16384, 9), (1024, 512, 160), (1024, 512, 161),
         (1024, 544, 256), (1024, 544, 257), (4096, 4096, 12),
         (16, 32, 5), (20, 128, 16), (33, 160, 15), (48, 256, 33), (1024, 64, 256), (1024, 64, 257)]


@pytest.mark.parametrize("rows,cols,batch", CASES)
@pytest.mark.parametrize("residual", [False, True])
def test_bit_exact_with_scalar_reference(ctx, rows, cols, batch, residual):
    w = orc.quantize_q4_0(gen([81, rows, cols], (rows, cols)))
    x = gen([82, cols, batch], (batch, cols))
    res = gen([83, rows, batch], (batch, rows)) if residual else None
    got = product(ctx, w, rows, cols, x, res)
    want = orc.gemm_q4_0_f32(w, x, batch, rows, cols)
    if residual:
        want = res + want
    assert_bitwise(got, want, f"gemm {rows}x{cols} batch {batch}")


# the tiled forms: 64 x 64 tiles at most one per CU and more, 128 x 128 tiles;
# whole and ragged tiles, rows in fours and not, one and two stages of blocks
TILED = [(1024, 64, 320), (1028, 96, 301), (1028, 288, 290), (1027, 64, 301), (4096, 64, 320),
         (4100, 64, 257), (4099, 288, 263), (8192, 64, 512), (8188, 64, 509), (8189, 288, 509)]


@pytest.mark.parametrize("rows,cols,batch", TILED)
@pytest.mark.parametrize("residual", [False, True])
def test_tiles_bit_exact_with_scalar_reference(ctx, rows, cols, batch, residual):
    test_bit_exact_with_scalar_reference(ctx, rows, cols, batch, residual)


def test_infinite_scales(ctx):
    """A weight block with an infinite scale and a row of one with NaN reach
    exactly the outputs the reference's do."""
    rows, cols, batch = 24, 320, 11
    w = orc.quantize_q4_0(gen([84], (rows, cols))).reshape(rows, cols // 32, 18).copy()
    w[3, 4, :2] = np.array([np.inf], np.float16).view(np.uint8)
    w[9, 0, :2] = np.array([np.nan], np.float16).view(np.uint8)
    x = gen([85], (batch, cols))
    got = product(ctx, w.reshape(-1, 18), rows, cols, x)
    want = orc.gemm_q4_0_f32(w.reshape(-1, 18), x, batch, rows, cols).reshape(got.shape)
    assert np.isnan(want[:, 9]).all() and not np.isfinite(want[:, 3]).any()
    assert np.array_equal(got, want, equal_nan=True)
