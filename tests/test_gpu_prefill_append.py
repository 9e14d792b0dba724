"""Prefills whose attention kernel appends the batch's K and V rows itself, at
the largest batches it takes and the first it does not, bit for bit against
the separate steps (rope, KV append, attention over the cache)."""
import numpy as np
import pytest

from slm_testlib import assert_bitwise, gen, load_product

P = load_product()
pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

# hd, heads, kv_heads, start, n: four, three, two and one head per KV head
CASES = [
    (128, 8, 2, 0, 2), (128, 8, 2, 60, 15), (128, 8, 2, 3, 16), (128, 8, 2, 3, 17),
    (64, 9, 3, 0, 16), (64, 9, 3, 31, 17), (16, 6, 2, 9, 16), (256, 4, 1, 16, 16),
    (32, 4, 2, 0, 31), (96, 4, 2, 1, 32), (96, 4, 2, 1, 33),
    (96, 4, 2, 1, 26), (96, 4, 2, 1, 27), (128, 4, 2, 0, 20), (128, 4, 2, 0, 21),
    (256, 2, 2, 5, 10), (256, 2, 2, 5, 11), (64, 2, 2, 3, 40), (64, 2, 2, 3, 41),
    (48, 6, 6, 0, 53), (48, 6, 6, 0, 54), (32, 4, 4, 9, 64),
    (48, 6, 6, 0, 16), (48, 6, 6, 7, 63), (16, 4, 4, 0, 64), (48, 6, 6, 0, 65), (256, 2, 2, 5, 64),
]


@pytest.mark.parametrize("hd,heads,kvh,start,n", CASES)
def test_same_as_the_separate_steps(hd, heads, kvh, start, n):
    dim, kvd, msl = hd * heads, hd * kvh, start + n + 3
    q, k, v = (torch.from_numpy(gen([91 + i, hd, start, n], (n, w))).cuda()
               for i, w in enumerate((dim, kvd, kvd)))
    with P.AttentionContext(dim, heads, kvh, msl, 2) as ctx:
        for layer in (0, 1):  # an earlier history, and a row behind that must stay
            for which in (0, 1):
                ctx.kv_write(layer, which, 0, gen([95, which], (msl, kvd)))
        out, want = torch.full_like(q, float("nan")), torch.full_like(q, float("nan"))
        rq = q.clone()
        torch.cuda.synchronize()
        ctx.prefill_dev(1, start, n, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr())
        ctx.kv_append_dev(0, start, n, k.data_ptr(), v.data_ptr())
        ctx.rope_apply_dev(rq.data_ptr(), n, dim, start)
        ctx.attend_batch_dev(0, start, n, rq.data_ptr(), want.data_ptr())
        ctx.sync()
        for which in (0, 1):
            assert_bitwise(ctx.kv_read(1, which, 0, msl), ctx.kv_read(0, which, 0, msl),
                           f"cache {'KV'[which]}")
        assert_bitwise(out.cpu().numpy(), want.cpu().numpy(), "output")
        assert np.isfinite(out.cpu().numpy()).all()
