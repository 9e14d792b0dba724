"""The split-bf16 prefill (head_dim 64 and 128) at the sizes where its forms, blocks
and key tiles begin and end, against float64 attention, and with values that
cannot be split."""
import numpy as np
import pytest

from slm_testlib import gen, load_product, split_form

P = load_product()
pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def run(heads, kvh, start, q, k, v, form=None):
    """attend_batch of rotated q [n][dim] over cache rows 0..start+n-1, in the
    form that the dispatch rules give the split kernel."""
    rows, n = k.shape[0], q.shape[0]
    form = form or split_form(q.shape[1], heads, kvh, start, n)
    with P.AttentionContext(q.shape[1], heads, kvh, max(rows, 16), 1) as ctx:
        ctx.kv_write(0, 0, 0, k)
        ctx.kv_write(0, 1, 0, v)
        qd = torch.from_numpy(q).cuda()
        out = torch.full_like(qd, float("nan"))
        torch.cuda.synchronize()
        assert ctx.prefill_kernel(start, n) == form
        ctx.attend_batch_dev(0, start, n, qd.data_ptr(), out.data_ptr())
        ctx.sync()
        return out.cpu().numpy()


def attend64(heads, kvh, start, q, k, v):
    """float64 attention; (out, per-element sum of |p v|, largest |score|)."""
    n, hd = q.shape[0], q.shape[1] // heads
    out, mag, smax = np.empty(q.shape), np.empty(q.shape), 0.0
    mask = np.arange(k.shape[0])[None, :] > start + np.arange(n)[:, None]
    for h in range(heads):
        g = h // (heads // kvh)
        hs, gs = slice(h * hd, (h + 1) * hd), slice(g * hd, (g + 1) * hd)
        s = q[:, hs].astype(np.float64) @ k[:, gs].astype(np.float64).T / np.sqrt(hd)
        s[mask] = -np.inf
        smax = max(smax, np.abs(s[~mask]).max())
        p = np.exp(s - s.max(1, keepdims=True))
        p /= p.sum(1, keepdims=True)
        out[:, hs] = p @ v[:, gs].astype(np.float64)
        mag[:, hs] = p @ np.abs(v[:, gs].astype(np.float64))
    return out, mag, smax


# hd, heads, kv_heads, start, n: every form with one, two and (consecutive) four
# heads per workgroup, of one, two, three, four, eight and more heads per KV
# head; block and tile edges (15/16/17 rows, 127 to 129 and 159 to 161 keys),
# odd and even block counts
CASES = {
    "split_keys": [
        (128, 2, 1, 112, 16), (128, 2, 1, 111, 17), (128, 2, 1, 113, 15), (128, 4, 1, 0, 128),
        (128, 4, 1, 0, 129), (128, 1, 1, 100, 28), (128, 1, 1, 127, 33), (128, 3, 1, 0, 160),
        (128, 3, 3, 30, 131), (128, 8, 1, 96, 65), (128, 12, 4, 0, 250), (128, 2, 2, 1000, 2),
        (128, 4, 2, 500, 47), (64, 32, 8, 0, 380), (64, 32, 8, 0, 384), (64, 24, 8, 5, 511),
        (64, 32, 8, 1, 1023)],
    "split_paired": [
        (128, 32, 8, 0, 545), (128, 32, 32, 3, 528), (64, 32, 32, 0, 1040),
        (64, 36, 12, 0, 1100), (64, 32, 16, 0, 1300)],
    "split_consecutive": [
        (128, 32, 8, 0, 1025), (128, 24, 8, 40, 1400), (128, 32, 16, 0, 1040),
        (64, 32, 8, 0, 2065), (64, 48, 6, 3, 1403), (64, 32, 32, 0, 2065),
        (64, 33, 11, 0, 2030), (64, 32, 16, 1, 2080)],
}
CASES = [(*c, form) for form, cases in CASES.items() for c in cases]


@pytest.mark.parametrize("hd,heads,kvh,start,n,form", CASES)
def test_against_float64(hd, heads, kvh, start, n, form):
    rows = start + n
    q = gen([71, heads, start, n], (n, heads * hd)) * np.float32(4)
    k = gen([72, heads, start, n], (rows, kvh * hd)) * np.float32(2)
    v = gen([73, heads, start, n], (rows, kvh * hd))
    ref, mag, smax = attend64(heads, kvh, start, q, k, v)
    got = run(heads, kvh, start, q, k, v, form)
    # Roundings of 2^-24: six per 32-key tile in an output sum and one in the
    # row sum, per score 24 accumulations (of partial sums taken as at most
    # twice the largest score, in log2 units) and the pre-scaled q, and a few
    # in exp2, the normalisation and the dropped products.
    tiles = (rows + 31) // 32
    bound = (7 * tiles + 2 * 25 * 1.4427 * smax + 16) * 2.0 ** -24
    err = np.abs(got - ref) / mag
    assert err.max() <= bound, (err.max(), bound)
    # and on average far below: the roundings are not all one way
    rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert rel < 3e-6, rel


@pytest.mark.parametrize("start,n", [(0, 97), (0, 127), (30, 97)])
def test_many_heads_before_row_128(start, n):
    """Batches too short for the split kernel with so many heads that they fill
    the CUs several times over."""
    test_against_float64(128, 1024, 64, start, n, "four_heads")


@pytest.mark.parametrize("hd,heads,kvh,start,n", [(128, 2, 1, 100, 60), (128, 32, 8, 0, 600),
                                                  (128, 32, 32, 0, 1100), (64, 32, 8, 0, 500)])
def test_values_that_cannot_be_split(hd, heads, kvh, start, n):
    """-inf scores drop their key, inf and near-overflow values travel, and
    earlier rows and other KV heads do not see them."""
    rows = start + n
    q = np.abs(gen([74, n], (n, heads * hd))) + np.float32(0.1)
    k = gen([75, n], (rows, kvh * hd))
    v = gen([76, n], (rows, kvh * hd))
    j_k, j_v, j_big = rows - 45, rows - 20, rows - 9
    # its probability stays small beside a running max that may lag by 2^8
    k[j_big, :hd] = -2
    k2, v2 = k.copy(), v.copy()
    k2[j_k, :hd] = -np.inf           # every score of KV head 0 there is -inf
    v2[j_v, 3] = np.inf
    v2[j_big, 5] = np.float32(3.4e38)  # rounds to a bf16 infinity
    got = run(heads, kvh, start, q, k2, v2)
    kr = k.copy()
    kr[j_k, :hd] = np.float32(-1e4)  # exp underflows to 0: the key drops out
    vr = v.copy()
    vr[j_v, 3] = 0
    vr[j_big, 5] = 0
    ref, mag, _ = attend64(heads, kvh, start, q, kr, vr)
    pos = start + np.arange(n)
    per = heads // kvh
    cols0 = np.arange(per) * hd      # KV head 0's query heads
    assert np.isposinf(got[np.ix_(pos >= j_v, cols0 + 3)]).all()
    big = got[np.ix_(pos >= j_big, cols0 + 5)]
    assert np.isfinite(big).all() and (big > 1e30).all()
    ok = np.ones(got.shape, bool)
    ok[np.ix_(pos >= j_v, cols0 + 3)] = False
    ok[np.ix_(pos >= j_big, cols0 + 5)] = False
    assert (np.abs(got - ref)[ok] <= 2e-5 * np.maximum(mag, 1e-3)[ok]).all()


@pytest.mark.parametrize("hd,heads,kvh,start,n", [(128, 2, 1, 100, 60), (128, 32, 8, 0, 600),
                                                  (64, 32, 8, 0, 500)])
def test_small_values(hd, heads, kvh, start, n):
    """V so small that its remainders lie below the least bf16."""
    rows = start + n
    q = gen([77, n], (n, heads * hd))
    k = gen([78, n], (rows, kvh * hd))
    v = gen([79, n], (rows, kvh * hd)) * np.float32(2.0 ** -122)
    v[:, 1] = 0
    ref, mag, smax = attend64(heads, kvh, start, q, k, v)
    got = run(heads, kvh, start, q, k, v)
    assert (got[:, 1] == 0).all()
    # Roundings of 2^-24: one per key in the output and row sums, per score hd/4
    # + 2 accumulations; and of 2^-150, the least f32's half, one per key.
    bound = (2 * rows + 2 * (hd / 4 + 3) * 1.4427 * smax + 16) * 2.0 ** -24
    assert (np.abs(got - ref) <= bound * mag + rows * 2.0 ** -150).all()


RANGE_CASES = [(128, 2, 1, 100, 60), (128, 32, 8, 0, 600), (128, 32, 32, 0, 1100),
               (64, 32, 8, 0, 500), (64, 32, 8, 3, 1300)]


@pytest.mark.parametrize("expo", [-120, 120])
@pytest.mark.parametrize("hd,heads,kvh,start,n", RANGE_CASES)
def test_scores_of_tiny_and_huge_operands(hd, heads, kvh, start, n, expo):
    """Ordinary scores of a q whose remainders lie below the least bf16 with a
    k that makes up for it, and the other way round."""
    rows = start + n
    q = gen([80, n], (n, heads * hd)) * np.float32(2.0 ** expo)
    k = gen([81, n], (rows, kvh * hd)) * np.float32(2.0 ** -expo)
    v = gen([82, n], (rows, kvh * hd))
    ref, mag, smax = attend64(heads, kvh, start, q, k, v)
    got = run(heads, kvh, start, q, k, v)
    # Roundings of 2^-24: one per key in the output and row sums, per score hd/4
    # + 3; and of q, pre-scaled, to a multiple of 2^-149.
    bound = (2 * rows + 2 * (hd / 4 + 3) * 1.4427 * smax + 16 + 64) * 2.0 ** -24
    assert (np.abs(got - ref) <= bound * mag).all(), (np.abs(got - ref) / mag).max() / bound


@pytest.mark.parametrize("hd,heads,kvh,start,n", RANGE_CASES)
def test_tiny_probabilities_of_huge_values(hd, heads, kvh, start, n):
    """Key 0 has all the weight but only zero values: what counts are the other
    keys' probabilities of 2^-125 to 2^-124."""
    rows = start + n
    scale = np.float32(1.4426950408889634) / np.sqrt(np.float32(hd))
    one = np.float32(1) / scale
    one = next(x for x in (one, np.nextafter(one, np.float32(0)), np.nextafter(one, np.float32(99)))
               if x * scale == 1)  # scores in log2 units are then k's first dim, exactly
    q = np.zeros((n, heads * hd), np.float32)
    q[:, ::hd] = one
    k = np.zeros((rows, kvh * hd), np.float32)
    k[1:, ::hd] = np.floor(np.abs(gen([83, n], (rows - 1, kvh))) * 64) % 64 / 64 - 125
    v = gen([84, n], (rows, kvh * hd)) * np.float32(2.0 ** 120)
    v[0] = 0
    ref, mag, _ = attend64(heads, kvh, start, np.where(q != 0, np.sqrt(hd) * np.log(2), 0.0), k, v)
    got = run(heads, kvh, start, q, k, v)
    # Roundings of 2^-24: one per key in the output and row sums, and a few in
    # exp2 and the normalisation.
    bound = (2 * rows + 16) * 2.0 ** -24
    assert (np.abs(got - ref) <= bound * mag).all()


@pytest.mark.parametrize("hd,heads,kvh,start,n", RANGE_CASES)
def test_values_below_the_least_bf16(hd, heads, kvh, start, n):
    """Values that bf16 rounds to zero, in some dims; the other dims hold zeros
    and ordinary values."""
    rows = start + n
    q = gen([85, n], (n, heads * hd))
    k = gen([86, n], (rows, kvh * hd))
    v = gen([87, n], (rows, kvh * hd))
    v[:, 1::3] *= np.float32(2.0 ** -138)
    v[:, 2::3] = 0
    ref, mag, smax = attend64(heads, kvh, start, q, k, v)
    got = run(heads, kvh, start, q, k, v)
    # as test_small_values
    bound = (2 * rows + 2 * (hd / 4 + 3) * 1.4427 * smax + 16) * 2.0 ** -24
    assert (np.abs(got - ref) <= bound * mag + rows * 2.0 ** -150).all()


@pytest.mark.parametrize("tiny", [False, True])
@pytest.mark.parametrize("hd,heads,kvh,start,n", RANGE_CASES)
def test_sums_that_cancel(hd, heads, kvh, start, n, tiny):
    """Equal probabilities of values that cancel in pairs, so that every other
    row's sums are zero; beside values too small for bf16, in one dim of 16."""
    rows = start + n
    q = np.zeros((n, heads * hd), np.float32)
    k = gen([88, n], (rows, kvh * hd))
    v = gen([89, n], (rows, kvh * hd))
    v[1::2] = -v[:rows // 2 * 2:2]
    if tiny:
        v[:, 5::16] = np.abs(v[:, 5::16]) * np.float32(2.0 ** -138)
    ref, mag, _ = attend64(heads, kvh, start, q, k, v)
    got = run(heads, kvh, start, q, k, v)
    # Roundings of 2^-24, one per key in the output and row sums; of 2^-150, one per key
    bound = (2 * rows + 16) * 2.0 ** -24
    assert (np.abs(got - ref) <= bound * mag + (rows * 2.0 ** -150 if tiny else 0)).all()
