"""The split-bf16 prefill's six bf16 products per f32 one, each by itself: inputs
whose results come down to one product of a probability and a value (of q and
k), so that little else is rounded and the bounds lie below what any one of the
six contributes.  The last test shows that on the CPU."""
import numpy as np
import pytest

from slm_testlib import gen, split_form
from test_gpu_prefill_split import run

# hd, heads, kv_heads, n, form; 160 rows come before the batch
START = 160
CASES = [(128, 2, 1, 20, "split_keys"), (128, 32, 8, 600, "split_paired"),
         (128, 32, 8, 1030, "split_consecutive"), (128, 32, 32, 1030, "split_consecutive"),
         (64, 32, 8, 400, "split_keys"), (64, 32, 32, 1040, "split_paired"),
         (64, 32, 8, 2065, "split_consecutive")]
# Keys 0 and 32, the first of either key split, score 0, which is then the
# running max throughout; HOT ones score below it, and all others vanish.  Dim d
# has one value that is not zero, that of key HOT[d % 16].
HOT = np.array([3, 8, 17, 30, 33, 40, 47, 63, 64, 78, 95, 100, 126, 127, 128, 159])


def full(seed, shape):
    """Values in [1, 2) with all their bits drawn."""
    bits = np.random.default_rng(seed).integers(0, 1 << 23, shape, dtype=np.uint32)
    return (bits | np.uint32(0x3F800000)).view(np.float32)


def scale_log2(hd):
    return np.float32(1.4426950408889634) / np.sqrt(np.float32(hd))


def value_inputs(hd):
    """Scores in log2 units, exact multiples of 2^-10, and values."""
    s = -np.random.default_rng([1, hd]).integers(1, 2048, 16).astype(np.float32) / 1024
    return s, full([2, hd], hd) * np.where(gen([3, hd], hd) < 0, -1, 1).astype(np.float32)


def score_inputs(hd, rows):
    """q (one dim, times 1 / scale) and k of the hot keys: scores of -2 to -16."""
    return full([4, hd], rows), -full([5, hd], 16) * np.float32([2, 4] * 8)


# Roundings of 2^-24: a probability's exp2 (two) and the same of the row sum,
# 17 additions of the row sum, two in the normalisation, six in the output sum
# and the products left out.
VALUE_BOUND = 31 * 2.0 ** -24
# The same, and the score's one at its full size (twice, up to 16, in log2
# units), in the probability and by at most two thirds in the row sum.
SCORE_BOUND = (31 + 2 * 16 * 0.6931 * 5 / 3) * 2.0 ** -24


def cache(hd, kvh, n, k_hot, v_hot, far):
    k, v = (np.zeros((START + n, kvh, hd), np.float32) for _ in range(2))
    k[..., 0] = far
    k[[0, 32], :, 0] = 0
    k[HOT, :, 0] = k_hot[:, None]
    d = np.arange(hd)
    v[HOT[d % 16], :, d] = v_hot[:, None]
    return k.reshape(START + n, -1), v.reshape(START + n, -1)


@pytest.mark.gpu
@pytest.mark.parametrize("hd,heads,kvh,n,form", CASES)
def test_products_with_values(hd, heads, kvh, n, form):
    s, w = value_inputs(hd)
    one = np.float32(1) / scale_log2(hd)
    one = next(x for x in (one, np.nextafter(one, np.float32(0)), np.nextafter(one, np.float32(99)))
               if x * scale_log2(hd) == 1)
    q = np.zeros((n, heads, hd), np.float32)
    q[..., 0] = one
    k, v = cache(hd, kvh, n, s, w, -200)
    got = run(heads, kvh, START, q.reshape(n, -1), k, v, form).reshape(n, heads, hd)
    p = np.exp2(s.astype(np.float64))
    want = p[np.arange(hd) % 16] * w / (2 + p.sum())
    assert (np.abs(got / want - 1) <= VALUE_BOUND).all(), np.abs(got / want - 1).max() * 2 ** 24


@pytest.mark.gpu
@pytest.mark.parametrize("hd,heads,kvh,n,form", CASES)
def test_products_of_scores(hd, heads, kvh, n, form):
    t, kh = score_inputs(hd, n * heads)
    q0 = (t / scale_log2(hd)).reshape(n, heads)
    q = np.zeros((n, heads, hd), np.float32)
    q[..., 0] = q0
    k, v = cache(hd, kvh, n, kh, np.ones(hd, np.float32), -300)
    got = run(heads, kvh, START, q.reshape(n, -1), k, v, form).reshape(n, heads, hd)
    t = (q0 * scale_log2(hd)).astype(np.float64)  # as the kernel pre-scales it, in f32
    p = np.exp2(t[..., None] * kh)
    want = (p / (2 + p.sum(-1, keepdims=True)))[..., np.arange(hd) % 16]
    assert (np.abs(got / want - 1) <= SCORE_BOUND).all(), np.abs(got / want - 1).max() * 2 ** 24


def planes(x):
    """x as three bf16 values (f32 arrays), each the rounded rest of the ones before."""
    out = []
    for _ in range(3):
        u = x.view(np.uint32)
        p = ((u + np.uint32(0x7FFF) + ((u >> np.uint32(16)) & np.uint32(1)))
             & np.uint32(0xFFFF0000)).view(np.float32)
        out.append(p.astype(np.float64))
        x = x - p
    return out


SIX = [(0, 0), (0, 1), (1, 0), (1, 1), (0, 2), (2, 0)]


def six_products(a, b, without=None):
    pa, pb = planes(a), planes(b)
    return sum(pa[i] * pb[j] for i, j in SIX if (i, j) != without)


@pytest.mark.parametrize("hd", [64, 128])
def test_bounds_lie_below_each_product(hd):
    s, w = value_inputs(hd)
    p = np.exp2(s.astype(np.float64)).astype(np.float32)[np.arange(hd) % 16]
    t, kh = score_inputs(hd, 40)  # 20 rows of two heads, the smallest case
    t, kh = (x.ravel().copy() for x in np.broadcast_arrays(t[:, None], kh[None]))

    def errors(without):
        value = np.abs(six_products(p, w, without) / (p.astype(np.float64) * w) - 1).max()
        d = six_products(t, kh, without) - t.astype(np.float64) * kh
        return value, np.abs(np.expm1(np.log(2) * d)).max() / 2  # half: the row sum's share

    assert errors(None)[0] < 2.0 ** -24 and errors(None)[1] < 2.0 ** -19
    for product in SIX:
        value, score = errors(product)
        assert value > 1.5 * VALUE_BOUND and score > 1.5 * SCORE_BOUND, (product, value, score)


def test_forms_named_are_those_of_the_dispatch_rules():
    for hd, heads, kvh, n, form in CASES:
        assert split_form(hd * heads, heads, kvh, START, n) == form
