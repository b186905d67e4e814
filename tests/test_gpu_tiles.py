"""The GEMM shapes for few rows (d32x32, 64x64), for F32 operands as BF16
terms (x64x64, x128x128) and the rule that picks among them, at the edges of
their tiles and of k, residual products in slices of K, and means of every
length, on an MI355X through the C ABI."""
import numpy as np
import pytest

import oracle
import turboembed_amd as T
from turboembed_amd import seam as S
from turboembed_amd.model import to_bf16_bits, with_dtype

import small
from test_gpu_parity import assert_close

pytestmark = pytest.mark.gpu

EDGES = [(1, 96, 64), (31, 32, 8), (32, 33, 72), (65, 100, 192), (129, 257, 100), (300, 384, 1536), (1100, 768, 320)]


def _rounded(x, dtype):
    if dtype == S.TURBO_DTYPE_F16:
        return x.astype(np.float16).astype(np.float64)
    if dtype == S.TURBO_DTYPE_BF16:
        return (to_bf16_bits(x).astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    return x.astype(np.float64)


def _operands(m, n, k):
    g = np.random.Generator(np.random.PCG64(m + 3 * n + 7 * k))
    return (g.standard_normal((m, k)).astype(np.float32), g.standard_normal((n, k)).astype(np.float32),
            g.standard_normal(n).astype(np.float32))


@pytest.mark.parametrize("dtype", [S.TURBO_DTYPE_F32, S.TURBO_DTYPE_F16, S.TURBO_DTYPE_BF16])
@pytest.mark.parametrize("tile", [0, 20, 21, 22, 23])
@pytest.mark.parametrize("mnk", EDGES)
def test_small_and_split_shapes_match_numpy(runtime, dtype, tile, mnk):
    m, n, k = mnk
    if dtype != S.TURBO_DTYPE_F32 and k % 8:
        k += 4   # 16-bit operands come in whole 16-byte vectors
    a, w, b = _operands(m, n, k)
    got = T.gemm_check(a, w, b, dtype=dtype, tile=tile)
    want = _rounded(a, dtype) @ _rounded(w, dtype).T + b
    # An F32 sum of k products of unit variance: k roundings of at most
    # 2^-24 of a partial sum (at most about 5 sqrt(k)) if every one went
    # the same way; they do not, and a tenth of that bounds them. (Every
    # shape's, the F32 core's 1.7e-5 at k = 100 too; a BF16 term's product
    # left out would pass here, and fails the two tests of the terms below.)
    bound = max(0.1 * k * 5 * np.sqrt(k) * 2.0 ** -24, 4e-6)
    assert np.abs(got - want).max() <= bound, (np.abs(got - want).max(), bound)


@pytest.mark.parametrize("mnk", [(200, 300, 772), (300, 256, 3072)])
def test_bf16_terms_are_no_further_off_than_the_f32_products(runtime, mnk):
    # Against 64 bits: three BF16 terms an operand, six products, must not
    # lose to the F32 matrix core's own sums (measured 3.4e-7 against 1.0e-6
    # at k = 3072).
    a, w, b = _operands(*mnk)
    want = a.astype(np.float64) @ w.astype(np.float64).T + b
    off = [np.linalg.norm(T.gemm_check(a, w, b, tile=t) - want) for t in (1, 20, 22, 23)]
    assert max(off[1:]) <= off[0], off


def test_operands_of_every_magnitude_keep_their_terms(runtime):
    # Rows and columns scaled by 2^-60 to 2^60: each output's error stays
    # relative to its own operands.
    m, n, k = 70, 90, 256
    a, w, _ = _operands(m, n, k)
    sa, sw = 2.0 ** np.linspace(-60, 60, m).round(), 2.0 ** np.linspace(60, -60, n).round()
    for t in (20, 22, 23):
        got = T.gemm_check((a * sa[:, None]).astype(np.float32), (w * sw[:, None]).astype(np.float32), tile=t)
        want = a.astype(np.float64) @ w.astype(np.float64).T
        assert np.abs(got.astype(np.float64) / sa[:, None] / sw[None, :] - want).max() <= 1e-5 * np.sqrt(k)


@pytest.mark.parametrize("value", [1 + 2.0 ** -7 - 2.0 ** -16, 1 + 2.0 ** -8 - 2.0 ** -17, 1 + 2.0 ** -8 + 2.0 ** -17])
@pytest.mark.parametrize("k", [16, 64, 768])
def test_bf16_terms_of_like_operands_lose_no_more_than_a_rounding(runtime, value, k):
    # Every product the same, so that what the six products leave out (at most
    # 2^-24 of each) and the roundings (one per 16 columns of k, one as the
    # small terms' sum, 2^-7 of the whole with five roundings per 16, is
    # added) may all go one way.
    x = np.float32(value)
    a, w = np.full((70, k), x), np.full((90, k), x)
    a[1::2] *= -1
    want = a.astype(np.float64) @ w.astype(np.float64).T
    bound = (2 + k / 16 * (1 + 5 / 128)) * 2.0 ** -24
    for tile in (22, 23):
        off = np.abs(T.gemm_check(a, w, tile=tile) / want - 1).max()
        assert off <= bound, (tile, off * 2 ** 24)


@pytest.mark.parametrize("tile", [22, 23])
def test_values_that_are_not_finite_are_the_f32_core_s(runtime, tile):
    # Infinities, a NaN, F32's largest value and sums past it, one to a row or
    # column in tiles of their own and shared ones: where the F32 matrix core
    # has an infinity, a NaN or a value, the BF16 terms have the same.
    m, n, k = 300, 260, 100
    a, w, b = _operands(m, n, k)
    big = np.finfo(np.float32).max
    a[3, 7], a[40, 99], a[41, 0], a[41, 50] = np.inf, -np.inf, np.inf, -np.inf
    a[130, 5], a[280, 64] = np.nan, big
    a[200], a[200, 3], w[:, 3] = 0.0, 2.0 ** 126, 4.0 * w[:, 3]   # products past F32's range, one a sum
    w[70, 3], w[255, 98] = -np.inf, np.nan
    w[10] = 2.0 ** -100
    with np.errstate(all="ignore"):
        got, want = T.gemm_check(a, w, b, tile=tile), T.gemm_check(a, w, b, tile=1)
    assert np.isinf(want).any(1)[[3, 40, 200, 280]].all() and np.isfinite(want[[200, 280], 10]).all()
    np.testing.assert_allclose(got, want, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("mnk", [(1, 64, 128), (65, 192, 384), (300, 2304, 768)])
def test_int8_shapes_have_the_same_bits(runtime, mnk):
    a, w, b = _operands(*mnk)
    want = T.gemm_check(a, w, b, dtype=S.TURBO_DTYPE_I8, tile=7)
    for t in (0, 5, 21):
        np.testing.assert_array_equal(T.gemm_check(a, w, b, dtype=S.TURBO_DTYPE_I8, tile=t), want)


@pytest.mark.parametrize("tier", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("family", ["bert", "modernbert"])
@pytest.mark.parametrize("inter", [1536, 2080])
def test_residual_products_in_slices_meet_the_oracle(context, monkeypatch, family, tier, inter):
    # Short runs cut FFN-out's K into slices that the add + LayerNorm adds
    # (2080: the last one shorter), from one token up; replayed and launched
    # directly, the same bits.
    build = getattr(small, family)
    desc = build(seed=71, hidden=128, heads=2, inter=inter, positions=96, std=0.05)
    precision = S.TURBO_PRECISION_EXACT if tier == "f32" else S.TURBO_PRECISION_FASTEST
    if tier == "bf16":
        desc, precision = with_dtype(desc, "bf16"), S.TURBO_PRECISION_MODEL
    model = context.load(desc)
    s = model.session(4, 96, precision)
    monkeypatch.setenv("TURBO_ROCM_GRAPHS", "0")
    direct = model.session(4, 96, precision)
    for batch, seq in ((1, 1), (1, 33), (4, 96)):
        ids, mask, types = small.ragged_rows(71 + seq, batch, seq, desc.vocab_size)
        types = None if family == "modernbert" else types
        got = s.embed(ids, mask, types)
        assert_close(got, oracle.encode(desc, ids, mask, types), s.compute_dtype)
        np.testing.assert_array_equal(direct.embed(ids, mask, types), got)
    direct.close()
    s.close()
    model.close()


def test_means_of_every_length_meet_the_oracle(context):
    # Ranges at the edges of the finish's 32 tokens and of a chunk's parts and
    # chunks, over masked tokens; a whole row's range the row's own mean bit for bit.
    desc = small.bert(seed=73, hidden=320, heads=5, inter=64, positions=600, std=0.1)
    g = np.random.Generator(np.random.PCG64(73))
    ids = g.integers(0, desc.vocab_size, size=(3, 599)).astype(np.int32)
    mask = np.ones((3, 599), np.int32)
    mask[0, g.choice(np.arange(1, 598), 150, replace=False)] = 0
    mask[0, 3] = 1
    mask[1, 100:180] = 0
    mask[2, 20:] = 0
    types = np.zeros_like(ids)
    lens = [1, 2, 31, 32, 33, 63, 64, 65, 255, 256, 257, 288, 289, 511, 512, 513]
    ranges = [(r, 3 + r, 3 + r + n) for r in (0, 1) for n in lens]
    ranges += [(1, 90, 110), (1, 60, 175), (2, 0, 20), (0, 0, 599)]
    model = context.load(desc)
    s = model.session(3, 600, S.TURBO_PRECISION_EXACT, max_ranges=len(ranges))
    s.write_ranges(ids, mask, ranges, types)
    s.run()
    got = s.read()
    assert_close(got, oracle.encode(desc, ids, mask, types, ranges=ranges), s.compute_dtype)
    rows = s.embed(ids, mask, types)
    np.testing.assert_array_equal(rows[0], got[-1])
    np.testing.assert_array_equal(rows[2], got[-2])
    s.close()
    model.close()


def test_a_model_without_layers_opens_with_split_bins(context):
    # Embeddings alone, on a session whose larger bins split their runs: the
    # split's rule has no layer to take its products' sizes from.
    desc = small.bert(seed=79, layers=0, positions=512)
    ids, mask, types = small.ragged_rows(79, 24, 512, desc.vocab_size)
    model = context.load(desc)
    s = model.session(64, 512, S.TURBO_PRECISION_EXACT)
    assert_close(s.embed(ids, mask, types), oracle.encode(desc, ids, mask, types), s.compute_dtype)
    s.close()
    model.close()
