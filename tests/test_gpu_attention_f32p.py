"""Attention with F32 probabilities on the matrix cores (F32 heads of 32 and
64, 16-bit heads of 32): rows at the edges of its 32-query, 32-key and
128-query blocks, masked keys through them, and windows, against the oracle on
an MI355X through the C ABI."""
import numpy as np
import pytest

import oracle
from turboembed_amd import seam as S
from turboembed_amd.model import with_dtype

import small
from test_gpu_parity import assert_close

pytestmark = pytest.mark.gpu


# (Heads of 64 on the F32 tier alone: the 16-bit ones take the other kernel.)
@pytest.mark.parametrize("tier, heads", [("f32", 4), ("f32", 2), ("f16", 4), ("bf16", 4)])
@pytest.mark.parametrize("family, window", [("bert", 0), ("modernbert", 16), ("modernbert", 40)])
def test_rows_at_block_edges_meet_the_oracle(context, tier, heads, family, window):
    # Weights N(0, 0.3) spread the scores over tens of units; N(0, 0.1) on
    # BF16, whose operands' rounding (2^-9 of each, the scores' 2^-9 of tens)
    # alone moves such softmaxes past the dtype's floor, as it does on the
    # kernel for heads of 64.
    seq, std = 300, 0.1 if tier == "bf16" else 0.3
    if family == "bert":
        desc = small.bert(seed=51, hidden=128, heads=heads, inter=256, positions=seq, std=std)
    else:
        desc = small.modernbert(seed=51, hidden=128, heads=heads, inter=192, positions=seq, window=window,
                                global_every=2, std=std)
    precision = S.TURBO_PRECISION_EXACT if tier == "f32" else S.TURBO_PRECISION_FASTEST
    if tier == "bf16":
        desc, precision = with_dtype(desc, "bf16"), S.TURBO_PRECISION_MODEL
    g = np.random.Generator(np.random.PCG64(51))
    lens = [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 257, 300]
    ids = g.integers(0, desc.vocab_size, size=(len(lens), seq)).astype(np.int32)
    mask = (np.arange(seq)[None, :] < np.array(lens)[:, None]).astype(np.int32)
    mask[8, 32:64] = 0             # a whole block of masked keys
    mask[10, [0, 31, 32, 96]] = 0
    mask[12, 5:290:3] = 0
    types = g.integers(0, 2, size=ids.shape).astype(np.int32) if family == "bert" else None
    model = context.load(desc)
    s = model.session(len(lens), seq, precision)
    got = s.embed(ids, mask, types)
    assert_close(got, oracle.encode(desc, ids, mask, types), s.compute_dtype)
    assert np.array_equal(s.embed(ids, mask, types), got)
    s.close()
    model.close()


@pytest.mark.parametrize("heads", [4, 2])
@pytest.mark.parametrize("family", ["bert", "modernbert"])
@pytest.mark.parametrize("scale", [1e4, 1e6])
def test_scores_of_any_size_meet_the_oracle(context, heads, family, scale):
    # Query and key weights scaled by 1e4 and 1e6: scores of 1e9 and 1e13,
    # whose ulps are far past exp's range, so all weight is on one key (or on
    # equal ones) and only the scores' differences may count.
    desc = getattr(small, family)(seed=51, hidden=128, heads=heads, inter=64, positions=200, std=0.2)
    for i, t in enumerate(desc.tensors):
        if family == "bert" and i >= 5 and (i - 5) % 16 in (0, 2):
            desc.tensors[i] = t * np.float32(scale)
        if family == "modernbert" and i >= 3 and (i - 3) % 6 == 1:
            desc.tensors[i][:256] *= np.float32(scale)
    ids, mask, types = small.ragged_rows(3, 6, 150, desc.vocab_size)
    types = None if family == "modernbert" else types
    model = context.load(desc)
    s = model.session(6, 150, S.TURBO_PRECISION_EXACT)
    assert_close(s.embed(ids, mask, types), oracle.encode(desc, ids, mask, types), s.compute_dtype)
    s.close()
    model.close()


@pytest.mark.parametrize("heads", [4, 2])
@pytest.mark.parametrize("window", [149, 150, 2 ** 31 - 156])
def test_windows_over_the_rows_length_reach_every_key(context, heads, window):
    desc = small.modernbert(seed=57, hidden=128, heads=heads, inter=64, positions=200, window=2 * window)
    ids, mask, _ = small.ragged_rows(3, 6, 150, desc.vocab_size)
    model = context.load(desc)
    s = model.session(6, 150, S.TURBO_PRECISION_EXACT)
    assert_close(s.embed(ids, mask), oracle.encode(desc, ids, mask, None), s.compute_dtype)
    s.close()
    model.close()


@pytest.mark.parametrize("tier, heads, value", [("f32", h, v) for h in (4, 2) for v in (np.inf, -np.inf, np.nan)] +
                         [("f16", 4, np.inf), ("f16", 4, -np.inf)])
def test_a_head_of_infinite_or_nan_scores_has_no_context(context, tier, heads, value):
    # One key column of head 1 infinite (a weight or a bias; on F16 a bias
    # past its range): each query's scores are infinities of either sign, the
    # largest infinite or all of them minus infinity. Or not a number. The
    # head then gives what one of zero values gives, in the first layer alone.
    width, at = 128 // heads, 128 // heads + 5
    value16 = np.copysign(1e6, value) if tier == "f16" else value

    def model_with(what):
        # (Layer 0's key weight and bias are tensors 7 and 8, its value ones 9 and 10.)
        desc = small.bert(seed=58, hidden=128, heads=heads, inter=64, positions=300, std=0.1, layers=2)
        if what == "zero values":
            desc.tensors[9][width:2 * width], desc.tensors[10][width:2 * width] = 0.0, 0.0
        elif what == "weight":
            desc.tensors[7][at, 3] = value
        else:
            desc.tensors[8][at] = value16
        return desc

    desc = model_with("zero values")
    ids, mask, types = small.ragged_rows(4, 9, 300, desc.vocab_size)
    want = oracle.encode(desc, ids, mask, types)
    precision = S.TURBO_PRECISION_EXACT if tier == "f32" else S.TURBO_PRECISION_FASTEST
    for what in ("bias",) if tier == "f16" else ("weight", "bias"):
        model = context.load(model_with(what))
        s = model.session(9, 300, precision)
        assert_close(s.embed(ids, mask, types), want, s.compute_dtype)
        s.close()
        model.close()
