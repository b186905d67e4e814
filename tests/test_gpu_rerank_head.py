"""The rerank run's head on the device against the host head over the same
session's CLS states, with and without a pooler and its bias, at widths and
row counts that end inside its tiles, and the states and scores it refuses, on
an MI355X through the C ABI."""
import numpy as np
import pytest

import turboembed_amd as T
from turboembed_amd import seam as S
from turboembed_amd.rerank import RerankHead, head_scores, pair_windows

import small

pytestmark = pytest.mark.gpu

START, END, SEQ = 1, 2, 24


def _pairs(n, vocab):
    """n pairs, the last of them three windows long: the run's windows pass
    max_batch = n."""
    g = np.random.Generator(np.random.PCG64(n))
    ids = lambda k: g.integers(3, vocab - 1, size=k).tolist()  # noqa: E731
    return [(ids(3), ids(1 + i % 15)) for i in range(n - 1)] + [(ids(4), ids(40))]


def _head(hidden, pooler, bias):
    g = np.random.Generator(np.random.PCG64(hidden))
    f = lambda *s: g.standard_normal(s).astype(np.float32) / np.float32(np.sqrt(hidden))  # noqa: E731
    return RerankHead(f(hidden), 0.125, f(hidden, hidden) if pooler else None, f(hidden) if pooler and bias else None)


def _host_scores(s, pairs, head):
    """The host head over the states of the windows in the run's own runs."""
    ids, types, lens, owner = [], [], [], []
    for i, (q, p) in enumerate(pairs):
        wi, wt, wl = pair_windows(q, p, START, END, query_tokens=8, max_tokens=SEQ)
        ids, types, lens, owner = ids + list(wi), types + list(wt), lens + list(wl), owner + [i] * len(wl)
    width = max(lens)
    mask = (np.arange(width)[None, :] < np.array(lens)[:, None]).astype(np.int32)
    ids, types = np.array(ids)[:, :width].copy(), np.array(types)[:, :width].copy()
    out = np.full(len(pairs), -np.inf, np.float32)
    for at in range(0, len(lens), s.max_batch):
        cut = slice(at, at + s.max_batch)
        states = s.embed(ids[cut], mask[cut], types[cut], pooling=S.TURBO_POOLING_CLS,
                         normalize=S.TURBO_NORMALIZE_NONE)
        np.maximum.at(out, owner[cut], head_scores(states, head))
    return out


@pytest.mark.parametrize("hidden, heads", [(8, 1), (24, 3), (72, 9), (320, 5)])
@pytest.mark.parametrize("n", [1, 17, 33])
@pytest.mark.parametrize("pooler, bias", [(True, True), (True, False), (False, False)])
def test_the_run_s_head_is_the_host_s(context, hidden, heads, n, pooler, bias):
    desc = small.bert(seed=83, hidden=hidden, heads=heads, inter=64)
    head = _head(hidden, pooler, bias)
    model = context.load(desc)
    s = model.session(n, SEQ, S.TURBO_PRECISION_EXACT, task=S.TURBO_TASK_RERANK)
    pairs = _pairs(n, desc.vocab_size)
    want = _host_scores(s, pairs, head)
    got = s.rerank(pairs, head, START, END, query_tokens=8)
    # Both round an F64 sum once: an F32 ulp apart where it lies between two
    # values; a pooled value on such a boundary moves its term by an ulp of 1.
    bound = 2.0 ** -23 * np.abs(want) + 2.0 ** -24 * np.abs(head.classifier_weight).max()
    assert (np.abs(got - want) <= bound).all(), (got, want)
    s.close()
    model.close()


def test_states_and_scores_that_are_not_finite_are_refused(context):
    # The vocabulary's last token has an infinite embedding: a pair that holds
    # it is refused, and the calls before and after it are not.
    desc = small.bert(seed=84, hidden=72, heads=9, inter=64)
    desc.tensors[0][-1, 3] = np.inf
    head = _head(72, True, True)
    model = context.load(desc)
    s = model.session(9, SEQ, S.TURBO_PRECISION_EXACT, task=S.TURBO_TASK_RERANK)
    pairs = _pairs(9, desc.vocab_size)
    want = s.rerank(pairs, head, START, END, query_tokens=8)
    assert np.isfinite(want).all()
    bad = list(pairs)
    bad[4] = (bad[4][0], [desc.vocab_size - 1])
    loud = RerankHead(np.copysign(np.float32(3e38), head.classifier_weight), 0.0)
    for p, h, what in ((bad, head, "non-finite rerank encoder output"), (pairs, loud, "overflows F32")):
        with pytest.raises(T.TurboError, match=what) as e:
            s.rerank(p, h, START, END, query_tokens=8)
        assert e.value.code == S.TURBO_E_INTERNAL
        np.testing.assert_array_equal(s.rerank(pairs, head, START, END, query_tokens=8), want)
    s.close()
    model.close()
