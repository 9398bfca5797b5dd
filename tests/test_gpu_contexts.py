"""Many contexts alive together: their error words share pages of pinned host memory, one
word each, so that a context has no pinned allocation of its own, and an error is
reported by its own context alone, also on a word that another context had before."""
import numpy as np
import pytest

from p3_compare import device_fields
from scream_amd import p3x
from scream_amd.inputs import make_columns

pytestmark = pytest.mark.gpu


def _mappings():
    with open("/proc/self/maps") as f:
        return sum(1 for _ in f)


def test_no_pinned_allocation_per_context(host_tables):
    first = p3x.Context(host_tables)
    before, n = _mappings(), 24
    kept = [p3x.Context(host_tables) for _ in range(n)]
    grown = _mappings() - before
    for c in kept:
        c.close()
    first.close()
    # the device tables and streams are 2.7 mappings each, a pinned allocation one more
    assert grown <= 3 * n, grown


def test_error_words_are_apart(host_tables):
    import torch
    inp = make_columns(40, 16, seed=3)
    bad = {k: v.copy() for k, v in inp.items()}
    bad["th"][5, 7] = -1.0
    stream = torch.cuda.current_stream().cuda_stream

    def step(ctx, fields):
        d, _ = device_fields(fields)
        ctx.main(d, 40, 16, 300.0, exchange_zeroed=True, stream=stream, async_=True)
        return d  # alive until the step has ended

    ctxs = [p3x.Context(host_tables) for _ in range(130)]  # three pages of 64 words
    failing = (0, 63, 64, 129)
    keep = [step(c, bad if n in failing else inp) for n, c in enumerate(ctxs)]
    want = [p3x.P3X_ERR_TEMPERATURE if n in failing else p3x.P3X_OK for n in range(len(ctxs))]
    assert [c.sync() for c in ctxs] == want
    assert all(c.sync() == p3x.P3X_OK for c in ctxs)  # reported once
    # a word that goes back with an error on it is clean for the next context
    keep.append(step(ctxs[64], bad))
    ctxs[64].close()
    again = p3x.Context(host_tables)
    assert again.sync() == p3x.P3X_OK
    keep.append(step(again, inp))
    assert again.sync() == p3x.P3X_OK
    for c in ctxs:
        c.close()
    keep.append(step(again, bad))
    assert again.sync() == p3x.P3X_ERR_TEMPERATURE
    again.close()
    np.testing.assert_equal(len(keep), len(ctxs) + 3)
