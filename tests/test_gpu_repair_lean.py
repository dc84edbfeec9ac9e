"""Grammar builds around the lean rounds' stops: a tie in the first rounds, ties
that set in once the counts have fallen, none at all, a grammar that ends within
a batch, and rule limits on both sides of a batch's length.  All integer: the
rules, the lengths and the sequence equal the oracle's.
"""
import numpy as np
import pytest

import oracle as oc

pytestmark = pytest.mark.gpu


def _tied(rng, n):
    """Every word as frequent as the next: the top count ties in most rounds."""
    return np.tile(rng.permutation(64).astype(np.uint16) << 7, n // 64 + 1)[:n]


def _skewed(rng, n):
    """A skewed alphabet: no tie while the counts are large, ties at the end."""
    return (np.minimum(rng.geometric(0.2, n), 400).astype(np.uint16)) << 7


def _late_tie(rng, n):
    """A skewed half, and words of their own pairs that all occur 9 times."""
    rare = np.repeat(np.arange(200, 260, dtype=np.uint16).reshape(-1, 2), 9, axis=0)
    return np.concatenate([_skewed(rng, n), (rng.permutation(rare).reshape(-1) << 7).astype(np.uint16)])


def _ends(rng, n):
    """Two words only: the grammar ends (or the top pair is one word's run) early."""
    return (rng.integers(0, 2, n).astype(np.uint16)) << 7


@pytest.mark.parametrize("max_rules", [1, 7, 8, 9, 40, 150])
@pytest.mark.parametrize("gen,n", [(_tied, 3000), (_skewed, 700), (_skewed, 40000), (_late_tie, 5000), (_ends, 64),
                                   (_ends, 9000), (_tied, 2)], ids=lambda v: getattr(v, "__name__", str(v)))
def test_lean_rounds(gpu, gen, n, max_rules):
    import torch

    import checkers_amd as ck
    words = np.ascontiguousarray(gen(np.random.default_rng(n + max_rules), n))
    raw = words.view(np.uint8)
    k = ck.repair_masked_bits(1, None)
    ref = oc.repair_build(raw, words.size, 2, k, max_rules, want_seq=True)
    got = ck.Repairer(words.size, 1, None, max_rules).build(torch.from_numpy(raw.copy()).to(gpu), want_seq=True)
    assert got["rules"] == ref["rules"]
    assert got["out_len"] == ref["out_len"] and got["max_pair"] == ref["max_pair"]
    assert np.array_equal(got["seq"], ref["seq"])
