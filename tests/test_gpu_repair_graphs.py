"""Builds on one workspace: the data decides how many rounds run and in which one a
lean batch stops, not which graphs exist, and the rules equal the oracle's behind
every length of the last batch."""
import numpy as np
import pytest

import oracle as oc

pytestmark = pytest.mark.gpu

PAIRS = 40


def _ties_in(rng, rnd):
    """40 pairs of words of their own, each rarer than the one before but for the one
    after `rnd`, shuffled: the rules take them in order, and only that round ties
    (what the shuffle makes adjacent occurs far less often)."""
    counts = 200 - 3 * np.arange(PAIRS)
    counts[rnd + 1] = counts[rnd]
    which = rng.permutation(np.repeat(np.arange(PAIRS), counts))
    return (np.stack([2 * which + 1, 2 * which + 2], 1).reshape(-1).astype(np.uint16)) << 7


@pytest.mark.parametrize("max_rules", [3, 8, 9, 10, 13, 30])
def test_graphs_per_workspace(max_rules, gpu):
    import torch

    import checkers_amd as ck
    n = int(_ties_in(np.random.default_rng(0), 5).size) + 3
    k = ck.repair_masked_bits(1, None)
    rp = ck.Repairer(n, 1, None, max_rules)
    before = ck.lib().ckr_repair_graphs_made()
    for rnd in (1, 3, 4, 5, 6, 7, 8, 9, 12, 14, 15, 21, 25):
        w = _ties_in(np.random.default_rng(rnd), rnd)
        words = np.concatenate([w, np.full(n - w.size, 500 << 7, np.uint16)])
        raw = words.view(np.uint8)
        ref = oc.repair_build(raw, n, 2, k, max_rules, want_seq=True)
        got = rp.build(torch.from_numpy(raw.copy()).to(gpu), want_seq=True)
        assert got["rules"] == ref["rules"] and got["out_len"] == ref["out_len"]
        assert np.array_equal(got["seq"], ref["seq"])
    made = ck.lib().ckr_repair_graphs_made() - before
    assert made <= 6, made


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("max_rules", [13, 30, 38])
def test_recounts_within_lean_batches(max_rules, mode, gpu):
    """Words without a tie among the pairs, so that lean batches run from the third
    round on; in mode 2 the table's limit is passed every few rounds, the rest of the
    batch leaves the sequence alone and the next full round counts again."""
    import torch

    import checkers_amd as ck
    w = _ties_in(np.random.default_rng(3), PAIRS - 2)
    raw = np.ascontiguousarray(w).view(np.uint8)
    ref = oc.repair_build(raw, w.size, 2, ck.repair_masked_bits(1, None), max_rules, want_seq=True)
    rp = ck.Repairer(w.size, 1, None, max_rules)
    src = torch.from_numpy(raw.copy()).to(gpu)
    old = ck.set_fast_paths(mode)
    try:
        for _ in range(2):
            got = rp.build(src, want_seq=True)
            assert got["rules"] == ref["rules"] and got["out_len"] == ref["out_len"]
            assert np.array_equal(got["seq"], ref["seq"])
        ck.profile_begin()  # (kernels one by one: what ran can be counted)
        got = rp.build(src)
        prof = ck.profile_end()
    finally:
        ck.set_fast_paths(old)
    assert got["rules"] == ref["rules"]
    lean = prof["repair_find_kernel"][0] - prof["repair_count_kernel"][0]
    stopped = prof["repair_find_kernel"][0] - max_rules
    assert lean > 0 and (stopped > 0 if mode == 2 else stopped == 0), prof


def test_small_counts_take_full_rounds(gpu):
    """Top counts below 64, where ties are common: no lean round is tried, so that a
    tie costs no extra batch."""
    import torch

    import checkers_amd as ck
    rng = np.random.default_rng(2)
    counts = 60 - np.arange(20)
    counts[6] = counts[5]
    which = rng.permutation(np.repeat(np.arange(20), counts))
    w = np.stack([2 * which + 1, 2 * which + 2], 1).reshape(-1).astype(np.uint16) << 7
    raw = np.ascontiguousarray(w).view(np.uint8)
    ref = oc.repair_build(raw, w.size, 2, ck.repair_masked_bits(1, None), 18)
    rp = ck.Repairer(w.size, 1, None, 18)
    ck.profile_begin()
    got = rp.build(torch.from_numpy(raw.copy()).to(gpu))
    prof = ck.profile_end()
    assert got["rules"] == ref["rules"]
    assert prof["repair_find_kernel"][0] == prof["repair_count_kernel"][0] == 18
